// Many Lz sectors of one fermions-on-the-sphere problem in single launches.
//
// The reference solves the sectors one after the other (FQHESphereFermionsTwoBodyGeneric.cc:270
// loops over Lz, each with its own FermionOnSphere, Hamiltonian and Lanczos).  Here the
// sectors of uneven dimension share one concatenated basis, one factor table and one low-bit
// rank table; a product over every active sector is one persistent launch whose workgroups
// stride over (sector, row-tile) work items, and the Lanczos vector operations are segmented
// by sector so that every sector keeps its own Krylov space.
//
// Block vectors of the set: per sector a [D_s][k] block, sectors concatenated in order, so
// global row g of sector s is offset_s + local row.
#include <algorithm>
#include <cstring>

#include "dh_index.h"
#include "dh_internal.h"
#include "dh_sphere_row.h"

// device-side subset-count table (same recursion as the single-sector basis)
static std::vector<int64_t> subset_table(int nOrb, int maxN, int& maxSum) {
  maxSum = 0;
  for (int i = 0; i < maxN; ++i) maxSum += nOrb - 1 - i;
  std::vector<int64_t> t((size_t)(nOrb + 1) * (maxN + 1) * (maxSum + 1), 0);
  auto idx = [&](int j, int n, int s) { return ((size_t)j * (maxN + 1) + n) * (maxSum + 1) + s; };
  t[idx(0, 0, 0)] = 1;
  for (int j = 0; j < nOrb; ++j)
    for (int n = 0; n <= maxN; ++n)
      for (int s = 0; s <= maxSum; ++s) {
        int64_t v = t[idx(j, n, s)];
        if (n >= 1 && s >= j) v += t[idx(j, n - 1, s - j)];
        t[idx(j + 1, n, s)] = v;
      }
  return t;
}

__global__ void ms_unrank_kernel(uint64_t* __restrict__ states, int64_t dim, int nbrOrbitals, int nbrFermions,
                                 int orbitalSum, const int64_t* __restrict__ T, int maxN, int maxSum) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  int64_t rem = i;
  int n = nbrFermions, s = orbitalSum;
  uint64_t state = 0;
  for (int j = nbrOrbitals - 1; j >= 0 && n > 0; --j) {
    int64_t c = 0;
    if (s >= j && s - j <= maxSum) c = T[((int64_t)j * (maxN + 1) + (n - 1)) * (maxSum + 1) + (s - j)];
    if (rem < c) {
      state |= (1ull << j);
      --n;
      s -= j;
    } else {
      rem -= c;
    }
  }
  states[i] = state;
}

extern "C" int dh_sector_set_create(dh_context* c, dh_sector_set** out, int N, int lzMax, const int* totalLz,
                                    int nbrSectors) {
  if (!c || !out || !totalLz || nbrSectors <= 0) return DH_E_ARG;
  *out = nullptr;
  if (c->closed) return dh_fail(c, DH_E_STATE, "context destroyed");
  if (N <= 0 || lzMax < 0 || N > lzMax + 1) return dh_fail(c, DH_E_ARG, "need 0 < nbr_fermions <= lz_max + 1");
  if (lzMax > 62) return dh_fail(c, DH_E_RANGE, "lz_max must be <= 62");
  hipSetDevice(c->device);
  const int nOrb = lzMax + 1;
  int maxSum;
  std::vector<int64_t> T = subset_table(nOrb, N, maxSum);
  auto Tat = [&](int j, int n, int s) -> int64_t {
    if (j < 0 || j > nOrb || n < 0 || n > N || s < 0 || s > maxSum) return 0;
    return T[((size_t)j * (N + 1) + n) * (maxSum + 1) + s];
  };
  dh_sector_set* S = new dh_sector_set();
  S->ctx = c;
  S->nbrFermions = N;
  S->lzMax = lzMax;
  S->nbrOrbitals = nOrb;
  S->nbrSectors = nbrSectors;
  S->offsets.assign(nbrSectors + 1, 0);
  for (int i = 0; i < nbrSectors; ++i) {
    int twice = totalLz[i] + N * lzMax;
    if (twice < 0 || (twice & 1)) {
      delete S;
      return dh_fail(c, DH_E_ARG, "a total_lz has the wrong parity or range");
    }
    int sum = twice >> 1;
    int64_t d = Tat(nOrb, N, sum);
    if (d <= 0 || d >= (1ll << 31)) {
      delete S;
      return dh_fail(c, DH_E_ARG, "a sector is empty or larger than 2^31");
    }
    S->totalLz.push_back(totalLz[i]);
    S->orbitalSum.push_back(sum);
    S->offsets[i + 1] = S->offsets[i] + d;
  }
  S->totalDim = S->offsets[nbrSectors];
  S->rankBits = dh_rank_split(nOrb);
  S->loSize = 1ll << S->rankBits;
  S->hiSize = 1ll << (nOrb - S->rankBits);
  // rank tables: one low table, one high table per sector (the sectors' high tables on host threads:
  // 133 sectors of 2^20 entries at 34 orbitals)
  std::vector<uint32_t> lo(S->loSize, 0), hi((size_t)S->hiSize * nbrSectors, 0);
  for (uint64_t l = 0; l < (uint64_t)S->loSize; ++l) {
    int n = 0, s = 0;
    int64_t acc = 0;
    for (uint64_t r = l; r; r &= r - 1) {
      int j = __builtin_ctzll(r);
      ++n;
      s += j;
      acc += Tat(j, n, s);
    }
    lo[l] = (uint32_t)acc;
  }
  dh_parallel_for(nbrSectors, [&](int sec) {
    for (uint64_t h = 0; h < (uint64_t)S->hiSize; ++h) {
      int popH = __builtin_popcountll(h), sumH = 0;
      for (uint64_t r = h; r; r &= r - 1) sumH += S->rankBits + __builtin_ctzll(r);
      int n = N - popH, s = S->orbitalSum[sec] - sumH;
      const int64_t last = S->offsets[sec + 1] - S->offsets[sec] - 1;
      hi[(size_t)sec * S->hiSize + h] = (uint32_t)last;
      if (n < 0 || s < 0) continue;
      int64_t acc = 0;
      for (uint64_t r = h; r; r &= r - 1) {
        int j = S->rankBits + __builtin_ctzll(r);
        ++n;
        s += j;
        acc += Tat(j, n, s);
      }
      hi[(size_t)sec * S->hiSize + h] = (uint32_t)(last - acc);
    }
  });
  const std::vector<uint16_t> lo16 = dh_rank_lo16(lo);
  int rc;
  int64_t* d_T = nullptr;
  if ((rc = dh_alloc(c, (void**)&d_T, sizeof(int64_t) * T.size())) ||
      (rc = dh_alloc(c, (void**)&S->d_states, sizeof(uint64_t) * S->totalDim)) ||
      (rc = dh_alloc(c, (void**)&S->d_rankLo, sizeof(uint32_t) * lo.size())) ||
      (rc = dh_alloc(c, (void**)&S->d_rankHi, sizeof(uint32_t) * hi.size())) ||
      (!lo16.empty() && (rc = dh_alloc(c, (void**)&S->d_rankLo16, sizeof(uint16_t) * lo16.size()))) ||
      (rc = dh_alloc(c, (void**)&S->d_offsets, sizeof(int64_t) * (nbrSectors + 1)))) {
    if (d_T) hipFree(d_T);
    dh_sector_set_destroy(S);
    return rc;
  }
  hipMemcpyAsync(d_T, T.data(), sizeof(int64_t) * T.size(), hipMemcpyHostToDevice, c->stream);
  hipMemcpyAsync(S->d_rankLo, lo.data(), sizeof(uint32_t) * lo.size(), hipMemcpyHostToDevice, c->stream);
  hipMemcpyAsync(S->d_rankHi, hi.data(), sizeof(uint32_t) * hi.size(), hipMemcpyHostToDevice, c->stream);
  if (S->d_rankLo16)
    hipMemcpyAsync(S->d_rankLo16, lo16.data(), sizeof(uint16_t) * lo16.size(), hipMemcpyHostToDevice, c->stream);
  hipMemcpyAsync(S->d_offsets, S->offsets.data(), sizeof(int64_t) * (nbrSectors + 1), hipMemcpyHostToDevice,
                 c->stream);
  for (int sec = 0; sec < nbrSectors; ++sec) {
    int64_t d = S->offsets[sec + 1] - S->offsets[sec];
    hipLaunchKernelGGL(ms_unrank_kernel, dim3((unsigned)((d + 255) / 256)), dim3(256), 0, c->stream,
                       S->d_states + S->offsets[sec], d, nOrb, N, S->orbitalSum[sec], d_T, N, maxSum);
  }
  hipError_t e = hipStreamSynchronize(c->stream);
  hipFree(d_T);
  if (e != hipSuccess) {
    dh_sector_set_destroy(S);
    return dh_fail(c, DH_E_HIP, std::string("sector set: ") + hipGetErrorString(e));
  }
  *out = S;
  return DH_OK;
}

extern "C" int dh_sector_set_destroy(dh_sector_set* S) {
  if (!S) return DH_E_ARG;
  dh_context* c = S->ctx;
  hipStreamSynchronize(c->stream);
  for (void* p : {(void*)S->d_states, (void*)S->d_rankLo, (void*)S->d_rankHi, (void*)S->d_rankLo16, (void*)S->d_offsets,
                  (void*)S->d_factors, (void*)S->d_pairOffset, (void*)S->d_work, (void*)S->d_coef,
                  (void*)S->d_pairInfo, (void*)S->d_sumPairOff, (void*)S->d_sumPairs, (void*)S->d_sumFactorOff,
                  (void*)S->d_cfactors, (void*)S->d_packedFactors, (void*)S->d_sumBase, (void*)S->d_orbit,
                  (void*)S->d_reorder, (void*)S->d_lut, (void*)S->d_phase, (void*)S->d_freeMask,
                  (void*)S->d_freeShift, (void*)S->d_partnerPos})
    if (p) hipFree(p);
  delete S;
  return DH_OK;
}

extern "C" int dh_sector_set_offsets(const dh_sector_set* S, int64_t* offsets) {
  if (!S || !offsets) return DH_E_ARG;
  std::memcpy(offsets, S->offsets.data(), sizeof(int64_t) * (S->nbrSectors + 1));
  return DH_OK;
}

extern "C" int dh_sector_set_get_states(dh_sector_set* S, uint64_t* states) {
  if (!S || !states) return DH_E_ARG;
  dh_context* c = S->ctx;
  DH_HIP(c, hipMemcpyAsync(states, S->d_states, sizeof(uint64_t) * S->totalDim, hipMemcpyDeviceToHost, c->stream));
  DH_HIP(c, hipStreamSynchronize(c->stream));
  return DH_OK;
}

extern "C" int dh_sector_set_factors(dh_sector_set* S, const double* factors, const int* pairOffset, int nbrFactors,
                                     double shift) {
  if (!S || !factors || !pairOffset) return DH_E_ARG;
  dh_context* c = S->ctx;
  const int nOrb = S->nbrOrbitals, nPairs = nOrb * (nOrb - 1) / 2;
  int expect = 0;
  for (int m1 = 0; m1 < nOrb; ++m1)
    for (int m2 = 0; m2 < m1; ++m2) {
      if (pairOffset[m1 * (m1 - 1) / 2 + m2] != expect) return dh_fail(c, DH_E_ARG, "pair_offset layout");
      int sum = m1 + m2;
      expect += std::min(sum, nOrb - 1) - (sum / 2 + 1) + 1;
    }
  if (pairOffset[nPairs] != expect || nbrFactors != expect) return dh_fail(c, DH_E_ARG, "nbr_factors layout");
  std::vector<double> packed;
  std::vector<int> sumBase;
  bool triangles;
  int rc = dh_pack_factors_checked(c, nOrb, factors, pairOffset, packed, sumBase, triangles);
  if (rc) return rc;
  hipStreamSynchronize(c->stream);
  for (void** p : {(void**)&S->d_factors, (void**)&S->d_pairOffset, (void**)&S->d_packedFactors, (void**)&S->d_sumBase}) {
    if (*p) hipFree(*p);
    *p = nullptr;
  }
  if ((rc = dh_alloc(c, (void**)&S->d_factors, sizeof(double) * std::max(1, nbrFactors))) ||
      (rc = dh_alloc(c, (void**)&S->d_pairOffset, sizeof(int) * (nPairs + 1))) ||
      (rc = dh_alloc(c, (void**)&S->d_packedFactors, sizeof(double) * std::max<size_t>(1, packed.size()))) ||
      (rc = dh_alloc(c, (void**)&S->d_sumBase, sizeof(int) * sumBase.size())))
    return rc;
  DH_HIP(c, hipMemcpyAsync(S->d_factors, factors, sizeof(double) * nbrFactors, hipMemcpyHostToDevice, c->stream));
  DH_HIP(c, hipMemcpyAsync(S->d_pairOffset, pairOffset, sizeof(int) * (nPairs + 1), hipMemcpyHostToDevice, c->stream));
  DH_HIP(c, hipMemcpyAsync(S->d_packedFactors, packed.data(), sizeof(double) * packed.size(), hipMemcpyHostToDevice,
                           c->stream));
  DH_HIP(c, hipMemcpyAsync(S->d_sumBase, sumBase.data(), sizeof(int) * sumBase.size(), hipMemcpyHostToDevice,
                           c->stream));
  DH_HIP(c, hipStreamSynchronize(c->stream));
  S->nbrFactors = nbrFactors;
  S->nbrPairs = nPairs;
  S->nbrPackedFactors = (int)packed.size();
  S->nbrPairSums = (int)sumBase.size();
  S->triangles = triangles;
  S->shift = shift;
  return DH_OK;
}

extern "C" int dh_sector_set_launch(dh_sector_set* S, int lanesPerRow, int blockSize) {
  if (!S) return DH_E_ARG;
  if (lanesPerRow != 1 && lanesPerRow != 2 && lanesPerRow != 4 && lanesPerRow != 8)
    return dh_fail(S->ctx, DH_E_ARG, "lanes_per_row in {1,2,4,8}");
  if (blockSize < 64 || blockSize > 1024 || (blockSize % 64)) return dh_fail(S->ctx, DH_E_ARG, "block_size");
  S->lanesPerRow = lanesPerRow;
  S->blockSize = blockSize;
  S->autoLaunch = false;
  return DH_OK;
}

extern "C" int dh_sector_set_row_mode(dh_sector_set* S, int mode) {
  if (!S) return DH_E_ARG;
  if (mode != DH_INDEX_RANK && mode != DH_INDEX_RANK_FREE && mode != DH_INDEX_RANK_RANGE)
    return dh_fail(S->ctx, DH_E_ARG, "row mode must be DH_INDEX_RANK, DH_INDEX_RANK_FREE or DH_INDEX_RANK_RANGE");
  if (S->kind == DH_SECTORS_TORUS_TRANSLATIONS && mode == DH_INDEX_RANK_FREE)
    return dh_fail(S->ctx, DH_E_ARG, "torus sets with magnetic translations have one row routine");
  S->rowMode = mode;
  return DH_OK;
}

extern "C" int dh_sector_set_blas_launch(dh_sector_set* S, int axpyGroupsPerCU, int64_t dotsRowsPerTile) {
  if (!S) return DH_E_ARG;
  if (axpyGroupsPerCU < 1 || axpyGroupsPerCU > 64) return dh_fail(S->ctx, DH_E_ARG, "axpy groups per CU in [1, 64]");
  if (dotsRowsPerTile < 0 || (dotsRowsPerTile && dotsRowsPerTile < 256))
    return dh_fail(S->ctx, DH_E_ARG, "dots rows per tile: 0 (automatic) or >= 256");
  S->axpyGroupsPerCU = axpyGroupsPerCU;
  S->dotsRowsPerTile = dotsRowsPerTile;
  return DH_OK;
}

// work descriptor of the active sectors for tiles of `rowsPerTile` rows:
// d_work[0..na) = sector ids, d_work[na..2na] = tile prefix
int64_t dh_sectors_active_rows(const dh_sector_set* S, const unsigned char* active, int* nActive) {
  int64_t rows = 0;
  *nActive = 0;
  for (int s = 0; s < S->nbrSectors; ++s) {
    if (active && !active[s]) continue;
    rows += S->offsets[s + 1] - S->offsets[s];
    ++*nActive;
  }
  return rows;
}

int dh_sectors_upload_work(dh_sector_set* S, const unsigned char* active, int64_t rowsPerTile, int* nActive,
                       int64_t* totalTiles) {
  dh_context* c = S->ctx;
  std::vector<int64_t> w;
  std::vector<int64_t> prefix(1, 0);
  for (int s = 0; s < S->nbrSectors; ++s) {
    if (active && !active[s]) continue;
    w.push_back(s);
    int64_t d = S->offsets[s + 1] - S->offsets[s];
    prefix.push_back(prefix.back() + (d + rowsPerTile - 1) / rowsPerTile);
  }
  int na = (int)w.size();
  w.insert(w.end(), prefix.begin(), prefix.end());
  size_t bytes = sizeof(int64_t) * w.size();
  if (bytes > S->workCap) {
    if (S->d_work) {
      DH_HIP(c, hipStreamSynchronize(c->stream));
      hipFree(S->d_work);
    }
    S->d_work = nullptr;
    int rc = dh_alloc(c, (void**)&S->d_work, std::max<size_t>(bytes, 4096));
    if (rc) return rc;
    S->workCap = std::max<size_t>(bytes, 4096);
  }
  int rc = dh_upload_async(c, S->d_work, w.data(), bytes);
  if (rc) return rc;
  *nActive = na;
  *totalTiles = prefix.back();
  return DH_OK;
}

struct SectorsArgs {
  const uint64_t* states;
  const int64_t* offsets;
  int nbrOrbitals, nbrFactors, nbrSums;  // packed factors and their per-sum bases
  const double* factors;
  const int* sumBase;
  const uint32_t* rankLo;
  const uint32_t* rankHi;
  const uint16_t* rankLo16;  // the low table in 16 bits, staged in LDS (LO_LDS)
  int rankBits;
  int64_t loSize, hiSize;
  double shift;
  const int64_t* work;  // active ids then prefix
  int nActive;
  int64_t totalTiles;
};

// tile -> position j in the active list (prefix in LDS)
__device__ __forceinline__ int tile_sector(const int64_t* sPrefix, int nActive, int64_t tile) {
  int lo = 0, hi = nActive;  // sPrefix[lo] <= tile < sPrefix[hi]
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (sPrefix[mid] <= tile)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// S32: the orbitals fit a 32-bit word, so the row routine runs on 32-bit state words (used for
// k <= 2).  Every sector has fewer than 2^31 states (the set refuses larger ones), so indices are
// 32-bit in both forms.
// FREE: the created pairs come from the set bits of the free-pair masks (dh_sphere_row).
// TRI: the factor matrices are triangles (dh_pack_sphere_factors).
// TABLES: the rank tables in LDS: 0 none, 1 the low one (16 bits), 2 the sector's high one too, staged when
// a workgroup's tiles enter a sector.
template <int K, int LPR, int TABLES, bool S32, bool FREE, bool TRI>
__global__ void __launch_bounds__(1024) sectors_hv_kernel(SectorsArgs a, const double* __restrict__ x,
                                                          double* __restrict__ y, int add) {
  extern __shared__ double smem[];
  double* sF = smem;
  int* sBase = reinterpret_cast<int*>(sF + a.nbrFactors);
  int64_t* sWork = reinterpret_cast<int64_t*>(smem) + ((a.nbrFactors * 8 + a.nbrSums * 4 + 7) / 8);
  uint16_t* sLo = reinterpret_cast<uint16_t*>(sWork + 2 * a.nActive + 1);
  for (int i = threadIdx.x; i < a.nbrFactors; i += blockDim.x) sF[i] = a.factors[i];
  for (int i = threadIdx.x; i < a.nbrSums; i += blockDim.x) sBase[i] = a.sumBase[i];
  for (int i = threadIdx.x; i < 2 * a.nActive + 1; i += blockDim.x) sWork[i] = a.work[i];
  uint32_t* sHi = reinterpret_cast<uint32_t*>(sLo + a.loSize);
  if constexpr (TABLES > 0)
    for (int i = threadIdx.x; i < a.loSize; i += blockDim.x) sLo[i] = a.rankLo16[i];
  __syncthreads();
  int staged = -1;  // the sector whose high table is in LDS
  // the low table: 16-bit copy in LDS, or the 32-bit table in global memory
  auto loAt = [&](uint32_t i) -> uint32_t {
    if constexpr (TABLES > 0)
      return sLo[i];
    else
      return a.rankLo[i];
  };
  const int64_t* sPrefix = sWork + a.nActive;
  const int lane = threadIdx.x % LPR;
  const int64_t rowsPerTile = blockDim.x / LPR;
  for (int64_t tile = dh_xcd_block(blockIdx.x, gridDim.x); tile < a.totalTiles; tile += gridDim.x) {
    const int j = tile_sector(sPrefix, a.nActive, tile);
    const int sec = (int)sWork[j];
    if constexpr (TABLES == 2) {
      if (sec != staged) {
        __syncthreads();  // the last tile's lookups are done
        for (int i = threadIdx.x; i < a.hiSize; i += blockDim.x) sHi[i] = a.rankHi[(int64_t)sec * a.hiSize + i];
        __syncthreads();
        staged = sec;
      }
    }
    const int64_t off = a.offsets[sec];
    const int64_t dim = a.offsets[sec + 1] - off;
    const uint32_t* hi;
    if constexpr (TABLES == 2)
      hi = sHi;
    else
      hi = a.rankHi + (int64_t)sec * a.hiSize;
    const int64_t local = (tile - sPrefix[j]) * rowsPerTile + threadIdx.x / LPR;
    const bool active = local < dim;
    const int64_t g = off + (active ? local : 0);
    const uint64_t s = active ? a.states[g] : 0ull;
    double acc[K];
#pragma unroll
    for (int v = 0; v < K; ++v) acc[v] = 0.0;
    dh_diagonal diag;
    if constexpr (S32) {
      const uint32_t last = (uint32_t)dim - 1u, mask = (1u << a.rankBits) - 1u;
      const int bits = a.rankBits;
      auto find = [&](uint32_t t) -> uint32_t { return dh_rank_of<false>(t, [&] { return loAt(t & mask); }, hi, bits, last); };
      diag = dh_sphere_row<K, LPR, FREE, TRI>((uint32_t)s, a.nbrOrbitals, sF, sBase, lane, find, x + off * K, acc);
    } else {
      // rankBits = ceil(orbitals / 2) <= 32, so t >> bits fits 32 bits
      const uint32_t last = (uint32_t)dim - 1u;
      const uint32_t mask = a.rankBits >= 32 ? 0xffffffffu : (1u << a.rankBits) - 1u;
      const int bits = a.rankBits;
      auto find = [&](uint64_t t) -> uint32_t {
        return dh_rank_of<dh_far_tables<uint64_t, (TABLES > 0)>>(
            t, [&] { return loAt((uint32_t)t & mask); }, hi, bits, last);
      };
      diag = dh_sphere_row<K, LPR, FREE, TRI>(s, a.nbrOrbitals, sF, sBase, lane, find, x + off * K, acc);
    }
    if constexpr (LPR > 1) {
#pragma unroll
      for (int v = 0; v < K; ++v)
        for (int o = LPR / 2; o > 0; o >>= 1) acc[v] += __shfl_xor(acc[v], o, LPR);
    }
    if (active && lane == 0) {
      const double* xr = x + g * K;
      double* yr = y + g * K;
#pragma unroll
      for (int v = 0; v < K; ++v) yr[v] = (add ? yr[v] : 0.0) + diag.term(xr[v], acc[v]) + a.shift * xr[v];
    }
  }
}

static SectorsArgs sectors_args(dh_sector_set* S, int nActive, int64_t totalTiles) {
  SectorsArgs a;
  a.states = S->d_states;
  a.offsets = S->d_offsets;
  a.nbrOrbitals = S->nbrOrbitals;
  a.nbrFactors = S->nbrPackedFactors;
  a.nbrSums = S->nbrPairSums;
  a.factors = S->d_packedFactors;
  a.sumBase = S->d_sumBase;
  a.rankLo = S->d_rankLo;
  a.rankHi = S->d_rankHi;
  a.rankLo16 = S->d_rankLo16;
  a.rankBits = S->rankBits;
  a.loSize = S->loSize;
  a.hiSize = S->hiSize;
  a.shift = S->shift;
  a.work = S->d_work;
  a.nActive = nActive;
  a.totalTiles = totalTiles;
  return a;
}

// Dynamic LDS for `na` active sectors and workgroups of bs threads: the packed factors and the work list,
// with the rank tables that go there (TABLES of the kernel): the low one while two workgroups' tables fit a
// CU, and the high one too while two still fit (up to 26 orbitals) or one that fills the CU (27 and 28
// orbitals, 1024 threads).  The high table's gathers are half of those that bound the product in the L1:
// 1.0 M rows on 25 orbitals 214 -> 201 us, k = 8 948 -> 811; 6.7 M rows on 28 orbitals 1595 -> 1549 us, k = 2
// 2228 -> 1706, k = 8 8605 -> 7032.
static size_t sectors_lds(const dh_sector_set* S, int na, int bs, int* tables) {
  const size_t base = ((size_t)S->nbrPackedFactors * 8 + (size_t)S->nbrPairSums * 4 + 7) / 8 * 8 + 8 * (2 * na + 1);
  const size_t lo = base + 2 * S->loSize, both = lo + 4 * S->hiSize;
  *tables = 0;
  if (!S->d_rankLo16) return base;
  if (both <= 79 * 1024 || (both <= 160 * 1024 && bs == 1024)) {
    *tables = 2;
    return both;
  }
  if (lo > 79 * 1024) return base;
  *tables = 1;
  return lo;
}

template <int K, int LPR>
static int sectors_hv_launch(dh_sector_set* S, int blockSize, bool freePairs, const double* x, double* y, int add,
                             const unsigned char* active) {
  dh_context* c = S->ctx;
  int64_t rowsPerTile = blockSize / LPR;
  int na;
  int64_t tiles;
  int rc = dh_sectors_upload_work(S, active, rowsPerTile, &na, &tiles);
  if (rc) return rc;
  if (tiles == 0) return DH_OK;
  int tables;
  const size_t lds = sectors_lds(S, na, blockSize, &tables);
  if (lds > 160 * 1024) return dh_fail(c, DH_E_RANGE, "staged tables exceed LDS");
  SectorsArgs a = sectors_args(S, na, tiles);
  auto launch = [&](auto kern) -> int {
    if (lds > 64 * 1024)
      DH_HIP(c, hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int perCU = dh_blocks_per_cu(c, kern, blockSize, lds);
    int64_t grid = std::max<int64_t>(1, std::min<int64_t>(tiles, (int64_t)c->nbrCU * perCU));
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(blockSize), lds, c->stream, a, x, y, add);
    DH_HIP(c, hipGetLastError());
    return DH_OK;
  };
  // 32-bit words for one or two vectors, where the integer work of the row routine dominates; for
  // more vectors the 64-bit form is faster on MI355X (its lower occupancy keeps more of the x
  // gathers in cache: 11.3 against 16.5 ms at k = 8 over the 91 sectors of N=10 2S=27)
  const bool s32 = K <= 2 && S->nbrOrbitals <= 32;
  auto pick = [&](auto lo, auto tri) -> int {
    constexpr int LO = decltype(lo)::value;
    constexpr bool TRI = decltype(tri)::value;
    if (freePairs)
      return s32 ? launch(sectors_hv_kernel<K, LPR, LO, (K <= 2), true, TRI>)
                 : launch(sectors_hv_kernel<K, LPR, LO, false, true, TRI>);
    return s32 ? launch(sectors_hv_kernel<K, LPR, LO, (K <= 2), false, TRI>)
               : launch(sectors_hv_kernel<K, LPR, LO, false, false, TRI>);
  };
  auto where = [&](auto tri) -> int {
    switch (tables) {
      case 0: return pick(std::integral_constant<int, 0>{}, tri);
      case 1: return pick(std::integral_constant<int, 1>{}, tri);
      default: return pick(std::integral_constant<int, 2>{}, tri);
    }
  };
  return S->triangles ? where(std::true_type{}) : where(std::false_type{});
}

// What a launch shape costs the sectors of a product, in passes of one wavefront over its rows, from the
// workgroups that fit a CU and the rounds that the tiles take: up to 16 wavefronts a CU run together, more share
// its units; a second lane saves 30 % of a pass; with the high rank table in L2 a pass takes 15 % longer.
// Ranks 190 measured products of 30 k to 500 k rows within 8 % of their fastest shape on average.
static double sectors_rounds(const dh_sector_set* S, const unsigned char* active, int na, int lanes, int bs) {
  int tables;
  const size_t lds = sectors_lds(S, na, bs, &tables);
  const int64_t cus = S->ctx->nbrCU, fit = std::max<int64_t>(1, std::min<int64_t>(160 * 1024 / lds, 2048 / bs));
  int64_t tiles = 0;
  for (int s = 0; s < S->nbrSectors; ++s)
    if (!active || active[s]) tiles += ((S->offsets[s + 1] - S->offsets[s]) * lanes + bs - 1) >> __builtin_ctz(bs);
  auto pass = [&](int64_t groups) { return std::max(1.0, groups * (bs / 64) / 16.0); };
  const int64_t full = tiles / (cus * fit), rest = tiles - full * cus * fit;
  const double rounds = full * pass(fit) + (rest ? pass((rest + cus - 1) / cus) : 0.0);
  return rounds * (lanes == 1 ? 1.0 : 0.7) * (tables == 2 ? 1.0 : 1.15);
}

// Lanes per row, workgroup size and row routine by rows per CU, k and the bytes of the staged tables, times in us on
// MI355X.  Few rows: eight lanes and the range loop, whose rows finish together (4173 rows: 14.7, 15.7 with 2 x
// 256 and the masks; k = 4 16.8 and 17.8); large tables are staged by 512 threads, as for a single space (1300
// rows on 26 orbitals 15.2, 18.7 with 256; k = 8, 7680 rows 20.4, 24.2).  Then lanes for wavefronts (26 k rows:
// 19.3 with 2 x 256, 21.5 with 1 x 256; k = 16 43.5 with 4 x 256, 49.9 with 2).  From 128 to 2048 rows a CU small
// workgroups spread best (164 k rows: 35.4 with 1 x 256, 40 with 1 x 512 and 1 x 1024; k = 4: 55 with 2 x 256, 60
// with 1 x 512, 71 by ranges; k = 8: 99, 125 by ranges; k = 16: 285 with 4 x 256, 375 with 2 x 512 by ranges).
// Where three of them at most fit a CU, one of another shape that sectors_rounds puts 25 % below is taken (246 k
// rows on 28 orbitals 71.7 with 1 x 1024, 134 with 1 x 256, k = 4 143 and 238; 329 k rows on 26 67 and 85; for
// k = 8 only from 900 rows a CU, 192 k rows 127 with 2 x 256 and 137 with 2 x 1024).
// Above, the tables in LDS bound the
// wavefronts of a CU: 1024 threads (1.0 M rows: 188, 232 at 256; 17.6 M rows with 29 orbitals: 5.4 ms, 8.4 at
// 512, 14.0 at 256), 512 once x outgrows the 256 MB behind the L2s and the gathers go to HBM (278 M rows: 191
// ms, 211 at 1024), for k = 4 512 when three workgroups fit (1.0 M rows, 25 orbitals: 314, 336 at 1024, 425 by
// ranges), and with both rank tables in L2 two lanes (1.7 M rows on 39 orbitals 706, 892 with one; k = 4 988
// and 1073).  k = 8: two lanes, 1024 threads where one workgroup's tables fill a CU (6.7 M rows: 6.0 ms, 7.0 with
// 2 x 512), 512 where more fit (1.0 M rows: 676, 725 at 1024), one lane with the high table in L2 (17.6 M rows
// 22.3 ms, 23.7 with two).  k = 16: two lanes, 512, and by ranges (2139, 2242 with the masks).
//
// The rows are those of the product's sectors: late in a batched solve few of them are still active (one sector
// of the set of 7 on 37 orbitals, 20 k of 5.2 M rows: 34 us, 98 with the set's shape).
static void sectors_shape(const dh_sector_set* S, int k, const unsigned char* active, int* lpr, int* bs,
                          bool* freePairs) {
  *lpr = S->lanesPerRow;
  *bs = S->blockSize;
  // DH_INDEX_RANK in a chosen shape: the free-pair masks for k <= 2, as for a single space
  *freePairs = S->rowMode == DH_INDEX_RANK_FREE || (S->rowMode == DH_INDEX_RANK && k <= 2);
  if (!S->autoLaunch) return;
  int na, tables;
  const int64_t rows = dh_sectors_active_rows(S, active, &na), perCU = rows / S->ctx->nbrCU;
  const size_t staged = sectors_lds(S, na, 256, &tables);
  bool masks = true;
  auto set = [&](int l, int b) { *lpr = l, *bs = b; };
  if (perCU < 32) {
    set(8, k <= 4 ? (staged > 16 * 1024 ? 512 : 256) : k == 8 && tables && staged > 40 * 1024 ? 512 : 256);
    masks = false;
  } else if (perCU < 128) {
    set(k == 16 ? 4 : 2, 256);
  } else if (perCU < 2048) {
    set(k <= 2 ? 1 : k == 16 ? 4 : 2, 256);
    if (tables && staged > 40 * 1024 && (k <= 4 || (k == 8 && perCU >= 900))) {
      const double small = sectors_rounds(S, active, na, *lpr, 256);
      double best = small / 1.25;
      for (int l = k == 8 ? 2 : 1; l <= 2; ++l)
        for (int b = 256; b <= 1024; b *= 2) {
          const double t = sectors_rounds(S, active, na, l, b);
          if (t <= best) best = t, set(l, b);
        }
    }
  } else if (k == 16) {
    set(2, 512);
    masks = false;
  } else if (!tables && k <= 4) {
    set(2, 1024);
  } else {
    const bool three = 3 * sectors_lds(S, na, 512, &tables) <= 160 * 1024;
    const bool oneFills = sectors_lds(S, na, 1024, &tables) > 79 * 1024 && tables == 2;
    if (k <= 2)
      set(1, rows * k <= (int64_t)1 << 25 ? 1024 : 512);
    else if (k == 4)
      set(1, three && !oneFills ? 512 : 1024);
    else
      oneFills ? set(2, 1024) : set(tables == 2 ? 2 : 1, 512);
  }
  if (S->rowMode == DH_INDEX_RANK) *freePairs = masks;
}

template <int K>
static int sectors_hv_lpr(dh_sector_set* S, const double* x, double* y, int add, const unsigned char* active) {
  int lpr, bs;
  bool freePairs;
  sectors_shape(S, K, active, &lpr, &bs, &freePairs);
  switch (lpr) {
    case 1: return sectors_hv_launch<K, 1>(S, bs, freePairs, x, y, add, active);
    case 2: return sectors_hv_launch<K, 2>(S, bs, freePairs, x, y, add, active);
    case 4: return sectors_hv_launch<K, 4>(S, bs, freePairs, x, y, add, active);
    default: return sectors_hv_launch<K, 8>(S, bs, freePairs, x, y, add, active);
  }
}

extern "C" int dh_sectors_hv(dh_sector_set* S, const double* x, double* y, int k, int add,
                             const unsigned char* active) {
  if (!S || !x || !y) return DH_E_ARG;
  if (S->kind == DH_SECTORS_MOMENTUM) return dh_lattice_sectors_hv(S, x, y, k, add, active);
  if (S->kind == DH_SECTORS_TORUS_TRANSLATIONS) return dh_torus_translation_sectors_hv(S, x, y, k, add, active);
  if (!S->d_factors) return dh_fail(S->ctx, DH_E_STATE, "factors not set");
  switch (k) {
    case 1: return sectors_hv_lpr<1>(S, x, y, add, active);
    case 2: return sectors_hv_lpr<2>(S, x, y, add, active);
    case 4: return sectors_hv_lpr<4>(S, x, y, add, active);
    case 8: return sectors_hv_lpr<8>(S, x, y, add, active);
    case 16: return sectors_hv_lpr<16>(S, x, y, add, active);
    default: return dh_fail(S->ctx, DH_E_ARG, "k must be 1, 2, 4, 8 or 16");
  }
}

// ----------------------------------------------------------------------------- segmented BLAS
// dots: partial[tile][b*KK + i] over the tile's rows, reduced per active sector afterwards
template <int K, int G>
__global__ void __launch_bounds__(256) sectors_dots_kernel(const double* __restrict__ V, int nbrBlocks,
                                                           int64_t totalDim, const double* __restrict__ W,
                                                           const int64_t* __restrict__ offsets,
                                                           const int64_t* __restrict__ work, int nActive,
                                                           int64_t rowsPerTile, double* __restrict__ partial,
                                                           bool pairs) {
  constexpr int KK = K * K;
  __shared__ double red[256 / 64][G * KK];  // dh_dots_tile's per-wavefront sums
  const int64_t tile = blockIdx.y;  // blocks of one tile are adjacent: its W rows stay in L2
  const int64_t* prefix = work + nActive;
  int lo = 0, hi = nActive;
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (prefix[mid] <= tile) lo = mid; else hi = mid;
  }
  const int sec = (int)work[lo];
  const int64_t off = offsets[sec], dim = offsets[sec + 1] - off;
  const int64_t r0 = (tile - prefix[lo]) * rowsPerTile;
  const int64_t r1 = min(dim, r0 + rowsPerTile);
  const int b0 = blockIdx.x * G;
  const int64_t total = (int64_t)nbrBlocks * KK;
  dh_dots_tile<K, G>(V, totalDim * K, nbrBlocks, b0, W, off + r0, off + r1, &red[0][0],
                     partial + tile * total + (int64_t)b0 * KK, pairs);
}

__global__ void sectors_reduce_kernel(const double* __restrict__ partial, const int64_t* __restrict__ work,
                                      int nActive, int64_t total, double* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int j = blockIdx.y;
  if (i >= total) return;
  const int64_t* prefix = work + nActive;
  double s = 0.0;
  for (int64_t t = prefix[j]; t < prefix[j + 1]; ++t) s += partial[t * total + i];
  out[(int64_t)j * total + i] = s;
}

template <int K>
static int sectors_dots(dh_sector_set* S, const double* V, int nb, const double* W, const unsigned char* active,
                        double* h_out) {
  dh_context* c = S->ctx;
  constexpr int G = DotsGroup<K>::value;
  // automatic tile: at least 8192 rows (4096 for k >= 4, whose one-block workgroups are few:
  // 3.9-4.0 against 2.5-3.6 TB/s at k = 8 over the 91 sectors of N=10 2S=27), and no more
  // than about 32768 tiles
  const int64_t rowsPerTile = S->dotsRowsPerTile
                                  ? S->dotsRowsPerTile
                                  : std::max<int64_t>(K >= 4 ? 4096 : 8192, (S->totalDim + 32767) / 32768);
  int na;
  int64_t tiles;
  int rc = dh_sectors_upload_work(S, active, rowsPerTile, &na, &tiles);
  if (rc) return rc;
  if (tiles == 0) return DH_OK;
  const int64_t total = (int64_t)nb * K * K;
  double* scratch;
  if ((rc = dh_scratch(c, sizeof(double) * (size_t)(tiles * total + (int64_t)na * total), &scratch))) return rc;
  double* d_out = scratch + tiles * total;
  dim3 grid((unsigned)((nb + G - 1) / G), (unsigned)tiles);
  hipLaunchKernelGGL((sectors_dots_kernel<K, G>), grid, dim3(256), 0, c->stream, V, nb, S->totalDim, W, S->d_offsets,
                     S->d_work, na, rowsPerTile, scratch, K == 1 && dh_pairs_aligned(V, S->totalDim, W));
  hipLaunchKernelGGL(sectors_reduce_kernel, dim3((unsigned)((total + 255) / 256), (unsigned)na), dim3(256), 0,
                     c->stream, scratch, S->d_work, na, total, d_out);
  DH_HIP(c, hipGetLastError());
  double* pin;
  if ((rc = dh_pinned(c, sizeof(double) * na * total, &pin))) return rc;
  DH_HIP(c, hipMemcpyAsync(pin, d_out, sizeof(double) * na * total, hipMemcpyDeviceToHost, c->stream));
  DH_HIP(c, hipStreamSynchronize(c->stream));
  std::memcpy(h_out, pin, sizeof(double) * na * total);
  return DH_OK;
}

extern "C" int dh_sectors_block_dots(dh_sector_set* S, const double* V, int nb, const double* W, int k,
                                     const unsigned char* active, double* out) {
  if (!S || !V || !W || !out || nb <= 0) return DH_E_ARG;
  switch (k) {
    case 1: return sectors_dots<1>(S, V, nb, W, active, out);
    case 2: return sectors_dots<2>(S, V, nb, W, active, out);
    case 4: return sectors_dots<4>(S, V, nb, W, active, out);
    case 8: return sectors_dots<8>(S, V, nb, W, active, out);
    case 16: return sectors_dots<16>(S, V, nb, W, active, out);
    default: return dh_fail(S->ctx, DH_E_ARG, "k must be 1, 2, 4, 8 or 16");
  }
}

// axpy / rmul: W[row][q] (+)= sum over (b, p) of V_b[row][p] C_j[(b*K+p)*K+q]; rmul uses W itself.
// The coefficients sit in LDS in slabs of `slab` basis blocks (dynamic LDS of slab * K * K
// doubles, so short bases leave room for more workgroups per CU). Basis rows are read U blocks at
// a time, so one lane keeps U independent loads in flight; at k = 1 with the nontemporal hint (each
// basis row is read once per pass).
template <int K, bool RMUL>
__global__ void __launch_bounds__(256) sectors_axpy_kernel(const double* __restrict__ V, int nb, int64_t totalDim,
                                                           double* __restrict__ W,
                                                           const int64_t* __restrict__ offsets,
                                                           const int64_t* __restrict__ work, int nActive,
                                                           int64_t totalTiles, int slab, const double* __restrict__ C) {
  constexpr int KK = K * K;
  constexpr int U = K == 1 ? 8 : (K == 2 ? 4 : (K == 4 ? 2 : 1));
  extern __shared__ double sC[];
  const int64_t* prefix = work + nActive;
  const int64_t stride = totalDim * K;
  // each workgroup walks a contiguous range of tiles, so it stays in one sector for many tiles:
  // the sector is found by advancing through the prefix, and a coefficient matrix that fits one
  // LDS slab is loaded only when the sector changes
  const int64_t first = totalTiles * blockIdx.x / gridDim.x, last = totalTiles * (blockIdx.x + 1) / gridDim.x;
  int lo = 0;
  while (lo + 1 < nActive && prefix[lo + 1] <= first) ++lo;
  int staged = -1;
  for (int64_t tile = first; tile < last; ++tile) {
    while (prefix[lo + 1] <= tile) ++lo;
    const int sec = (int)work[lo];
    const int64_t off = offsets[sec], dim = offsets[sec + 1] - off;
    const int64_t r = (tile - prefix[lo]) * blockDim.x + threadIdx.x;
    const bool active = r < dim;
    const int64_t row = off + (active ? r : 0);
    const double* Cj = C + (int64_t)lo * nb * KK;
    double acc[K];
#pragma unroll
    for (int q = 0; q < K; ++q) acc[q] = 0.0;
    for (int s0 = 0; s0 < nb; s0 += slab) {
      const int ns = min(slab, nb - s0);
      if (nb > slab || staged != lo) {
        __syncthreads();
        for (int i = threadIdx.x; i < ns * KK; i += blockDim.x) sC[i] = Cj[(int64_t)s0 * KK + i];
        __syncthreads();
        staged = lo;
      }
      if (active) {
        const double* vb = (RMUL ? W : V + (int64_t)s0 * stride) + row * K;
        int b = 0;
        for (; b + U <= ns; b += U) {
          double v[U][K];
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < K; ++p) v[u][p] = (RMUL || K > 1) ? vb[(int64_t)(b + u) * stride + p]
                                                                  : dh_stream_load(vb + (int64_t)(b + u) * stride + p);
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int p = 0; p < K; ++p)
#pragma unroll
              for (int q = 0; q < K; ++q) acc[q] += v[u][p] * sC[(b + u) * KK + p * K + q];
        }
        for (; b < ns; ++b) {
#pragma unroll
          for (int p = 0; p < K; ++p) {
            const double v = (RMUL || K > 1) ? vb[(int64_t)b * stride + p] : dh_stream_load(vb + (int64_t)b * stride + p);
#pragma unroll
            for (int q = 0; q < K; ++q) acc[q] += v * sC[b * KK + p * K + q];
          }
        }
      }
    }
    if (active) {
#pragma unroll
      for (int q = 0; q < K; ++q) {
        if (RMUL)
          W[row * K + q] = acc[q];
        else
          W[row * K + q] += acc[q];
      }
    }
  }
}

template <int K, bool RMUL>
static int sectors_axpy(dh_sector_set* S, const double* V, int nb, double* W, const unsigned char* active,
                        const double* h_c) {
  dh_context* c = S->ctx;
  int na;
  int64_t tiles;
  int rc = dh_sectors_upload_work(S, active, 256, &na, &tiles);
  if (rc) return rc;
  if (tiles == 0) return DH_OK;
  size_t bytes = sizeof(double) * (size_t)na * nb * K * K;
  if (bytes > S->coefCap) {
    if (S->d_coef) {
      DH_HIP(c, hipStreamSynchronize(c->stream));
      hipFree(S->d_coef);
    }
    S->d_coef = nullptr;
    if ((rc = dh_alloc(c, (void**)&S->d_coef, bytes))) return rc;
    S->coefCap = bytes;
  }
  if ((rc = dh_upload_async(c, S->d_coef, h_c, bytes))) return rc;
  // LDS slab: the whole coefficient block when it fits 32 KiB, else 32 KiB pieces
  const int slab = std::min(nb, std::max(1, 4096 / (K * K)));
  const size_t lds = sizeof(double) * (size_t)slab * K * K;
  int64_t grid = std::min<int64_t>(tiles, (int64_t)c->nbrCU * S->axpyGroupsPerCU);
  hipLaunchKernelGGL((sectors_axpy_kernel<K, RMUL>), dim3((unsigned)grid), dim3(256), lds, c->stream, V, nb,
                     S->totalDim, W, S->d_offsets, S->d_work, na, tiles, slab, S->d_coef);
  DH_HIP(c, hipGetLastError());
  return DH_OK;
}

extern "C" int dh_sectors_block_axpy(dh_sector_set* S, const double* V, int nb, double* W, int k,
                                     const unsigned char* active, const double* coef) {
  if (!S || !V || !W || !coef || nb <= 0) return DH_E_ARG;
  switch (k) {
    case 1: return sectors_axpy<1, false>(S, V, nb, W, active, coef);
    case 2: return sectors_axpy<2, false>(S, V, nb, W, active, coef);
    case 4: return sectors_axpy<4, false>(S, V, nb, W, active, coef);
    case 8: return sectors_axpy<8, false>(S, V, nb, W, active, coef);
    case 16: return sectors_axpy<16, false>(S, V, nb, W, active, coef);
    default: return dh_fail(S->ctx, DH_E_ARG, "k must be 1, 2, 4, 8 or 16");
  }
}

extern "C" int dh_sectors_block_rmul(dh_sector_set* S, double* W, int k, const unsigned char* active,
                                     const double* m) {
  if (!S || !W || !m) return DH_E_ARG;
  switch (k) {
    case 1: return sectors_axpy<1, true>(S, W, 1, W, active, m);
    case 2: return sectors_axpy<2, true>(S, W, 1, W, active, m);
    case 4: return sectors_axpy<4, true>(S, W, 1, W, active, m);
    case 8: return sectors_axpy<8, true>(S, W, 1, W, active, m);
    case 16: return sectors_axpy<16, true>(S, W, 1, W, active, m);
    default: return dh_fail(S->ctx, DH_E_ARG, "k must be 1, 2, 4, 8 or 16");
  }
}

extern "C" int64_t dh_sector_set_dimension(const dh_sector_set* S) { return S ? S->totalDim : -1; }
