// Spin-1/2 chain H.v by tiles: the rows of one pattern of the chain's first L - LO sites
// (SpinChainHamiltonian::LowLevelAddMultiply, Spin/src/Hamiltonian/SpinChainHamiltonian.cc:257).
//
// Site 0 is the most significant in the order of the states (up first), so a tile is one contiguous range
// of C(LO, n) rows, n the up spins among the last LO sites, in the order of the LO-site patterns with n up.
// Per tile, not per row: the antiparallel bonds among the first sites move the whole tile by one distance
// (coalesced reads of x), the bond between the two parts moves the rows of one value of its lower site by
// one distance, and the wrap bond goes to one other tile, at a rank that the pattern table holds.  Only the
// bonds among the last LO sites are per row, and their targets are in the tile: x of the tile is in LDS.
#include "dh_internal.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int kLoMin = 10, kLoMax = 14;
constexpr uint32_t kParallel = 0x80000000u;

constexpr uint32_t binom_c(int n, int k) {
  uint64_t v = 1;
  for (int i = 0; i < k; ++i) v = v * (n - i) / (i + 1);
  return (uint32_t)v;
}

// Tables of LO last sites: the 2^LO patterns by number of up spins, then in the order of the states (bits
// 0-15; bits 16-31: the rank of the pattern with its last site flipped among those of its number of up
// spins), and the distances [b][c][pair] that a flip of bond (b, b + 1) moves a row, c the up spins at bits
// >= b and pair its two bits (kParallel: no flip).
constexpr size_t tile_words(int lo) { return (size_t(1) << lo) + (size_t)(lo - 1) * 64; }
constexpr size_t tile_offset(int lo) {
  size_t o = 0;
  for (int l = kLoMin; l < lo; ++l) o += tile_words(l);
  return o;
}

__device__ uint32_t pattern_rank(uint32_t p, int lo, const uint32_t* __restrict__ binom) {
  uint32_t rank = 0;
  for (int j = 0; j < lo; ++j) {
    const int c = __popc(p >> j);  // a down site comes after the patterns with this site up
    if (!((p >> j) & 1u) && c > 0) rank += binom[(lo - 1 - j) * 33 + c - 1];
  }
  return rank;
}

// one row of workgroups per table, the last one for the zeros behind them
constexpr size_t kZeroWords = size_t(1) << kLoMax;

__global__ void spin_tile_table_kernel(uint32_t* __restrict__ out, const uint32_t* __restrict__ binom) {
  const int lo = kLoMin + blockIdx.y;
  uint32_t* table = out;
  for (int l = kLoMin; l < lo; ++l) table += tile_words(l);
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (lo > kLoMax) {
    table[i] = 0;
    return;
  }
  if (i < (1u << lo)) {
    const int n = __popc(i);
    uint32_t at = pattern_rank(i, lo, binom);
    for (int m = 0; m < n; ++m) at += binom[lo * 33 + m];
    table[at] = i | (pattern_rank(i ^ (1u << (lo - 1)), lo, binom) << 16);
  }
  if (i < (uint32_t)(lo - 1) * 64) {
    const int b = i >> 6, c = (i >> 2) & 15, pair = i & 3;
    uint32_t step = kParallel;
    if ((pair == 1 || pair == 2) && c > 0) {
      const uint32_t d = binom[(lo - 2 - b) * 33 + c - 1];
      step = pair == 1 ? d : 0u - d;
    }
    table[(1u << lo) + i] = step;
  }
}

struct SpinTileArgs {
  const uint32_t *table, *binom;
  const double* zeros;  // as many as a tile has
  int L, nbrUp, periodic;
  unsigned firstTile, endTile;
  unsigned chunk;  // consecutive tiles of one XCD
  double base;     // shift + a quarter of the bonds' Jz
  uint32_t classOff[kLoMax + 1];
  double halfJ[32], halfJz[32];
};

// A tile of one row (all of its last sites up, or all down), by its first K threads: no flips in the tile.
template <int K>
__device__ void spin_tile_row(const SpinTileArgs& a, int h, uint32_t start, uint32_t wrapRow, int delta, uint32_t P,
                              bool lastUp, const double* __restrict__ x, double* __restrict__ y, int add) {
  const int L = a.L, j = threadIdx.x;
  const uint32_t high = (P ^ (P >> 1)) & ((1u << (h - 1)) - 1u);
  double off = 0.0, diag = a.base;
  auto bond = [&](int i, uint32_t row) {
    diag -= a.halfJz[i];
    off += a.halfJ[i] * x[(size_t)row * K + (j < K ? j : 0)];
  };
  for (uint32_t m = high; m; m &= m - 1) {
    const int i = __builtin_ctz(m);
    bond(i, start + __builtin_amdgcn_readlane(delta, i));
  }
  if ((((P >> (h - 1)) & 1u) != 0) != lastUp) bond(h - 1, start + __builtin_amdgcn_readlane(delta, h - 1));
  if (a.periodic && ((P & 1u) != 0) != lastUp) bond(L - 1, wrapRow);
  if (j < K) {
    double* yr = y + (size_t)start * K + j;
    off += diag * x[(size_t)start * K + j];
    *yr = (add ? *yr : 0.0) + off;
  }
}

// two doubles, and two whose row starts at any multiple of 8 bytes (one vector)
typedef double Pair16 __attribute__((ext_vector_type(2)));
typedef double Pair8 __attribute__((ext_vector_type(2), aligned(8)));

// A thread takes Q neighbouring rows at a time, two for one vector: a wavefront's 8-byte loads take the L1
// nearly as many cycles as 16-byte ones.  Every read of a round is unconditional and issued before the work in
// LDS (bonds that are not there read zeros): behind branches each waited for the one before.
//
// By rows (spin_rank_kernel) a row takes 540 vector instructions a wavefront, 87 % of the time at 28 sites;
// by tiles 190, and the L1 (50 %), the vector units (47 %) and the LDS (24 %) share the time.  28 sites, 40 M
// rows: 658 us by rows, 454 by tiles, 129 for a copy of the vector; G = 4 instead of 2 460, 256 threads 485.
// 24 sites, open, different couplings, four vectors: 97 by rows, 76 by tiles.
template <int K, int LO, int BD, int G, bool UNIFORM>
__global__ void __launch_bounds__(BD) spin_tile_kernel(SpinTileArgs a, const double* __restrict__ x,
                                                       double* __restrict__ y, int add, int64_t first,
                                                       int64_t count) {
  constexpr int Q = K == 1 ? 2 : 1, D = Q * K / 2;  // rows and pairs of doubles of a thread
  constexpr uint32_t kRows = binom_c(LO, LO / 2), kBytes = 8 * K, kZero = kRows * kBytes;
  constexpr int kDoubles = kRows * K + Q * K;
  using Pair = typename std::conditional<K == 1, Pair8, Pair16>::type;
  __shared__ __align__(16) double sX[kDoubles];  // the tile's x, and zeros for the parallel bonds
  __shared__ uint32_t sStep[(LO - 1) * 64];      // in bytes of sX
  const int L = a.L, h = L - LO, lane = threadIdx.x & 63;
  // chunks of consecutive tiles go to the XCDs in turn: neighbours share an L2, and every XCD has its share
  // of the large tiles whatever the magnetisation
  const unsigned xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  const unsigned tile = a.firstTile + ((at / a.chunk) * 8 + xcd) * a.chunk + at % a.chunk;
  if (tile >= a.endTile) return;
  const uint32_t P = ~(__brev(tile) >> (32 - h)) & ((1u << h) - 1u);
  const int n = a.nbrUp - __popc(P);
  if (n < 0 || n > LO) return;
  // lane i < h: site i's part of the tile's first row, and the distance of the flip of bond (i, i + 1)
  const int up = (P >> (lane & 31)) & 1, c = __popc(P >> (lane & 31)) + n;
  const bool site = lane < h;
  uint32_t start = site && !up && c > 0 ? a.binom[(L - 1 - lane) * 33 + c - 1] : 0;
  int delta = site && c > 0 ? (int)a.binom[(L - 2 - lane) * 33 + c - 1] : 0;
  // the tile across the wrap bond: site 0 flipped, n2 up among the last sites
  const int up0 = P & 1, n2 = up0 ? n + 1 : n - 1;
  const bool wraps = a.periodic && n2 >= 0 && n2 <= LO;
  const int up2 = lane == 0 ? !up : up, c2 = lane == 0 ? c : c + n2 - n;
  uint32_t wstart = wraps && site && !up2 && c2 > 0 ? a.binom[(L - 1 - lane) * 33 + c2 - 1] : 0;
  const int size = (int)a.binom[LO * 33 + n];
  const int nUpFirst = n > 0 ? (int)a.binom[(LO - 1) * 33 + n - 1] : 0;  // rows with the first of the LO sites up
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) start += __shfl_xor(start, o, 32);
  start = __builtin_amdgcn_readfirstlane(start);
  const int64_t row0 = start;
  int begin = (int)max((int64_t)0, first - row0), end = (int)min((int64_t)size, first + count - row0);
  if (gridDim.y > 1) {  // a range of few tiles: several workgroups share a tile's rows
    const int share = (end - begin + (int)gridDim.y - 1) / (int)gridDim.y;
    begin += (int)blockIdx.y * share;
    end = min(end, begin + share);
  }
  if (begin >= end) return;
  if (!up) delta = -delta;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) wstart += __shfl_xor(wstart, o, 32);
  wstart = __builtin_amdgcn_readfirstlane(wstart);
  const uint32_t* patterns = a.table + a.classOff[n];
  if (size == 1) return spin_tile_row<K>(a, h, start, wstart + (patterns[0] >> 16), delta, P, n != 0, x, y, add);
  const double* xt = x + (size_t)start * K;
  // the thread's part of the tile, of the distances and its first patterns in flight at once
  constexpr int kPairs = kRows * K / 2, kLoads = (kPairs + BD - 1) / BD, kSteps = ((LO - 1) * 64 + BD - 1) / BD;
  const int pairs = size * K / 2;
  Pair own[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int e = i * BD + (int)threadIdx.x;
    own[i] = Pair{0.0, 0.0};
    if (e < pairs) own[i] = reinterpret_cast<const Pair*>(xt)[e];
  }
  double lastOwn = xt[size * K - 1];  // an odd number of doubles
  uint32_t step[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) step[i] = a.table[(1u << LO) + min(i * BD + (int)threadIdx.x, (LO - 1) * 64 - 1)];
  uint32_t eNext[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) eNext[q] = patterns[min(begin + Q * (int)threadIdx.x, size - Q) + q];
  const uint32_t high = (P ^ (P >> 1)) & ((1u << (h - 1)) - 1u);
  const int upLast = (P >> (h - 1)) & 1;
  const int crossDelta = __builtin_amdgcn_readlane(delta, h - 1);
  const double halfJ0 = a.halfJ[0];
  double diagHigh = a.base;
  if constexpr (UNIFORM)
    diagHigh -= a.halfJz[0] * (double)__popc(high);
  else
    for (uint32_t m = high; m; m &= m - 1) diagHigh -= a.halfJz[__builtin_ctz(m)];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int e = i * BD + (int)threadIdx.x;
    if (e < pairs) reinterpret_cast<double2*>(sX)[e] = make_double2(own[i].x, own[i].y);
  }
  if (2 * pairs < size * K && threadIdx.x == 0) sX[size * K - 1] = lastOwn;
  if (threadIdx.x < Q * K) sX[kZero / 8 + threadIdx.x] = 0.0;
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    const int e = i * BD + (int)threadIdx.x;
    if (e < (LO - 1) * 64) sStep[e] = step[i] == kParallel ? kParallel : step[i] * kBytes;
  }
  __syncthreads();
  // the same rounds for every thread (lane i holds bond i's distance)
  for (int rb = begin; rb < end; rb += Q * BD) {
    const int mine = rb + Q * (int)threadIdx.x;
    const int r = min(mine, size - Q);  // past the end: the last rows again, not stored
    // the next G bonds among the first sites; where there are no more, zeros
    Pair vh[G][D];
    uint32_t m = high;
    auto whole = [&] {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int i = m ? __builtin_ctz(m) : 0;
        const double* xb = m ? xt + (int64_t)__builtin_amdgcn_readlane(delta, i) * K : a.zeros;
        m &= m - 1;
#pragma unroll
        for (int j = 0; j < D; ++j) vh[g][j] = reinterpret_cast<const Pair*>(xb + r * K)[j];
      }
    };
    uint32_t left = high;
    whole();
    uint32_t e[Q];
    bool cross[Q], wrap[Q];
    double vc[Q * K], vw[Q * K];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int rq = r + q;
      e[q] = eNext[q];
      cross[q] = (rq < nUpFirst) != (upLast != 0);
      wrap[q] = a.periodic && ((e[q] >> (LO - 1)) & 1u) != (uint32_t)up0;
      const double* pc = xt + (int64_t)(rq + (cross[q] ? crossDelta : 0)) * K;
      const double* pw = x + (size_t)(wrap[q] ? wstart + (e[q] >> 16) : start + rq) * K;
#pragma unroll
      for (int j = 0; j < K; ++j) vc[q * K + j] = pc[j];
#pragma unroll
      for (int j = 0; j < K; ++j) vw[q * K + j] = pw[j];
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) eNext[q] = patterns[min(mine + Q * BD, size - Q) + q];
    double acc[Q * K];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint32_t p = e[q] & 0xffffu, flips = (p ^ (p >> 1)) & ((1u << (LO - 1)) - 1u);
      double diag = diagHigh;
      if constexpr (UNIFORM) {
        diag -= a.halfJz[0] * (double)(__popc(flips) + (cross[q] ? 1 : 0) + (wrap[q] ? 1 : 0));
      } else {
#pragma unroll
        for (int b = 0; b < LO - 1; ++b)
          if ((flips >> b) & 1u) diag -= a.halfJz[h + b];
        if (cross[q]) diag -= a.halfJz[h - 1];
        if (wrap[q]) diag -= a.halfJz[L - 1];
      }
      const uint32_t at0 = (uint32_t)(r + q) * kBytes;
      double* ac = acc + q * K;
      auto sx = [&](uint32_t bytes, int j) {
        return reinterpret_cast<const double*>(reinterpret_cast<const char*>(sX) + bytes)[j];
      };
#pragma unroll
      for (int j = 0; j < K; ++j) ac[j] = diag * sx(at0, j);
#pragma unroll
      for (int b = 0; b < LO - 1; ++b) {
        const uint32_t s = p >> b;
        const uint32_t d = sStep[b * 64 + ((__popc(s) << 2) | (s & 3u))];
        const uint32_t to = min(at0 + d, kZero);  // kParallel leaves the tile: the zeros
        const double cf = UNIFORM ? halfJ0 : a.halfJ[h + b];
        if constexpr (K == 1) {
          ac[0] += cf * sx(to, 0);
        } else {
#pragma unroll
          for (int j = 0; j < K; j += 2) {
            const double2 v = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(sX) + to + 8 * j);
            ac[j] += cf * v.x;
            ac[j + 1] += cf * v.y;
          }
        }
      }
    }
    for (;;) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const double cf = UNIFORM ? halfJ0 : a.halfJ[left ? __builtin_ctz(left) : 0];
        left &= left - 1;
#pragma unroll
        for (int j = 0; j < D; ++j) {
          acc[2 * j] += cf * vh[g][j].x;
          acc[2 * j + 1] += cf * vh[g][j].y;
        }
      }
      if (!m) break;
      whole();
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int j = 0; j < K; ++j) {
        acc[q * K + j] += (UNIFORM ? halfJ0 : a.halfJ[h - 1]) * (cross[q] ? vc[q * K + j] : 0.0);
        acc[q * K + j] += (UNIFORM ? halfJ0 : a.halfJ[L - 1]) * (wrap[q] ? vw[q * K + j] : 0.0);
      }
    double* yr = y + (size_t)(start + r) * K;
    if (mine == r && mine + Q <= end) {
#pragma unroll
      for (int j = 0; j < D; ++j) {
        Pair o = {acc[2 * j], acc[2 * j + 1]};
        if (add) o += reinterpret_cast<const Pair*>(yr)[j];
        reinterpret_cast<Pair*>(yr)[j] = o;
      }
    } else if (mine < end) {  // one vector, the last row alone
      const int q = Q == 1 ? 0 : min(mine - r, Q - 1);
      const double v = Q == 1 ? acc[0] : q ? acc[Q - 1] : acc[0];
      yr[q] = (add ? yr[q] : 0.0) + v;
    }
  }
}

// the tile of a row: the down sites of its first L - lo, site 0 in the highest bit
unsigned tile_of_row(const dh_basis* b, int lo, int64_t row) {
  const int L = b->chainLength;
  unsigned tile = 0;
  int n = b->nbrUp;
  for (int i = 0; i < L - lo; ++i) {
    const int64_t up = n > 0 ? (int64_t)dh_binom_host(L - 1 - i, n - 1) : 0;  // rows with site i up come first
    const bool down = row >= up;
    tile = tile << 1 | down;
    if (down)
      row -= up;
    else
      --n;
  }
  return tile;
}

template <int K, int LO, int BD, int G>
int spin_tile_launch(dh_hamiltonian* h, bool uniform, const double* x, double* y, int add, int64_t first,
                     int64_t count) {
  dh_context* c = h->ctx;
  const dh_basis* b = h->basis;
  SpinTileArgs a;
  a.table = b->d_spinTile + tile_offset(LO);
  a.binom = b->d_binom;
  a.L = b->chainLength;
  a.nbrUp = b->nbrUp;
  a.periodic = h->periodic;
  a.firstTile = tile_of_row(b, LO, first);
  a.endTile = tile_of_row(b, LO, first + count - 1) + 1;
  a.chunk = std::min(128u, (a.endTile - a.firstTile + 7) / 8);
  const unsigned perRound = 8 * a.chunk, tiles = (a.endTile - a.firstTile + perRound - 1) / perRound * perRound;
  // A range of rows in few tiles (a whole product has 256 at least) leaves CUs idle: one workgroup per round of
  // a tile's rows then, with the same values (10000 of 40 M rows: 10.2 -> 5.5 us with equal couplings, 16.7 ->
  // 8.0 with different ones; k = 8, 10000 of 2.7 M 11.8 -> 8.2).
  constexpr unsigned kRounds = (binom_c(LO, LO / 2) + (K == 1 ? 2 : 1) * BD - 1) / ((K == 1 ? 2 : 1) * BD);
  const unsigned parts = std::max(1u, std::min(kRounds, (unsigned)c->nbrCU / tiles));
  a.zeros = reinterpret_cast<const double*>(b->d_spinTile + tile_offset(kLoMax + 1));
  a.base = h->shift;
  for (int i = 0; i < 32; ++i) {
    a.halfJ[i] = 0.5 * h->J[i];
    a.halfJz[i] = 0.5 * h->Jz[i];
    if (i < a.L - 1 || (i == a.L - 1 && a.periodic)) a.base += 0.25 * h->Jz[i];
  }
  a.classOff[0] = 0;
  for (int n = 1; n <= kLoMax; ++n) a.classOff[n] = a.classOff[n - 1] + (n <= LO + 1 ? binom_c(LO, n - 1) : 0);
  if (uniform)
    hipLaunchKernelGGL((spin_tile_kernel<K, LO, BD, G, true>), dim3(tiles, parts), dim3(BD), 0, c->stream, a, x, y, add,
                       first, count);
  else
    hipLaunchKernelGGL((spin_tile_kernel<K, LO, BD, G, false>), dim3(tiles, parts), dim3(BD), 0, c->stream, a, x, y, add,
                       first, count);
  DH_HIP(c, hipGetLastError());
  return DH_OK;
}

}  // namespace

size_t dh_spin_tile_bytes() { return sizeof(uint32_t) * (tile_offset(kLoMax + 1) + kZeroWords); }

int dh_spin_tile_tables(dh_basis* b) {
  dh_context* c = b->ctx;
  hipLaunchKernelGGL(spin_tile_table_kernel, dim3(kZeroWords / 256, kLoMax - kLoMin + 2), dim3(256), 0, c->stream,
                     b->d_spinTile, b->d_binom);
  DH_HIP(c, hipGetLastError());
  return DH_OK;
}

// Last sites per tile.  About 30 KB of x, 31 to 35 KB of LDS with the distances, so that four (k = 16 and the
// 512-thread workgroups, by their wavefronts as well) or five (k = 8) tiles share a CU; for one vector on chains
// below 26 sites 12, for more and smaller tiles (24 sites 25.6 us, 27.5 with 14; 28 sites 501 and 454).
static int spin_tile_sites(const dh_hamiltonian* h, int k) {
  switch (k) {
    case 1: return h->basis->chainLength >= 26 ? 14 : 12;
    case 2: return 13;
    case 4: return 12;
    case 8: return 11;
    default: return 10;
  }
}

// Enough tiles to fill the CUs, and rows enough in them: a tile costs 3.7 ns however few rows it has.  Lines where
// the time by rows and by tiles meet, with that of the row kernel first (us):
// - one vector, equal couplings: from 256 tiles on a ring (20 sites 7.0 and 6.5), 512 on an open chain (20
//   sites 6.0 and 6.3, 21 sites 8.2 and 7.0); different ones from 1024 (21 sites 9.1 and 10.1 open, 10.3 and
//   10.2 on a ring; 22 sites 17.6 and 12.3).  Blocks of k: from 512 (21 sites, k = 4: 15.1 and 13.2).
// - tiles half full on average (24 sites, Sz = 4, 0.52 full: 39.0 and 30.7, k = 4 71.8 and 71.0), 0.6 with
//   different couplings on open chains of few tiles (22 sites, 0.53 full: 11.0 and 11.9, k = 4 18.3 and 20.2).
// - two vectors, whose rows of 16 bytes gain least: 0.6 with equal couplings (24 sites, 0.56 full: 37.4 and
//   39.3; 23 sites, 0.65 full: 26.9 and 22.7); with different ones on a ring 0.6 up to 1024 tiles (22 sites, 0.57
//   full: 14.0 and 15.7; 23 sites, 0.65 full: 29.6 and 25.9) and 0.7 above (26 sites, 0.69 full: 202 and 206; 0.74
//   full: 216 and 210), on an open chain 0.7 with 512 tiles (22 sites, 0.73 full: 17.9 and 16.9) and never with
//   more (24 sites, 0.71 full: 43.0 and 45.9; 26 sites, 0.74 full: 201 and 203).
bool dh_spin_tiles(const dh_hamiltonian* h, bool uniform, int k) {
  const dh_basis* b = h->basis;
  const int lo = spin_tile_sites(h, k), split = b->chainLength - lo;
  const bool ring = h->periodic != 0;
  if (!b->d_spinTile || split < (k == 1 ? (uniform ? (ring ? 8 : 9) : 10) : 9)) return false;
  if (k == 2 && !uniform && !ring && split > 9) return false;
  int tenths = !uniform && !ring && split <= 10 ? 6 : 5;
  if (k == 2) tenths = uniform || (ring && split <= 10) ? 6 : 7;
  return 10 * (b->dim >> split) >= (int64_t)tenths * binom_c(lo, lo / 2);
}

int dh_spin_tile_hv(dh_hamiltonian* h, bool uniform, const double* x, double* y, int k, int add, int64_t first,
                    int64_t count) {
  switch (k) {
    case 1:
      if (spin_tile_sites(h, 1) == 14) return spin_tile_launch<1, 14, 512, 2>(h, uniform, x, y, add, first, count);
      return spin_tile_launch<1, 12, 256, 4>(h, uniform, x, y, add, first, count);
    case 2: return spin_tile_launch<2, 13, 512, 2>(h, uniform, x, y, add, first, count);
    case 4: return spin_tile_launch<4, 12, 512, 1>(h, uniform, x, y, add, first, count);
    case 8: return spin_tile_launch<8, 11, 256, 1>(h, uniform, x, y, add, first, count);
    default: return spin_tile_launch<16, 10, 128, 1>(h, uniform, x, y, add, first, count);
  }
}
