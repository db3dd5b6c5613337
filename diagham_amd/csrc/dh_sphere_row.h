// Per-row accumulation of the fermions-on-the-sphere product, shared by the single-sector
// and the multi-sector kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "dh_index.h"
#include "dh_internal.h"

// Bit helpers over the state word: 64-bit words in general, 32-bit words when the orbitals fit
// (half the instructions for every shift, mask, ctz and popcount of the row routine).
__device__ __forceinline__ int dh_ctz(uint64_t v) { return __builtin_ctzll(v); }
__device__ __forceinline__ int dh_ctz(uint32_t v) { return __builtin_ctz(v); }

// Off-diagonal factors of annihilated pair i of one sum in LDS (dh_pack_sphere_factors): a square's row,
// or one triangle.  The entry of sBase packs where the sum's table starts and its number of pairs.
template <bool TRI>
struct dh_row_factors {
  const double* f;
  int i;
  __device__ __forceinline__ dh_row_factors(const double* sF, int entry, int i_) : i(i_) {
    f = sF + (entry & DH_SUM_BASE_MASK);
    if (!TRI) f += __mul24(i_, (int)((unsigned)entry >> DH_SUM_BASE_BITS));
  }
  __device__ __forceinline__ double operator()(int j) const {
    if (!TRI) return f[j];
    // a 24-bit multiply (positions stay below 2^12) instead of the quarter-rate 32-bit one
    const unsigned mx = (unsigned)max(i, j), mn = (unsigned)min(i, j);
    return f[(__umul24(mx, mx + 1u) >> 1) + mn];
  }
};

// ALL: every load of the row is issued before the first multiply-add.  The compiler does that by itself up to 8
// vectors; for 16 it may take two loads at a time, for a fifth wavefront per SIMD that the LDS does not allow (3.4 M
// rows of 28 orbitals: 8.6 ms with the loads together, 10.0 in twos).
template <int K, bool ALL = false, typename I>
__device__ __forceinline__ void dh_gather_fma(double* acc, const double* __restrict__ x, I idx, double coef) {
  const double* xr = x + (size_t)idx * K;
  if constexpr (ALL) {
    double2 p[K / 2];
#pragma unroll
    for (int v = 0; v < K / 2; ++v) p[v] = reinterpret_cast<const double2*>(xr)[v];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < K / 2; ++v) {
      acc[2 * v] += coef * p[v].x;
      acc[2 * v + 1] += coef * p[v].y;
    }
  } else if constexpr (K % 2 == 0) {
#pragma unroll
    for (int v = 0; v < K; v += 2) {
      double2 p = *reinterpret_cast<const double2*>(xr + v);
      acc[v] += coef * p.x;
      acc[v + 1] += coef * p.y;
    }
  } else {
#pragma unroll
    for (int v = 0; v < K; ++v) acc[v] += coef * xr[v];
  }
}

__host__ __device__ __forceinline__ uint64_t dh_bitrev(uint64_t v) { return __builtin_bitreverse64(v); }
__host__ __device__ __forceinline__ uint32_t dh_bitrev(uint32_t v) { return __builtin_bitreverse32(v); }

// What a row state s tells about the pairs (m3 > m4) of one orbital sum S, as 32-bit masks over their
// positions i = m3 - lo(S), m3 = lo(S) + i, m4 = m4hi(S) - i, lo(S) = S/2 + 1, m4hi(S) = (S - 1)/2
// (at most 31 positions for 62 orbitals).
//
// free(S): both orbitals free in s.  Word f of the free orbitals, shifted so that m3 lands on bit i,
// and f reversed, shifted so that m4 lands on bit i; both are zero beyond the orbitals.
// sign(S): parity of the occupied orbitals in [m4, m3), from the prefix parities P (bit m: parity of
// the occupied orbitals below m) in the same way.
//
// A term that annihilates pair a and creates pair b of the same sum, b != a: two pairs of one sum are
// nested, m4 < n2 < n1 < m3 or n2 < m4 < m3 < n1, so they have no orbital in common, b has to be free
// in s itself, and taking n1, n2 out of s changes the number of orbitals in [m4, m3) by 0 or 2.  Its
// sign, popc(s >> n1) + popc(s >> n2) + popc(t >> m3) + popc(t >> m4), is thus
// sign(S)[a] + sign(S)[b].  The term b = a is diagonal: -F(a, a).
template <typename U>
struct dh_row_masks {
  static constexpr int W = 8 * sizeof(U);
  U f, rf, par, rpar;
  __host__ __device__ __forceinline__ dh_row_masks(U s, int nbrOrbitals) {
    const U full = nbrOrbitals >= W ? ~U(0) : ((U(1) << nbrOrbitals) - U(1));
    f = ~s & full;
    rf = dh_bitrev(f);
    par = s << 1;
#pragma unroll
    for (int o = 1; o < W; o <<= 1) par ^= par << o;
    rpar = dh_bitrev(par);
  }
  __host__ __device__ __forceinline__ uint32_t free(int m3lo, int m4hi) const {
    return (uint32_t)(f >> m3lo) & (uint32_t)(rf >> (W - 1 - m4hi));
  }
  __host__ __device__ __forceinline__ uint32_t sign(int m3lo, int m4hi) const {
    return (uint32_t)(par >> m3lo) ^ (uint32_t)(rpar >> (W - 1 - m4hi));
  }
};

// the factor c with the sign that bit 31 - c of the position mask q gives its position
__device__ __forceinline__ double dh_negate_by(double c, uint32_t signAtBit31) {
  return __hiloint2double(__double2hiint(c) ^ (int)(signAtBit31 & 0x80000000u), __double2loint(c));
}

// The diagonal coefficient of a row, -F(a, a) over its pairs a, in two doubles: each n1's pairs are subtracted
// together, and what the subtraction rounds off is kept (Dekker's fast two-sum: exact while the sum is the
// larger, which it is from the third n1 on for factors of one sign).  The caller adds the diagonal term last,
// after the sums of the row's lanes have met: it is the largest by far, so a rounding after it costs the most.
// Error against exactly summed elements, relative to the norm of the product: N=6 2S=15, k = 8, 1.26e-16 with
// one double and the term on lane 0, 0.92 with the elements one by one, 0.59 so; N=8 2S=21 1.22, 1.13 and 0.59;
// N=10 2S=27 1.09, 4.15 and 0.56.
struct dh_diagonal {
  double sum = 0.0, rest = 0.0;
  __device__ __forceinline__ void subtract(double v) {
    const double s = sum - v;
    rest += (sum - s) - v;
    sum = s;
  }
  // acc + this times x
  __device__ __forceinline__ double term(double x, double acc) const { return fma(sum, x, fma(rest, x, acc)); }
};

// Two-body terms of row state s: for every occupied pair n1 > n2 (annihilated) and every other pair
// m3 > m4 of the same orbital sum that is free in s (created), one gather; the diagonal terms are
// summed into one coefficient (returned, the same on every lane).  FREE walks the set bits of the free mask; otherwise every
// position is tried against it (fewer registers).  Positions run from the highest down, and lane
// `lane` of the row's LPR lanes takes every LPR-th (free) one.  Target indices come from
// `find(target)`; x is indexed relative to `xbase`.
//
// A term costs 23 vector instructions on 32-bit and 28 on 64-bit words (36 and 46 before the masks over
// positions, the square factor rows, and the diagonal terms apart), which leaves the gathers as the
// bound: N=12 2S=33 Lz=0, k = 1, 5.6 -> 4.5 ms with the vector units busy 60 % of it (89 % before) and
// one L1 access in every cycle, 27 per 64-lane gather.
// For K <= 2 the multiply-add of a term is deferred to the next term, after that term's index loads
// are issued: a term's gather and the next term's index loads are then in flight together (the terms
// are still added in their order, so FREE and the range form agree to the bit at one lane per row).
// Wider K keep one gather in flight per term: their registers would lower the occupancy that hides
// the latency there.
template <int K, int LPR, bool FREE, bool TRI, typename U, typename Find>
__device__ __forceinline__ dh_diagonal dh_sphere_row(U s, int nbrOrbitals, const double* __restrict__ sF,
                                                     const int* __restrict__ sBase, int lane, Find find,
                                                     const double* __restrict__ xbase, double* acc) {
  constexpr bool PIPE = K <= 2;
  double pend[K];
  double pendCoef = 0.0;
  dh_diagonal diag;
#pragma unroll
  for (int v = 0; v < K; ++v) pend[v] = 0.0;
  const dh_row_masks<U> masks(s, nbrOrbitals);
  for (U r1 = s; r1; r1 &= r1 - 1) {
    const int n1 = dh_ctz(r1);
    const double* diagRow = sF + __mul24(n1, n1 - 1) / 2;  // !TRI
    double diag1 = 0.0;  // of this n1
    for (U r2 = s & ((U(1) << n1) - U(1)); r2; r2 &= r2 - 1) {
      const int n2 = dh_ctz(r2);
      if (!TRI) diag1 += diagRow[n2];
      const int sum = n1 + n2, m3lo = (sum >> 1) + 1, m4hi = (sum - 1) >> 1;
      uint32_t pm = masks.free(m3lo, m4hi);
      if (FREE && !TRI && !pm) continue;
      const U t = s ^ (U(1) << n1) ^ (U(1) << n2);
      const int entry = sBase[sum], i = n1 - m3lo;
      const dh_row_factors<TRI> F(sF, entry, i);
      if (TRI) diag1 += F(i);
      uint32_t q = masks.sign(m3lo, m4hi);
      q ^= (uint32_t)-(int)((q >> i) & 1u);  // relative to the annihilated pair
      // the created pair at position 31 - c (bit: its bit in a position mask), its sign in bit 31 of sg
      auto term = [&](int c, uint32_t bit, uint32_t sg) {
        const auto idx = find(t | (U(bit) << m3lo) | (U(1) << (m4hi - 31 + c)));
        const double coef = dh_negate_by(F(31 - c), sg);
        if constexpr (PIPE) {
          // the previous term first, then this term's gather into the same registers (no copy,
          // so nothing waits for the gather before the next term's index loads)
          const double* xr = xbase + (size_t)idx * K;
#pragma unroll
          for (int v = 0; v < K; ++v) acc[v] = fma(pendCoef, pend[v], acc[v]);
#pragma unroll
          for (int v = 0; v < K; ++v) pend[v] = xr[v];
          pendCoef = coef;
        } else {
          dh_gather_fma<K, K == 16>(acc, xbase, idx, coef);
        }
      };
      if constexpr (FREE) {
        if constexpr (LPR > 1)
          for (int l = 0; l < lane && pm; ++l) pm ^= 0x80000000u >> __builtin_clz(pm);
        while (pm) {
          const int c = __builtin_clz(pm);
          const uint32_t bit = 0x80000000u >> c;
          pm ^= bit;
#pragma unroll
          for (int l = 1; l < LPR; ++l)  // past the other lanes' next ones
            if (pm) pm ^= 0x80000000u >> __builtin_clz(pm);
          term(c, bit, q << c);
        }
      } else {
        for (int j = (int)((unsigned)entry >> DH_SUM_BASE_BITS) - 1 - lane; j >= 0; j -= LPR)
          if ((pm >> j) & 1u) term(31 - j, 1u << j, q << (31 - j));
      }
    }
    diag.subtract(diag1);
  }
  if constexpr (PIPE) {
#pragma unroll
    for (int v = 0; v < K; ++v) acc[v] = fma(pendCoef, pend[v], acc[v]);
  }
  return diag;
}

// The same terms with the created-pair loop unrolled four-wide: a lane computes four targets
// (a slot past the last pair or on an occupied orbital looks up the row's own state with a zero
// coefficient), issues their index lookups together and then their four gathers, so four
// dependent chains are in flight per lane.  `s` must be a state of the space (the padding
// slots look it up).
template <int K, int LPR, bool TRI, typename U, typename Find>
__device__ __forceinline__ dh_diagonal dh_sphere_row_x4(U s, int nbrOrbitals, const double* __restrict__ sF,
                                                        const int* __restrict__ sBase, int lane, Find find,
                                                        const double* __restrict__ xbase, double* acc) {
  const dh_row_masks<U> masks(s, nbrOrbitals);
  dh_diagonal diag;
  for (U r1 = s; r1; r1 &= r1 - 1) {
    const int n1 = dh_ctz(r1);
    double diag1 = 0.0;
    for (U r2 = s & ((U(1) << n1) - U(1)); r2; r2 &= r2 - 1) {
      const int n2 = dh_ctz(r2);
      const int sum = n1 + n2, m3lo = (sum >> 1) + 1, m4hi = (sum - 1) >> 1;
      const U t = s ^ (U(1) << n1) ^ (U(1) << n2);
      const int entry = sBase[sum], i = n1 - m3lo, np = (int)((unsigned)entry >> DH_SUM_BASE_BITS);
      const dh_row_factors<TRI> F(sF, entry, i);
      diag1 += TRI ? F(i) : sF[__mul24(n1, n1 - 1) / 2 + n2];
      const uint32_t pm = masks.free(m3lo, m4hi);
      uint32_t q = masks.sign(m3lo, m4hi);
      q ^= (uint32_t)-(int)((q >> i) & 1u);
      for (int jb = lane; jb < np; jb += 4 * LPR) {
        decltype(find(s)) idx[4];
        double coef[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = min(jb + u * LPR, np - 1);  // clamped so that every shift stays in range
          const bool ok = (jb + u * LPR < np) && ((pm >> j) & 1u);
          const double c = ok ? F(j) : 0.0;
          coef[u] = dh_negate_by(c, q << (31 - j));
          idx[u] = find(ok ? (t | (U(1) << (m3lo + j)) | (U(1) << (m4hi - j))) : s);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) dh_gather_fma<K>(acc, xbase, idx[u], coef[u]);
      }
    }
    diag.subtract(diag1);
  }
  return diag;
}
