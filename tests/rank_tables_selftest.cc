// Rank lookups of the product kernels on the host (compiled as HIP host code): for every number of orbitals
// and every form of the lookup that a kernel takes for it, the entries of a state with its top orbital
// occupied are read from the places where they belong.  The tables are address space without memory
// (62 orbitals take 8 GiB each), with the two entries written.
#include <sys/mman.h>

#include <cstdio>
#include <cstring>

#include "dh_index.h"
#include "dh_internal.h"

static uint32_t* reserve(size_t words) {
  void* p = mmap(nullptr, words * sizeof(uint32_t), PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : static_cast<uint32_t*>(p);
}

template <typename U, bool LO_IN_LDS>
static int check(int orbitals, uint32_t* lo, uint32_t* hi) {
  constexpr bool FAR = dh_far_tables<U, LO_IN_LDS>;
  const int bits = dh_rank_split(orbitals);
  const uint64_t loMask = (1ull << bits) - 1ull;
  int wrong = 0;
  for (uint64_t state : {(1ull << (orbitals - 1)) | 1ull, (1ull << (orbitals - 1)) | (1ull << (bits - 1)),
                         ((1ull << (orbitals - 1)) - 1ull) | (1ull << (orbitals - 1))}) {
    hi[state >> bits] = 1000;
    lo[state & loMask] = 17;
    const U t = (U)state;
    const uint32_t l = dh_entry<FAR>(lo, (uint32_t)(t & (U)loMask));
    wrong += dh_rank_of<FAR>(t, [&] { return l; }, hi, bits, 5000u) != 983u;
    wrong += dh_rank_of<FAR>(t, [&] { return l; }, hi, bits, 400u) != 400u;  // clamped
    hi[state >> bits] = 0;
    lo[state & loMask] = 0;
  }
  return wrong;
}

int main() {
  for (int orbitals = 2; orbitals <= 63; ++orbitals) {
    const int bits = dh_rank_split(orbitals);
    const size_t loWords = size_t(1) << bits, hiWords = size_t(1) << (orbitals - bits);
    uint32_t *lo = reserve(loWords), *hi = reserve(hiWords);
    if (!lo || !hi) return std::printf("no address space\n"), 2;
    const int w32 = orbitals <= 32 ? check<uint32_t, false>(orbitals, lo, hi) + check<uint32_t, true>(orbitals, lo, hi) : 0;
    const int lds = loWords <= (size_t(1) << 15) ? check<uint64_t, true>(orbitals, lo, hi) : 0;  // dh_rank_lo16
    const int far = check<uint64_t, false>(orbitals, lo, hi);
    std::printf("%d %d\n", orbitals, w32 + lds + far);
    munmap(lo, loWords * sizeof(uint32_t));
    munmap(hi, hiWords * sizeof(uint32_t));
  }
  return 0;
}
