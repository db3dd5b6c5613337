// Masks over pair positions of the sphere rows (dh_row_masks), compiled as HIP host code: every orbital sum of
// every state up to 12 orbitals and of many states of up to 63, on 32- and 64-bit words.  Prints the number of
// checks and of mismatches.
#include <cstdio>

#include "dh_sphere_row.h"

static long checks, wrong;
static void expect(bool ok) {
  ++checks;
  wrong += !ok;
}

// sign of annihilating n1 > n2 of s and creating m3 > m4 on what is left: popcounts at and above each operator
static int reference_sign(uint64_t s, int n1, int n2, int m3, int m4) {
  const uint64_t t = s ^ (1ull << n1) ^ (1ull << n2);
  return (__builtin_popcountll(s >> n1) + __builtin_popcountll(s >> n2) + __builtin_popcountll(t >> m3) +
          __builtin_popcountll(t >> m4)) & 1;
}

template <typename U>
static void check_state(uint64_t s, int orbitals) {
  const dh_row_masks<U> masks((U)s, orbitals);
  for (int sum = 1; sum <= 2 * orbitals - 3; ++sum) {
    const int lo = sum / 2 + 1, m4hi = (sum - 1) / 2, np = std::min(sum, orbitals - 1) - lo + 1;
    const uint32_t f = masks.free(lo, m4hi), q = masks.sign(lo, m4hi);
    for (int i = 0; i < 32; ++i) {
      const int a = lo + i, b = sum - a;
      const bool pair = i < np;
      const bool free = pair && !((s >> a) & 1) && !((s >> b) & 1);
      expect(((f >> i) & 1) == free);
      if (!pair || !((s >> a) & 1) || !((s >> b) & 1)) continue;
      // annihilated pair i: the created pairs are the free ones of s and the pair itself, with the sign -1
      const uint64_t t = s ^ (1ull << a) ^ (1ull << b);
      for (int j = 0; j < np; ++j) {
        const int c = lo + j, d = sum - c;
        const bool created = !((t >> c) & 1) && !((t >> d) & 1);
        expect(created == (j == i || ((f >> j) & 1)));
        if (!created) continue;
        const int sign = reference_sign(s, a, b, c, d);
        expect(j == i ? sign == 1 : sign == (((q >> i) ^ (q >> j)) & 1));
      }
    }
  }
}

int main() {
  for (int orbitals = 2; orbitals <= 12; ++orbitals)
    for (uint64_t s = 0; s < (1ull << orbitals); ++s) {
      check_state<uint32_t>(s, orbitals);
      check_state<uint64_t>(s, orbitals);
    }
  uint64_t r = 88172645463325252ull;
  for (int orbitals : {28, 31, 32, 33, 47, 61, 62, 63})
    for (int n = 0; n < 300; ++n) {
      r ^= r << 13, r ^= r >> 7, r ^= r << 17;
      const uint64_t s = r & ((1ull << orbitals) - 1) & (n % 3 ? ~0ull : (r >> 17 | r << 47));
      check_state<uint64_t>(s, orbitals);
      if (orbitals <= 32) check_state<uint32_t>(s, orbitals);
    }
  std::printf("%ld %ld\n", checks, wrong);
  return 0;
}
