// The three-operation quotient q = a*y, q + (a - b*q)*y with y = 1/b rounded
// to nearest (gpu-comcot_amd/csrc/fastdiv.h) against IEEE division.  For
// every significand b, every a whose quotient lies within 16 / (2 b) ulp of
// a rounding midpoint is tried (the only ones that an error of some 2^-23 ulp
// before the last rounding can move), and 24 others per b.  Scaling by
// powers of two changes nothing, so significands stand for all operands in
// range.  Prints the number of pairs tried and of wrong quotients.
#include <math.h>
#include <stdint.h>
#include <stdio.h>

static uint32_t inverse(uint32_t b) {  // of odd b modulo 2^32
  uint32_t x = b;
  for (int k = 0; k < 5; ++k) x *= 2 - b * x;
  return x;
}

static bool wrong(float a, float b, float y) {
  const float q = a * y;
  return fmaf(fmaf(-b, q, a), y, q) != a / b;
}

int main() {
  unsigned long long tried = 0, bad = 0;
#pragma omp parallel for schedule(dynamic, 4096) reduction(+ : tried, bad)
  for (uint32_t B = 1u << 23; B < (1u << 24); ++B) {
    const float b = (float)B, y = (float)(1.0 / (double)b);
    const int t = __builtin_ctz(B);
    // a * 2^p = b * m + s, m odd in [2^24, 2^25): p = 24 for a >= b, else 25
    for (int p = 24; p <= 25 && t <= 4; ++p)
      for (int s = -16; s <= 16; ++s) {
        if (s == 0 || (s & ((1 << t) - 1))) continue;
        const uint64_t mod = 1ull << (p - t);
        uint64_t m = (uint64_t)inverse(B >> t) * (uint32_t)(-(s >> t)) & (mod - 1);
        if (!(m & 1)) continue;
        for (; m < (1ull << 25); m += mod) {
          if (m < (1ull << 24)) continue;
          const __int128 n = (__int128)B * m + s;
          const uint64_t A = (uint64_t)(n >> p);
          if (A < (1u << 23) || A >= (1u << 24) || (p == 24) != (A >= B)) continue;
          ++tried;
          bad += wrong((float)A, b, y);
        }
      }
    for (uint32_t k = 0; k < 24; ++k) {
      const uint32_t A = k == 0 ? B : (1u << 23) | ((B * 2654435761u * (k + 1) + k * 40503u) >> 9);
      ++tried;
      bad += wrong((float)A, b, y);
    }
  }
  printf("%llu %llu\n", tried, bad);
  return 0;
}
