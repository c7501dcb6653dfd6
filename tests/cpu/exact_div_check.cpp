// QuotientByReciprocal (exact_div.h) against IEEE division on the CPU: every
// pair of 24-bit significands whose quotient lies within 2^-23 ulp of a
// midpoint between two floats (all others round right by the header's error
// bound), then random pairs over the exponents it is used for, exact
// quotients, zero dividends and zero divisors. Prints "ok".
//
// Pairs near a midpoint: with N odd the 25-bit midpoint, A / D is within
// c / (2 D) ulp of it when A 2^s = D N + c (s = 24 for A >= D, else 25), so
// |c| <= 3, and N follows from N = -c / D mod 2^s.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>

#include "exact_div.h"

using namespace muonx;

static uint64_t InverseMod2(uint64_t odd) {
  uint64_t x = odd;
  for (int i = 0; i < 6; ++i) x *= 2 - odd * x;
  return x;
}

static bool Same(float a, float d) { return QuotientByReciprocal(a, d, 1.0f / d) == a / d; }

int main() {
  uint64_t tested = 0, bad = 0;
  for (uint64_t D = 1ull << 23; D < (1ull << 24); ++D) {
    for (int s = 24; s <= 25; ++s) {
      for (int c = -3; c <= 3; ++c) {
        if (c == 0) continue;
        uint64_t dp = D;
        int cp = c, bits = s;
        while (!(dp & 1) && !(cp & 1)) {
          dp >>= 1;
          cp /= 2;
          --bits;
        }
        if (!(dp & 1)) continue;  // no such N
        const uint64_t mod = 1ull << bits;
        for (uint64_t N = (InverseMod2(dp) * uint64_t(-int64_t(cp))) & (mod - 1); N < (1ull << 25); N += mod) {
          if (N < (1ull << 24) || !(N & 1)) continue;
          const int64_t num = int64_t(D * N) + c;
          if (num & ((1ll << s) - 1)) continue;
          const uint64_t A = uint64_t(num) >> s;
          if (A < (1ull << 23) || A >= (1ull << 24) || (A >= D) != (s == 24)) continue;
          ++tested;
          bad += !Same(float(A), float(D));
        }
      }
    }
  }
  std::mt19937_64 g(7);
  auto sig = [&] { return 1.0f + float(g() >> 41) * 0x1p-23f; };
  for (int k = 0; k < 20000000; ++k) {
    const float a = std::ldexp(sig(), int(g() % 160) - 99), d = std::ldexp(sig(), int(g() % 80) - 60);
    bad += !DivisorOk(d) || !Same((g() & 1) ? a : -a, (g() & 1) ? d : -d);
    const float q = std::ldexp(float(g() >> 52), int(g() % 40) - 20), p = float(g() >> 52);
    bad += p != 0.0f && !Same(q * p, p);  // exact quotients (24 bits in all)
  }
  bad += !Same(0.0f, 3.0f) || !Same(-0.0f, -0.7f);
  for (const float a : {0.0f, 1.5f, -2.0f}) bad += !std::isnan(QuotientByReciprocal(a, 0.0f, 1.0f / 0.0f));
  bad += CoordinateOk(INFINITY) || CoordinateOk(NAN) || CoordinateOk(1e-30f) || DivisorOk(NAN) || DivisorOk(1e-20f);
  if (tested < 10000000 || bad) {
    std::printf("%llu near-midpoint pairs, %llu wrong\n", (unsigned long long)tested, (unsigned long long)bad);
    return 1;
  }
  std::puts("ok");
  return 0;
}
