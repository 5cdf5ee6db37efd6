// noise_engine.h -- the reference's Brownian noise stream: the minimal
// standard engine x <- 16807 x mod 2^31 - 1 (std::default_random_engine of
// the reference's toolchain, random_generator.C:43-67, :96-99) and N(0, 1)
// values by the polar method (Marsaglia & Bray 1964), word for word and bit
// for bit what std::normal_distribution gives on that engine.
//
// std::normal_distribution took 36 ns a value (2.8 ms for 25,600 beads): each
// of its uniforms works out the number of engine words it needs through long
// double logarithms.  Here that number is the constant 2, and the four words
// of a candidate come from one state by the powers of the multiplier instead
// of one after the other.
#pragma once

#include <cmath>
#include <cstdint>

namespace ggem {

class NoiseEngine {
 public:
  explicit NoiseEngine(uint64_t s = 1) { seed(s); }
  void seed(uint64_t s) {
    s_ = s % kM;
    if (s_ == 0) s_ = 1;
  }
  // f(i, v) for i = 0 .. n - 1: n N(0, 1) values of a fresh distribution
  // (a pair's second value is dropped when n is odd)
  template <class F>
  void normals(int64_t n, F&& f) {
    for (int64_t i = 0; i < n;) {
      double x, y, r2;
      do candidate(x, y, r2);
      while (r2 > 1.0 || r2 == 0.0);
      const double mult = std::sqrt(-2 * std::log(r2) / r2);
      f(i++, y * mult);
      if (i < n) f(i++, x * mult);
    }
  }
  // the engine past n N(0, 1) values of a fresh distribution
  void skip(int64_t n) {
    for (int64_t i = 0; i < n; i += 2) {
      double x, y, r2;
      do candidate(x, y, r2);
      while (r2 > 1.0 || r2 == 0.0);
    }
  }

 private:
  static constexpr uint64_t kM = 2147483647, kA = 16807;
  static constexpr uint64_t kA2 = kA * kA % kM, kA3 = kA2 * kA % kM, kA4 = kA3 * kA % kM;
  // a s mod 2^31 - 1 for a, s below it: the two 31-bit halves of the product
  // added, reduced once
  static uint64_t mul(uint64_t a, uint64_t s) {
    const uint64_t p = a * s, q = (p & kM) + (p >> 31);
    return q >= kM ? q - kM : q;
  }
  // one uniform in [0, 1) from two words (53 bits asked of 31 bits each):
  // (w0 + w1 R)/R^2, R = 2^31 - 2 the engine's range
  static double uniform(uint64_t w0, uint64_t w1) {
    constexpr double R = 2147483646.0, R2 = R * R;
    const double u = (double(w0 - 1) + double(w1 - 1) * R) / R2;
    return u < 1.0 ? u : 0x1.fffffffffffffp-1;
  }
  void candidate(double& x, double& y, double& r2) {
    const uint64_t w0 = mul(kA, s_), w1 = mul(kA2, s_), w2 = mul(kA3, s_), w3 = mul(kA4, s_);
    s_ = w3;
    x = 2.0 * uniform(w0, w1) - 1.0;
    y = 2.0 * uniform(w2, w3) - 1.0;
    r2 = x * x + y * y;
  }
  uint64_t s_ = 1;
};

}  // namespace ggem
