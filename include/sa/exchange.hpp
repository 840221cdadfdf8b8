// exchange.hpp -- the lane-wise replica-exchange decision shared by the
// parallel-tempering driver and the batched engine.
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

namespace sa {

// Lanes k < n of one 64-lane word: lane k of systems i and i+1 exchange when
// dE*dB > 0 or u < exp(dB*dE), with dE = -(E_i[k] - E_{i+1}[k]) in float and
// dB = 1/T_i - 1/T_{i+1} (creat_mask, src/parallel_tempering.hpp:141-162).
// `accepted` is increased by the number of exchanging lanes.
inline uint64_t exchange_word(const float *Ei, const float *Ej, double dB, double u, int n, int &accepted) {
  uint64_t m = 0;
  for (int k = 0; k < n; ++k) {
    const float dE = -(Ei[k] - Ej[k]);
    if (((dE * dB) > 0.) || u < std::exp(dB * dE)) {
      m |= 1ULL << k;
      ++accepted;
    }
  }
  return m;
}

// The rule of exchange_word as a threshold: for dB >= 0 a lane exchanges iff dE >= t.  The
// rule holds for dE >= 0 (u < 1), and u < exp(dB * dE) does not come back as dE decreases,
// so t is found by bisection over the negative floats with the rule itself.
inline float exchange_threshold(double dB, double u) {
  auto value = [](uint32_t bits) {
    float f;
    bits |= 0x80000000u;  // -|f|, larger magnitudes for larger bits
    std::memcpy(&f, &bits, sizeof f);
    return f;
  };
  auto holds = [&](uint32_t bits) {
    const float dE = value(bits);
    return ((dE * dB) > 0.) || u < std::exp(dB * dE);
  };
  uint32_t lo = 0, hi = 0x7f800000u;  // holds at -0, not at -infinity (dB > 0)
  if (holds(hi - 1)) return -INFINITY;
  while (hi - lo > 1) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (holds(mid)) lo = mid;
    else hi = mid;
  }
  return value(lo);
}

}  // namespace sa
