// Largest absolute error of cossin_turn against float64 over float arguments in [-1/2, 1/2]:
// evenly spaced ones and their neighbours at the octant bounds, and small ones.
#include "common.hpp"

#include <cmath>
#include <cstdio>

int main() {
  double worst = 0, rel = 0;
  auto check = [&](float f) {
    float c, s;
    bippamd::cossin_turn(f, c, s);
    const double a = 2 * M_PI * static_cast<double>(f);
    const double ec = std::fabs(c - std::cos(a)), es = std::fabs(s - std::sin(a));
    worst = std::fmax(worst, std::fmax(ec, es));
    if (std::fabs(f) >= 1e-30f && std::fabs(f) < 0.125f)  // (rounding is relative to there)
      rel = std::fmax(rel, es / std::fabs(std::sin(a)));
  };
  for (int k = -(1 << 23); k <= 1 << 23; ++k) check(static_cast<float>(k) / (1 << 24));
  for (int k = -4; k <= 4; ++k)
    for (int q = -64; q <= 64; ++q) {
      float f = k / 8.0f;
      for (int i = 0; i < std::abs(q); ++i) f = std::nextafterf(f, q < 0 ? -1.0f : 1.0f);
      if (std::fabs(f) <= 0.5f) check(f);
    }
  for (float f = 1e-30f; f < 0.125f; f *= 1.01f) check(f), check(-f);
  std::printf("%.6e %.6e\n", worst, rel);
  return 0;
}
