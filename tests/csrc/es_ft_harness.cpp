// Errors of es_ft_table against long double, and of the plain sum with a cosine per node and
// entry, over the tables that plans build: every kernel width, grids of 192 and 1728 points.
// Prints worst and mean square errors relative to phi(0), worst relative errors.
#include <hip/hip_runtime.h>

#include "host_runtime.hpp"
#include "kernels.hpp"
#include "nufft_host.hpp"

#include <cstdio>

namespace {
using namespace bippamd;

struct Err {
  double abs = 0, rel = 0, square = 0;
};

void measure(double xi0, double dxi, int n, const std::vector<double>& x, const std::vector<double>& ew,
             Err& tab, Err& plain) {
  const std::vector<double> t = es_ft_table(xi0, dxi, n, x, ew);
  long double phi0 = 0;
  for (double e : ew) phi0 += 2 * static_cast<long double>(e);
  for (int j = 0; j < n; ++j) {
    long double exact = 0;
    double sum = 0;
    for (size_t i = 0; i < x.size(); ++i) {
      exact += 2 * static_cast<long double>(ew[i]) *
               cosl((static_cast<long double>(xi0) + static_cast<long double>(j) * dxi) * x[i]);
      sum += ew[i] * std::cos(std::fabs(xi0 + j * dxi) * x[i]);
    }
    auto note = [&](Err& e, double v) {
      const double d = std::fabs(static_cast<double>(v - exact));
      e.abs = std::fmax(e.abs, static_cast<double>(d / phi0));
      e.rel = std::fmax(e.rel, static_cast<double>(d / fabsl(exact)));
      e.square += static_cast<double>(d * d / (phi0 * phi0));
    };
    note(tab, t[j]);
    note(plain, 2 * sum);
  }
}
}  // namespace

int main() {
  Err tab, plain;
  for (int w = 2; w <= 16; ++w) {
    std::vector<double> x, gw;
    gauss_legendre01(64, x, gw);
    const std::vector<double> ew = es_ft_weights(2.3 * w, x, gw);
    const double pi = 3.14159265358979323846, xi_max = 1.05 * pi * w / 4 + 1e-3, d = xi_max / 2048;
    measure(-d, d, 2051, x, ew, tab, plain);
    for (int nf1 : {192, 1728}) measure(0.0, 0.5 * w * 2 * pi / (2 * nf1), nf1 / 2 + 1, x, ew, tab, plain);
  }
  for (const Err& e : {tab, plain}) std::printf("%.4e %.4e %.4e\n", e.abs, e.rel, std::sqrt(e.square));
  return 0;
}
