// Launchers of the NUFFT's transforms on the stub runtime: every kernel's dynamic LDS limit is
// set before its first launch, also where the first attempt to set it failed.
#include "hip_stub.hpp"

#include "../../bipp_amd/csrc/nufft3.hip"

namespace {

using namespace bippamd;

template <typename R>
void axis(int n1, int n2) {
  N3AxisParams<R> p{};
  p.n_levels = 2;
  p.nx = 64;
  p.xw = {0, 64};
  p.no = 3;
  p.other = {0, 3};
  p.operm_n1 = p.operm_n2 = 1;
  p.axis_stride = 64;
  p.n = n1 * n2;
  p.n1 = n1;
  p.n2 = n2;
  p.in = p.out = {0, p.n};
  p.outer_stride = 64LL * p.n;
  EXPECT(launch_fft_axis<R>(p, nullptr));
}

template <typename R>
void lines(int n) {
  N3LineParams<R> p{};
  p.n_levels = 2;
  p.n = n;
  p.ny = p.nz = 5;
  p.yw = p.zw = {0, 5};
  p.in = p.out = {0, n};
  launch_fft_lines<R>(p, nullptr);
}

template <class F>
unsigned one(F launch) {
  stub::last = {};
  launch();
  std::printf("threads %u, LDS %zu, limit %zu\n", stub::last.threads, stub::last.lds, stub::last.limit);
  EXPECT(stub::last.kernel && stub::last.lds <= stub::last.limit);
  return stub::last.threads;
}

// both forms of a kernel template, the smaller workgroup first
template <typename R>
void both_forms(int s1, int s2, int l1, int l2) {
  const unsigned small = one([=] { axis<R>(s1, s2); }), large = one([=] { axis<R>(l1, l2); });
  EXPECT(small == 512 && large == 1024);
  for (int n : {16, 54, 256, 1080, 2000, 2048}) one([=] { lines<R>(n); });
}

}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "limits") {
    both_forms<float>(24, 25, 60, 80);
    both_forms<double>(24, 25, 48, 50);
  } else if (name == "limit_fails_once") {
    stub::attribute_failures = 1;
    bool threw = false;
    try {
      axis<float>(60, 80);
    } catch (const std::exception&) {
      threw = true;
    }
    EXPECT(threw && stub::launches == 0);
    one([] { axis<float>(60, 80); });
  } else {
    return 2;
  }
  return 0;
}
