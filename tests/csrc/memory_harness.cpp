// Host side of the eigenpair imager and of the buffer pool on the stub runtime, one scenario
// per run (its name is the argument).
#include "hip_stub.hpp"

#include "../../bipp_amd/csrc/imager.cpp"

#include <vector>

namespace bippamd {
void launch_widen(const float* in, double* out, long long n, hipStream_t) {
  for (long long i = 0; i < n; ++i) out[i] = in[i];
}
}  // namespace bippamd

namespace {

BippContextImpl* context() {
  auto* c = new BippContextImpl;
  c->impl = std::make_unique<ContextImpl>(BIPP_PU_GPU);
  return c;
}

struct Imager {
  static constexpr size_t NA = 12, NB = 9, NI = 3, NP = 10;
  std::vector<float> lmn, uvw, d;
  std::vector<cplx<float>> v;
  BippImager h = nullptr;

  explicit Imager(BippContextImpl* c)
      : lmn(3 * NP, 0.25f), uvw(3 * NA * NA, 1.0f), d(NI * NB, 2.0f), v(NA * NB, mk<float>(3, 4)) {
    EXPECT(bipp_imager_create(c, BIPP_COMPUTE_MIXED, 2, NA, NB, NI, NP, lmn.data(), NP, &h) ==
           BIPP_SUCCESS);
  }
  BippError add() {
    return bipp_imager_add(h, 2.0f, 0.5f, uvw.data(), NA * NA, v.data(), NA, d.data(), NB);
  }
};

// Pinned memory runs out while the staging buffers grow, at the k-th allocation of that growth:
// the add fails, the ones after it stay inside the buffers.
void staging_growth_fails() {
  for (int staged : {16, 64}) {
    int failed = 0;
    for (int k = 0;; ++k, ++failed) {
      Imager im(context());
      for (int q = 0; q < staged; ++q) EXPECT(im.add() == BIPP_SUCCESS);
      stub::pin.fail_after = k;
      const BippError e = im.add();
      stub::pin.fail_after = -1;
      for (int q = 0; q < staged; ++q) EXPECT(im.add() == BIPP_SUCCESS);
      EXPECT(stub::intact(stub::pin));
      size_t n = 0;
      EXPECT(bipp_imager_num_added(im.h, &n) == BIPP_SUCCESS);
      EXPECT(n == 2 * (size_t)staged + (e == BIPP_SUCCESS));
      if (e == BIPP_SUCCESS) break;
    }
    EXPECT(failed > 0);
  }
}

// A batch that fails after its first upload was enqueued: the stream is waited for before the call
// returns, since the staging buffers are written or handed on next.
void failed_flush_waits() {
  Imager im(context());
  for (int k = 0; k < 3; ++k) EXPECT(im.add() == BIPP_SUCCESS);
  float out[Imager::NP];
  stub::dev.fail_after = 1;
  const int before = stub::stream_waits;
  EXPECT(bipp_imager_get(im.h, 0, out) != BIPP_SUCCESS);
  EXPECT(stub::dev.fail_after == 0 && stub::stream_waits > before);
}

// Blocks that a context's pool holds go back when an allocation fails for want of them: in a
// buffer outside any scope (as those of synthesis handles and batched eigensolves are), in
// another context's scope, and for pinned memory.
void pool_gives_way() {
  BippContextImpl *a = context(), *b = context();
  {
    PoolScope scope(a->impl->pool);
    DevBuf d;
    d.get(40 << 20);
    PinnedBuf p;
    p.get(20 << 20);
  }
  EXPECT(stub::dev.used == 40 << 20 && stub::pin.used == 20 << 20);  // held, not in use
  stub::dev.limit = 64 << 20;
  stub::pin.limit = 32 << 20;
  {
    DevBuf d;
    EXPECT(d.get(50 << 20));
    EXPECT(stub::dev.used == 50 << 20);
  }
  EXPECT(stub::dev.used == 0);
  {
    PoolScope scope(a->impl->pool);
    DevBuf d;
    d.get(40 << 20);
    PinnedBuf p;
    p.get(20 << 20);
  }
  {
    PoolScope scope(b->impl->pool);
    DevBuf d;
    EXPECT(d.get(60 << 20));
    PinnedBuf p;
    EXPECT(p.get(30 << 20));
  }
  // with nothing left to give back the failure is reported, and the next call succeeds
  DevBuf d;
  bool threw = false;
  try {
    d.get(65 << 20);
  } catch (const BippException&) {
    threw = true;
  }
  EXPECT(threw && d.p == nullptr && d.cap == 0);
  EXPECT(d.get(64 << 20));
  d.drop();
  // a context that is gone is no longer asked
  b->release();
  stub::dev.fail_after = 0;
  threw = false;
  try {
    d.get(1);
  } catch (const BippException&) {
    threw = true;
  }
  EXPECT(threw);
}

}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "staging_growth_fails")
    staging_growth_fails();
  else if (name == "failed_flush_waits")
    failed_flush_waits();
  else if (name == "pool_gives_way")
    pool_gives_way();
  else
    return 2;
  return 0;
}
