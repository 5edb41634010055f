// Eigenpair imager: stage B of image synthesis on eigenpairs a dataset already holds.
//
// Replaces the per-sample loop of nufft_synthesis (src/nufft_synthesis.cpp:74-170) and the
// NUFFTInterface::add / get_image pair behind it (src/nufft_interface.hpp:13-21,
// src/gpu/nufft.hpp:28-235).  Samples are staged in pinned host memory until a batch is full
// (the reference's sampleBatchSize, src/nufft_synthesis.cpp:97-103), then one launch turns
// every (sample, image) into virtual visibilities VV = V diag(scale dScaled) V^H
// (src/host/virtual_vis.cpp:19-73) and one partitioned type-3 NUFFT, or the direct sum,
// adds Re sum_ij VV_ij exp(+i uvw_ij . x) to every image.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "bipp_hip.h"
#include "eig_host.hpp"
#include "host_runtime.hpp"
#include "imager_prep.hpp"
#include "kernels.hpp"
#include "nufft_host.hpp"

using namespace bippamd;

struct BippImagerImpl {
  BippContextImpl* ctx = nullptr;
  BippCompute compute = BIPP_COMPUTE_MIXED;
  int imager = 2;
  int n_ant = 0, n_beam = 0, n_img = 0, n_pix = 0;
  N3Options opt;
  size_t batch_req = 0;  // requested samples per batch, 0: automatic
  size_t batch = 0;      // samples per batch
  size_t staged = 0;     // samples that the staging buffers hold
  size_t count = 0;      // staged samples
  size_t n_added = 0;
  double pix_lo[3] = {0, 0, 0}, pix_hi[3] = {0, 0, 0};
  PinnedBuf h_uvw, h_v, h_d, h_sc, h_wl;
  DevBuf d_uvw, d_v, d_d, d_sc, d_wl, v_r, w_r, uvw_scale, antisym, lmn64, lmn32, img;
  DevBuf vv, uvw_r;
  N3Runner<float> n3f;
  N3Runner<double> n3d;

  bool img_double() const { return compute == BIPP_COMPUTE_FP64; }
  size_t nn() const { return (size_t)n_ant * n_ant; }
  size_t sample_bytes() const {
    return sizeof(float) * 3 * nn() + 8 * (size_t)n_ant * n_beam +
           sizeof(float) * ((size_t)n_img * n_beam + 2);
  }

  // Room for one more staged sample.  The buffers grow with the samples that come (pinning a
  // whole batch of several hundred MB for a few samples took most of a call).
  void ensure_staging() {
    if (!batch) {
      size_t b = batch_req;
      if (b == 0) {
        // the reference's automatic batch: about 2 GB of points at 20 bytes per baseline
        b = std::max<size_t>(1, 2000000000ULL / (20ULL * nn()));
        b = std::min<size_t>(b, 4096);
      }
      // staging stays within 1 GiB of pinned memory
      batch = std::max<size_t>(1, std::min<size_t>(b, (1ULL << 30) / sample_bytes()));
      staged = std::min(staged, batch);
    }
    if (count < staged) return;
    const size_t room = std::min(batch, std::max<size_t>(16, 2 * staged));
    grow(h_uvw, sizeof(float) * 3 * nn(), room);
    grow(h_v, 8 * (size_t)n_ant * n_beam, room);
    grow(h_d, sizeof(float) * (size_t)n_img * n_beam, room);
    grow(h_sc, sizeof(float), room);
    grow(h_wl, sizeof(float), room);
    staged = room;  // only now: an allocation that failed above leaves the old room
  }
  // `b` with room for `room` samples of `bytes` each, the first `count` kept
  void grow(PinnedBuf& b, size_t bytes, size_t room) {
    if (b.cap >= bytes * room) return;
    PinnedBuf n;
    n.get(bytes * room);
    if (count) std::memcpy(n.p, b.p, bytes * count);
    n.swap(b);
  }

  void add(float wl, float scale, const float* uvw, size_t lduvw, const void* v, size_t ldv,
           const float* dsc, size_t ldd) {
    ensure_staging();
    const size_t k = count;
    float* u = static_cast<float*>(h_uvw.p) + k * 3 * nn();
    for (int c3 = 0; c3 < 3; ++c3) std::memcpy(u + c3 * nn(), uvw + c3 * lduvw, sizeof(float) * nn());
    unsigned char* vd = static_cast<unsigned char*>(h_v.p) + k * 8 * (size_t)n_ant * n_beam;
    for (int e = 0; e < n_beam; ++e)
      std::memcpy(vd + 8 * (size_t)e * n_ant, static_cast<const unsigned char*>(v) + 8 * (size_t)e * ldv,
                  8 * (size_t)n_ant);
    float* dd = static_cast<float*>(h_d.p) + k * (size_t)n_img * n_beam;
    for (int l = 0; l < n_img; ++l)
      std::memcpy(dd + (size_t)l * n_beam, dsc + (size_t)l * ldd, sizeof(float) * n_beam);
    static_cast<float*>(h_sc.p)[k] = scale;
    static_cast<float*>(h_wl.p)[k] = wl;
    ++count;
    ++n_added;
    if (count == batch) flush();
  }

  void flush() {
    if (!count) return;
    const int nS = static_cast<int>(count);
    count = 0;  // a failure below drops the staged samples
    try {
      process(nS);
    } catch (...) {
      // the staging buffers may still be read by an upload
      (void)hipStreamSynchronize(ctx->impl->stream);
      throw;
    }
    ctx->impl->sync();  // the staging buffers are refilled by the next add
  }

  // uploads the staged samples and adds them to the images, on the stream
  void process(int nS) {
    hipStream_t st = ctx->impl->stream;
    float* du = d_uvw.as<float>(3 * nn() * nS);
    BIPP_HIP(hipMemcpyAsync(du, h_uvw.p, sizeof(float) * 3 * nn() * nS, hipMemcpyHostToDevice, st));
    void* dv = d_v.get(8 * (size_t)n_ant * n_beam * nS);
    BIPP_HIP(hipMemcpyAsync(dv, h_v.p, 8 * (size_t)n_ant * n_beam * nS, hipMemcpyHostToDevice, st));
    float* dd = d_d.as<float>((size_t)n_img * n_beam * nS);
    BIPP_HIP(hipMemcpyAsync(dd, h_d.p, sizeof(float) * n_img * n_beam * nS, hipMemcpyHostToDevice, st));
    float* ds = d_sc.as<float>(nS);
    BIPP_HIP(hipMemcpyAsync(ds, h_sc.p, sizeof(float) * nS, hipMemcpyHostToDevice, st));
    float* dw = d_wl.as<float>(nS);
    BIPP_HIP(hipMemcpyAsync(dw, h_wl.p, sizeof(float) * nS, hipMemcpyHostToDevice, st));
    std::vector<float> hwl(static_cast<float*>(h_wl.p), static_cast<float*>(h_wl.p) + nS);
    if (compute == BIPP_COMPUTE_FP32)
      run<float, float>(nS, du, dv, dd, ds, dw, hwl, n3f);
    else if (compute == BIPP_COMPUTE_FP64)
      run<double, double>(nS, du, dv, dd, ds, dw, hwl, n3d);
    else
      run<double, float>(nS, du, dv, dd, ds, dw, hwl, n3f);
  }

  // R: virtual-visibility precision; TG: NUFFT grid and image precision
  template <typename R, typename TG>
  void run(int nS, const float* du, const void* dv, const float* dd, const float* ds,
           const float* dw, const std::vector<float>& hwl, N3Runner<TG>& n3) {
    ContextImpl& c = *ctx->impl;
    hipStream_t st = c.stream;
    EigPairPrep<R> pp;
    pp.n_ant = n_ant;
    pp.n_beam = n_beam;
    pp.n_img = n_img;
    pp.v_in = static_cast<const cplx<float>*>(dv);
    pp.d_in = dd;
    pp.scale = ds;
    pp.wl = dw;
    pp.v_out = v_r.as<cplx<R>>((size_t)n_ant * n_beam * nS);
    pp.w_out = w_r.as<R>((size_t)n_img * n_beam * nS);
    pp.uvw_scale = uvw_scale.as<double>(nS);
    launch_eigpair_prep<R>(pp, nS, st);
    const double* l64 = static_cast<const double*>(lmn64.p);
    N3Source src;
    src.mode = N3_SRC_UVW;
    src.n_ant_max = n_ant;
    src.n_rows_const = n_ant;
    src.uvw = du;
    src.uvw_stride = 3LL * nn();
    src.lduvw = (long long)nn();
    src.uvw_scale = pp.uvw_scale;
    if (imager == 2 || compute != BIPP_COMPUTE_FP32) {
      unsigned char* anti = antisym.as<unsigned char>(nS);
      src.antisym = anti;
      launch_uvw_antisym(src, nS, anti, st);
    }
    if (imager == 2) {
      n3.template values<R>(c, nS, n_img, n_beam, n_ant, nullptr, pp.v_out,
                            (long long)n_ant * n_beam, n_ant, pp.w_out);
      n3.image(c, src, nS, n_img, opt, pix_lo, pix_hi, l64, n_pix, img.p,
               compute == BIPP_COMPUTE_FP32);
      return;
    }
    if (compute != BIPP_COMPUTE_FP32) {
      n3.template direct<R>(c, src, nS, n_img, n_beam, pp.v_out, (long long)n_ant * n_beam, n_ant,
                            pp.w_out, l64, n_pix, static_cast<TG*>(img.p));
      return;
    }
    // float32 direct sum per (sample, image) of the reference's arithmetic, float32 phases
    // (src/host/kernels/nuft_sum.cpp)
    if constexpr (sizeof(R) == 4) {
      const long long n2 = (long long)nn();
      cplx<R>* vvb = vv.as<cplx<R>>(n2);
      const R* lm = static_cast<const R*>(lmn32.p);
      for (int k = 0; k < nS; ++k) {
        const double sc = 2.0 * 3.14159265358979323846 / static_cast<double>(hwl[k]);
        const float* uk = du + (size_t)k * 3 * n2;
        R* u = uvw_r.as<R>(3 * n2);
        for (int l = 0; l < n_img; ++l) {
          launch_virtual_vis<R>(1, n_ant, n_beam, pp.v_out + (size_t)k * n_ant * n_beam, n_ant, 0,
                                pp.w_out + ((size_t)k * n_img + l) * n_beam, 0, vvb, 0, st);
          launch_scale_uvw<R>(n2, uk, n2, sc, u, u + n2, u + 2 * n2, st);
          launch_nuft_sum<R>(R(1), (int)n2, vvb, u, u + n2, u + 2 * n2, n_pix, lm, lm + n_pix,
                             lm + 2 * (size_t)n_pix, static_cast<R*>(img.p) + (size_t)l * n_pix, st);
        }
      }
    }
  }
};

extern "C" {

BippError bipp_imager_create(BippContext ctx, BippCompute compute, int imager, size_t nAntenna,
                             size_t nBeam, size_t nImages, size_t nPixel, const float* lmn,
                             size_t ldlmn, BippImager* out) {
  return guard([&] {
    require(ctx && out, BIPP_INVALID_HANDLE_ERROR, "null handle");
    require(lmn != nullptr, BIPP_INVALID_POINTER_ERROR, "null pixel array");
    require(imager == 1 || imager == 2, BIPP_INVALID_PARAMETER_ERROR,
            "imager must be 1 (direct sum) or 2 (type-3 NUFFT)");
    require(nAntenna >= 1 && nAntenna <= 4096, BIPP_INVALID_PARAMETER_ERROR,
            "number of antennas must be in [1, 4096]");
    require(nBeam >= 1 && nBeam <= 4096, BIPP_INVALID_PARAMETER_ERROR,
            "number of beams must be in [1, 4096]");
    require(nImages >= 1 && nImages <= 64, BIPP_INVALID_PARAMETER_ERROR,
            "number of images must be in [1, 64]");
    require(nPixel >= 1 && nPixel < (1ULL << 31), BIPP_INVALID_PARAMETER_ERROR,
            "number of pixels out of range");
    require(ldlmn >= nPixel, BIPP_INVALID_PARAMETER_ERROR, "ldlmn < nPixel");
    require(compute == BIPP_COMPUTE_FP64 || compute == BIPP_COMPUTE_FP32 ||
                compute == BIPP_COMPUTE_MIXED,
            BIPP_INVALID_PARAMETER_ERROR, "unknown compute mode");
    PoolScope scope(ctx->impl->pool);
    auto h = std::make_unique<BippImagerImpl>();
    h->ctx = ctx;
    h->compute = compute;
    h->imager = imager;
    h->n_ant = (int)nAntenna;
    h->n_beam = (int)nBeam;
    h->n_img = (int)nImages;
    h->n_pix = (int)nPixel;
    hipStream_t st = ctx->impl->stream;
    // eight running extremes per component (the compiler keeps them in a vector register);
    // each starts from the first pixel and moves on a strict comparison
    for (int c3 = 0; c3 < 3; ++c3) {
      const float* v = lmn + c3 * ldlmn;
      float lo[8], hi[8];
      for (int k = 0; k < 8; ++k) lo[k] = hi[k] = v[0];
      size_t q = 0;
      for (; q + 8 <= nPixel; q += 8)
        for (int k = 0; k < 8; ++k) {
          lo[k] = v[q + k] < lo[k] ? v[q + k] : lo[k];
          hi[k] = v[q + k] > hi[k] ? v[q + k] : hi[k];
        }
      for (; q < nPixel; ++q) {
        lo[0] = v[q] < lo[0] ? v[q] : lo[0];
        hi[0] = v[q] > hi[0] ? v[q] : hi[0];
      }
      for (int k = 1; k < 8; ++k) {
        lo[0] = lo[k] < lo[0] ? lo[k] : lo[0];
        hi[0] = hi[k] > hi[0] ? hi[k] : hi[0];
      }
      h->pix_lo[c3] = lo[0];
      h->pix_hi[c3] = hi[0];
    }
    float* d32 = h->lmn32.as<float>(3 * nPixel);
    for (int c3 = 0; c3 < 3; ++c3)
      BIPP_HIP(hipMemcpyAsync(d32 + c3 * nPixel, lmn + c3 * ldlmn, sizeof(float) * nPixel,
                              hipMemcpyHostToDevice, st));
    launch_widen(d32, h->lmn64.as<double>(3 * nPixel), 3LL * nPixel, st);
    const size_t isz = h->img_double() ? 8 : 4;
    void* im = h->img.get(isz * nImages * nPixel);
    BIPP_HIP(hipMemsetAsync(im, 0, isz * nImages * nPixel, st));
    BIPP_HIP(hipStreamSynchronize(st));
    ctx->retain();
    *out = h.release();
  });
}

BippError bipp_imager_destroy(BippImager h) {
  return guard([&] {
    if (!h) return;
    BippContextImpl* c = h->ctx;
    (void)hipStreamSynchronize(c->impl->stream);
    delete h;
    c->release();
  });
}

BippError bipp_imager_set_tolerance(BippImager h, double tol) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    require(tol > 0 && tol < 1, BIPP_INVALID_PARAMETER_ERROR, "tolerance must be in (0, 1)");
    h->opt.tol = tol;
  });
}

BippError bipp_imager_set_partition(BippImager h, int method, const size_t* dims) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    set_partition(h->opt, method, dims);
  });
}

BippError bipp_imager_set_sample_batch_size(BippImager h, size_t n) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    require(h->count == 0, BIPP_INVALID_PARAMETER_ERROR,
            "the sample batch size cannot change while samples are staged");
    h->batch_req = n;
    h->batch = 0;
  });
}

BippError bipp_imager_add(BippImager h, float wl, float scale, const float* uvw, size_t lduvw,
                          const void* v, size_t ldv, const float* dScaled, size_t lddScaled) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    require(uvw && v && dScaled, BIPP_INVALID_POINTER_ERROR, "null array");
    require(lduvw >= h->nn() && ldv >= (size_t)h->n_ant && lddScaled >= (size_t)h->n_beam,
            BIPP_INVALID_PARAMETER_ERROR, "leading dimension too small");
    require(wl > 0, BIPP_INVALID_PARAMETER_ERROR, "wavelength must be positive");
    PoolScope scope(h->ctx->impl->pool);
    h->add(wl, scale, uvw, lduvw, v, ldv, dScaled, lddScaled);
  });
}

BippError bipp_imager_get(BippImager h, size_t imgIdx, float* image) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    require(image != nullptr, BIPP_INVALID_POINTER_ERROR, "null image");
    require(imgIdx < (size_t)h->n_img, BIPP_INVALID_PARAMETER_ERROR, "image index out of range");
    PoolScope scope(h->ctx->impl->pool);
    h->flush();
    hipStream_t st = h->ctx->impl->stream;
    if (h->img_double()) {
      std::vector<double> t(h->n_pix);
      BIPP_HIP(hipMemcpyAsync(t.data(), static_cast<double*>(h->img.p) + imgIdx * h->n_pix,
                              sizeof(double) * h->n_pix, hipMemcpyDeviceToHost, st));
      BIPP_HIP(hipStreamSynchronize(st));
      for (int q = 0; q < h->n_pix; ++q) image[q] = static_cast<float>(t[q]);
    } else {
      BIPP_HIP(hipMemcpyAsync(image, static_cast<float*>(h->img.p) + imgIdx * h->n_pix,
                              sizeof(float) * h->n_pix, hipMemcpyDeviceToHost, st));
      BIPP_HIP(hipStreamSynchronize(st));
    }
  });
}

BippError bipp_imager_num_added(BippImager h, size_t* n) {
  return guard([&] {
    require(h && n, BIPP_INVALID_HANDLE_ERROR, "null handle");
    *n = h->n_added;
  });
}

BippError bipp_imager_nufft_partition(BippImager h, int32_t* dims, int32_t* boxes) {
  return guard([&] {
    require(h != nullptr, BIPP_INVALID_HANDLE_ERROR, "null handle");
    const bool d64 = h->compute == BIPP_COMPUTE_FP64;
    if (dims)
      for (int d = 0; d < 3; ++d) dims[d] = d64 ? h->n3d.last_dims[d] : h->n3f.last_dims[d];
    if (boxes) *boxes = d64 ? h->n3d.last_boxes : h->n3f.last_boxes;
  });
}

}  // extern "C"
