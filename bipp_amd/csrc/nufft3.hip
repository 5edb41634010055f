// Type-3 NUFFT (3-D, non-uniform baselines -> non-uniform pixels) for the Bluebild
// image sum  f_l(x_q) = sum_j c_lj exp(+i u_j . x_q),  image_l += Re f_l.
//
// Replaces the neonufft PlanT3 calls of src/host/nufft.hpp:196-216 and
// src/gpu/nufft.hpp:198-216 (sign +1, real part accumulated into a float image).  The
// algorithm is the published two-stage type-3 scheme (Lee & Greengard 2005; Barnett,
// Magland & af Klinteberg 2019) with the "exponential of semicircle" kernel
// phi(z) = exp(beta (sqrt(1 - z^2) - 1)), restated per dimension as:
//   centre   u = C + u',  x = D + x';   c'_j = c_j exp(i u'_j . D)
//   rescale  t_j = u'_j / gamma,  s_q = gamma x'_q,  gamma = nf1 / (2 sigma1 S)
//   spread   b_l = sum_j c'_j psi(l h1 - t_j)                 (grid of nf1, h1 = 2 pi / nf1)
//   type 2   F(s) = sum_l b_l exp(i l h1 s)                     (deconvolve by phi2^, FFT on
//            a grid of nf2 = sigma2 nf1, interpolate at h1 s)
//   correct  f(x_q) = exp(i C . x_q) h1 F(s_q) / psi^(s_q)       (per dimension)
// The same points serve every energy level: one spread pass accumulates all levels, the
// kernel weights of a point are computed once.
//
// Data layout in HBM: grid[level][z][y][x] complex (x fastest), nf2 per axis.  Axes longer
// than 128 that are not contiguous are transformed in two passes (n = n1 n2) and keep
// their frequencies in the permuted order  position = (k mod n1) n2 + k / n1,  which the
// interpolation reads directly (no transpose passes).
#include "common.hpp"
#include "kernels.hpp"
#include "nufft3.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

namespace bippamd {

namespace {

constexpr int SP_BIN = 8;    // spread block edge: one wavefront per 8^3 block
constexpr int SP_WMAX = 16;  // largest kernel width
constexpr int SP_MAXR = 9;   // neighbour bin ranges per block: (nback + 1)^2 with nback <= 2
constexpr int FFT_NT = 512;  // FFT workgroup: ~2 radix-4 butterflies per thread per stage

template <typename R>
__device__ __forceinline__ R es_kernel(R z, R beta) {
  const R t = R(1) - z * z;
  return t > R(0) ? exp(beta * (sqrt(t) - R(1))) : R(0);
}
// float: the exponent beta (sqrt(t) - 1) lies in [-beta, 0] (beta <= 2.38 * 16), so the
// hardware base-2 exponential and square root (about 1 ulp each, normal arguments only) need
// no range reduction or denormal scaling; their error is below the ~1e-6 relative error that
// rounding the exponent itself already gives.
template <>
__device__ __forceinline__ float es_kernel<float>(float z, float beta) {
  const float t = 1.0f - z * z;
  const float e = __builtin_amdgcn_exp2f(beta * 1.44269504088896341f *
                                         (__builtin_amdgcn_sqrtf(fmaxf(t, 0.0f)) - 1.0f));
  return t > 0.0f ? e : 0.0f;
}

// phi(xi) (the Fourier transform of the kernel) from its table by the cubic through the four
// nearest entries; phi is even and the table starts one step below zero.
__device__ __forceinline__ double ft_lookup(const double* tab, int n, double inv_delta,
                                            double xi) {
  const double u = fabs(xi) * inv_delta + 1.0;
  int k = static_cast<int>(u);
  k = min(max(k, 1), n - 3);
  const double t = u - k;
  const double tm1 = t - 1.0, tm2 = t - 2.0, tp1 = t + 1.0;
  return tab[k - 1] * (-t * tm1 * tm2 / 6.0) + tab[k] * (tp1 * tm1 * tm2 / 2.0) +
         tab[k + 1] * (-tp1 * t * tm2 / 2.0) + tab[k + 2] * (tp1 * t * tm1 / 6.0);
}

// --------------------------------------------------------------------------------------
// Points of a slot (sample s, slot t): whether the slot carries a point, its u (radians per
// unit direction cosine), the offset of its value in the sample's VV matrix (lower
// triangle), whether that value is conjugated, and its multiplicity.
// --------------------------------------------------------------------------------------
struct SlotPoint {
  double u[3];
  int src;
  int conj;
  float mult;
};

__device__ __forceinline__ bool slot_point(const N3Source& p, int s, long long t, SlotPoint& sp) {
  const int n = p.n_rows ? p.n_rows[s] : p.n_rows_const;
  if (p.mode == N3_SRC_PAIRS) {
    // column-major lower triangle: t = T(b) + (a - b), T(b) = b (2 N - b + 1) / 2
    const long long N = p.n_ant_max;
    const double q = 2.0 * N + 1.0;
    int b = static_cast<int>(floor(0.5 * (q - sqrt(q * q - 8.0 * static_cast<double>(t)))));
    auto T = [&](long long c) { return c * (2 * N - c + 1) / 2; };
    if (b < 0) b = 0;
    if (b > N - 1) b = static_cast<int>(N - 1);
    while (b > 0 && T(b) > t) --b;          // guard rounding of the square root
    while (b < N - 1 && T(b + 1) <= t) ++b;
    const int a = static_cast<int>(t - T(b)) + b;
    if (a >= n || (p.merge_auto && a == b && a > 0)) return false;
    const double* pos = p.pos + (size_t)s * p.pos_stride;  // [3][apad] positions / wavelength
#pragma unroll
    for (int d = 0; d < 3; ++d)
      sp.u[d] = 6.283185307179586 * (pos[d * p.apad + a] - pos[d * p.apad + b]);
    // the merged a == b point reads the trace slot (0, 1)
    sp.src = (p.merge_auto && a == b) ? static_cast<int>(p.ld_vv) : static_cast<int>(a + p.ld_vv * b);
    sp.conj = 0;
    sp.mult = a == b ? 1.f : 2.f;  // (a,b) and (b,a) are conjugate: 2 Re(.)
    return true;
  }
  const int N = p.n_ant_max;
  const int j = static_cast<int>(t / N), i = static_cast<int>(t - (long long)j * N);
  if (i >= n || j >= n) return false;
  const bool anti = p.antisym[s] != 0;
  if (anti && i < j) return false;                           // stands with its mirror (j, i)
  if (anti && p.merge_auto && i == j && i > 0) return false;  // diagonal merged at (0, 0)
  const float* uv = p.uvw + (size_t)s * p.uvw_stride + (i + (long long)N * j);
  const double sc = p.uvw_scale[s];
#pragma unroll
  for (int d = 0; d < 3; ++d) sp.u[d] = sc * static_cast<double>(uv[d * p.lduvw]);
  if (anti && p.merge_auto && i == j) {
    sp.src = static_cast<int>(p.ld_vv);
    sp.conj = 0;
  } else if (i >= j) {
    sp.src = static_cast<int>(i + p.ld_vv * j);
    sp.conj = 0;
  } else {
    sp.src = static_cast<int>(j + p.ld_vv * i);  // VV(i, j) = conj(VV(j, i))
    sp.conj = 1;
  }
  sp.mult = (anti && i != j) ? 2.f : 1.f;
  return true;
}

// Point records: one thread per listed slot (or per slot of every sample); counts per bin
// and each point's rank in its bin (fill = 0), or the records and values written into their
// bins' sorted ranges at those ranks (fill = 1).  Both launches compute a point's bin from
// the same operations.
__global__ void n3_points_kernel(N3PointsParams p) {
  const long long sps = p.src.slots_per_sample();
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= p.n_list) return;
  const unsigned long long slot = p.slot_list ? p.slot_list[i] : static_cast<unsigned long long>(i);
  const int s = static_cast<int>(slot / sps);
  const long long t = static_cast<long long>(slot - (unsigned long long)s * sps);
  SlotPoint sp;
  if (!slot_point(p.src, s, t, sp)) return;
  double cell[3];
  N3Point pt;
  int bin[3];
  double ph = 0;
  for (int d = 0; d < 3; ++d) {
    const double up = sp.u[d] - p.C[d];
    ph += up * p.D[d];
    cell[d] = up * p.inv_gh[d];  // t / h1 in grid units
    if (p.phase_fp32) cell[d] = static_cast<double>(static_cast<float>(up) * static_cast<float>(p.inv_gh[d]));
    const int l0 = static_cast<int>(ceil(cell[d] - 0.5 * p.w));
    pt.fr[d] = static_cast<float>(cell[d] - l0);
    pt.l0[d] = l0 + p.off[d];
    // the plan keeps every support inside [-nf1/2, nf1/2); the clamp only keeps the bin
    // index in range (cells outside a block are never written by it)
    bin[d] = min(max(pt.l0[d], 0) / p.bin_size[d], p.nbins[d] - 1);
  }
  const int binid = (bin[2] * p.nbins[1] + bin[1]) * p.nbins[0] + bin[0];
  if (!p.fill) {
    p.rank[i] = atomicAdd(&p.bin_count[binid], 1u);
    return;
  }
  const unsigned dst = p.bin_start[binid] + p.rank[i];
  double ps, pc;
  if (p.phase_fp32) {
    float fs, fc;
    const float fph = static_cast<float>(sp.u[0] - p.C[0]) * static_cast<float>(p.D[0]) +
                      static_cast<float>(sp.u[1] - p.C[1]) * static_cast<float>(p.D[1]) +
                      static_cast<float>(sp.u[2] - p.C[2]) * static_cast<float>(p.D[2]);
    sincosf(fph, &fs, &fc);
    ps = fs;
    pc = fc;
  } else {
    const double turns = ph * 0.15915494309189535;
    const double f = turns - rint(turns);
    sincospi(2.0 * f, &ps, &pc);
  }
  // the multiplicity (1 or 2) scales the pre-phase exactly
  pt.ph[0] = static_cast<float>(pc) * sp.mult;
  pt.ph[1] = static_cast<float>(ps) * sp.mult;
  p.pts[dst] = pt;
  // the point's values of every level, conjugated for an upper-triangle entry
  const float sgn = sp.conj ? -1.f : 1.f;
  if (p.vv_double) {
    const cplx<double>* v = static_cast<const cplx<double>*>(p.vv) + (size_t)s * p.n_levels * p.vv_stride + sp.src;
    cplx<double>* o = static_cast<cplx<double>*>(p.vals) + (size_t)dst * p.n_levels;
    for (int lv = 0; lv < p.n_levels; ++lv) {
      const cplx<double> c = v[(size_t)lv * p.vv_stride];
      o[lv] = mk<double>(c.re, sgn * c.im);
    }
  } else {
    const cplx<float>* v = static_cast<const cplx<float>*>(p.vv) + (size_t)s * p.n_levels * p.vv_stride + sp.src;
    cplx<float>* o = static_cast<cplx<float>*>(p.vals) + (size_t)dst * p.n_levels;
    for (int lv = 0; lv < p.n_levels; ++lv) {
      const cplx<float> c = v[(size_t)lv * p.vv_stride];
      o[lv] = mk<float>(c.re, sgn * c.im);
    }
  }
}

// One workgroup per sample: is its uvw antisymmetric with a zero diagonal?  (Exact float
// comparisons: baselines formed as p_i - p_j satisfy it exactly.)
__global__ __launch_bounds__(256) void uvw_antisym_kernel(N3Source p, unsigned char* out) {
  const int s = blockIdx.x;
  const int N = p.n_ant_max;
  const float* uv = p.uvw + (size_t)s * p.uvw_stride;
  int bad = 0;
  for (long long t = threadIdx.x; t < (long long)N * N && !bad; t += blockDim.x) {
    const int j = static_cast<int>(t / N), i = static_cast<int>(t - (long long)j * N);
    if (i < j) continue;
    for (int d = 0; d < 3; ++d) {
      const float a = uv[i + (long long)N * j + d * p.lduvw];
      const float b = uv[j + (long long)N * i + d * p.lduvw];
      if (i == j ? a != 0.0f : a != -b) bad = 1;
    }
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) out[s] = bad ? 0 : 1;
}

// min / max of u over the points of item k (a sample, or a listed range of slots), the item's
// slots split over gridDim.y workgroups; workgroup (k, y) writes out[6 (k gridDim.y + y)].
__global__ __launch_bounds__(256) void slot_range_kernel(N3Source p,
                                                         const unsigned long long* list,
                                                         const unsigned* begin,
                                                         const unsigned* count, double* out) {
  __shared__ double red[2][3][256];
  const int k = blockIdx.x;
  const long long sps = p.slots_per_sample();
  const long long n = list ? static_cast<long long>(count[k]) : sps;
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  const long long step = (long long)blockDim.x * gridDim.y;
  for (long long i = blockIdx.y * (long long)blockDim.x + threadIdx.x; i < n; i += step) {
    const unsigned long long slot =
        list ? list[static_cast<long long>(begin[k]) + i] : (unsigned long long)k * sps + i;
    const int s = static_cast<int>(slot / sps);
    SlotPoint sp;
    if (!slot_point(p, s, static_cast<long long>(slot - (unsigned long long)s * sps), sp)) continue;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lo[d] = fmin(lo[d], sp.u[d]);
      hi[d] = fmax(hi[d], sp.u[d]);
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    red[0][d][threadIdx.x] = lo[d];
    red[1][d][threadIdx.x] = hi[d];
  }
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        red[0][d][threadIdx.x] = fmin(red[0][d][threadIdx.x], red[0][d][threadIdx.x + off]);
        red[1][d][threadIdx.x] = fmax(red[1][d][threadIdx.x], red[1][d][threadIdx.x + off]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 3) {
    double* o = out + 6 * ((size_t)k * gridDim.y + blockIdx.y);
    o[threadIdx.x] = red[0][threadIdx.x][0];
    o[3 + threadIdx.x] = red[1][threadIdx.x][0];
  }
}

// The partial ranges of an item (`parts` of them, parts <= 64) into one; a wavefront per item.
__global__ __launch_bounds__(64) void slot_range_reduce_kernel(const double* part, int parts,
                                                               double* out) {
  const int k = blockIdx.x;
  const double* q = part + 6 * ((size_t)k * parts + threadIdx.x);
#pragma unroll
  for (int d = 0; d < 6; ++d) {
    double v = static_cast<int>(threadIdx.x) < parts ? q[d] : (d < 3 ? 1e300 : -1e300);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const double o = __shfl_xor(v, m, 64);
      v = d < 3 ? fmin(v, o) : fmax(v, o);
    }
    if (threadIdx.x == 0) out[6 * (size_t)k + d] = v;
  }
}

// Slots per workgroup of the box assignment and of the counting sort by box, and the number
// of boxes up to which a workgroup counts in LDS and adds its totals with one atomic per box.
// A few boxes hold all points, so one atomic per point serialises on their counters: 11.0 ms
// for 1.6 million slots in two boxes, each of the two kernels, against 0.03 ms.  Above the bound
// the points spread over so many counters that the totals would save nothing (at least 8
// slots per box and workgroup below it).
constexpr int PART_PER = 16;
constexpr int PART_LDS_GROUPS = 512;

// Box of every slot's point (-1 without a point) and the point count of every box.
__global__ __launch_bounds__(256) void n3_partition_kernel(N3PartParams p, int n_groups) {
  __shared__ unsigned cnt[PART_LDS_GROUPS];
  const bool lds = n_groups <= PART_LDS_GROUPS;
  if (lds) {
    for (int g = threadIdx.x; g < n_groups; g += 256) cnt[g] = 0;
    __syncthreads();
  }
  const long long sps = p.src.slots_per_sample();
  const long long n_slots = sps * p.n_samples;
  const long long i0 = blockIdx.x * (256LL * PART_PER) + threadIdx.x;
  for (int r = 0; r < PART_PER; ++r) {
    const long long i = i0 + 256LL * r;
    if (i >= n_slots) break;
    const int s = static_cast<int>(i / sps);
    SlotPoint sp;
    if (!slot_point(p.src, s, i - (long long)s * sps, sp)) {
      p.group_of[i] = -1;
      continue;
    }
    int g = 0;
    for (int d = 2; d >= 0; --d) {
      const double x = p.inv[d] * (sp.u[d] - p.lo[d]);
      const int k = x > 0.0 ? static_cast<int>(fmin(x, static_cast<double>(p.dims[d] - 1))) : 0;
      g = g * p.dims[d] + k;
    }
    p.group_of[i] = g;
    atomicAdd(lds ? &cnt[g] : &p.group_count[g], 1u);
  }
  if (!lds) return;
  __syncthreads();
  for (int g = threadIdx.x; g < n_groups; g += 256)
    if (cnt[g]) atomicAdd(&p.group_count[g], cnt[g]);
}

// slot ids in box order (counting sort)
__global__ __launch_bounds__(256) void n3_group_scatter_kernel(long long n_slots, int n_groups,
                                                               const int* group_of,
                                                               const unsigned* group_start,
                                                               unsigned* group_fill,
                                                               unsigned long long* list) {
  __shared__ unsigned cnt[PART_LDS_GROUPS], base[PART_LDS_GROUPS];
  const long long i0 = blockIdx.x * (256LL * PART_PER) + threadIdx.x;
  if (n_groups > PART_LDS_GROUPS) {
    for (int r = 0; r < PART_PER; ++r) {
      const long long i = i0 + 256LL * r;
      if (i >= n_slots) break;
      const int g = group_of[i];
      if (g >= 0) list[group_start[g] + atomicAdd(&group_fill[g], 1u)] = static_cast<unsigned long long>(i);
    }
    return;
  }
  for (int g = threadIdx.x; g < n_groups; g += 256) cnt[g] = 0;
  __syncthreads();
  int gr[PART_PER];
  unsigned rank[PART_PER];
#pragma unroll
  for (int r = 0; r < PART_PER; ++r) {
    const long long i = i0 + 256LL * r;
    gr[r] = i < n_slots ? group_of[i] : -1;
    rank[r] = gr[r] >= 0 ? atomicAdd(&cnt[gr[r]], 1u) : 0u;
  }
  __syncthreads();
  for (int g = threadIdx.x; g < n_groups; g += 256)
    base[g] = cnt[g] ? group_start[g] + atomicAdd(&group_fill[g], cnt[g]) : 0u;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PART_PER; ++r)
    if (gr[r] >= 0) list[base[gr[r]] + rank[r]] = static_cast<unsigned long long>(i0 + 256LL * r);
}

// exclusive scan helpers (counts -> starts)
__global__ void scan_block_kernel(const unsigned* in, unsigned* out, unsigned* block_sums, int n) {
  __shared__ unsigned sh[1024];
  const int i = blockIdx.x * 1024 + threadIdx.x;
  const unsigned v = i < n ? in[i] : 0u;
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const unsigned t = threadIdx.x >= off ? sh[threadIdx.x - off] : 0u;
    __syncthreads();
    sh[threadIdx.x] += t;
    __syncthreads();
  }
  if (i < n) out[i] = sh[threadIdx.x] - v;
  if (threadIdx.x == 1023) block_sums[blockIdx.x] = sh[1023];
}

__global__ void scan_add_kernel(unsigned* out, const unsigned* block_offsets, int n) {
  const int i = blockIdx.x * 1024 + threadIdx.x;
  if (i < n) out[i] += block_offsets[blockIdx.x];
}


// --------------------------------------------------------------------------------------
// Spreading with output ownership.  One wavefront owns an 8^3 block (cells l + nf1/2 in
// [8 b, 8 b + 8) per axis) or, where blocks are few, one of gridDim.y shares of its points.
// The points of the bins that can reach the block (a point of bin c covers cells [l0, l0 + w),
// l0 in bin c) are tested 64 at a time; the ones that meet the block are kept until there are
// 64 of them, then expanded in LDS: kernel weights of the block's 8 columns, rows and slabs
// (zero outside the support) and values.
//
// Over the points q the block is the product C[(y, z)][(x, re/im), level] =
// sum_q A[(y, z)][q] B[q][(x, re/im), level] with A = wy wz and B = wx v, taken four points at
// a time by 16x16x4 matrix instructions: tile m of A holds the rows (y, z = 2 m) and
// (y, z = 2 m + 1), tile lv of B the level lv, and a lane forms its operands from a few LDS
// reads.  The 64 points are placed in the order of their first z, so that four neighbours
// reach about the same z pairs, and the tiles of the others are passed over (about 0.4 of
// them at w = 6).  The kernel is bound by the matrix instructions (32 cycles each in float,
// 16 per four points of 4 levels before the passed-over ones) and, behind them, the weights.
// Measured against sums on the vector ALU (a lane per row, four wavefronts per block, weights
// for every tested point): 500 samples of 256 antennas, 4 levels, w = 6: 9.43 to 4.27 ms (6.98
// before the kept points and the z order, 4.62 with three wavefronts per SIMD instead of four);
// two or four wavefronts per block 5.88 and 5.53 ms against 4.62, their last points filling
// fewer lanes.  12 samples of 512 antennas, 6 levels in one launch: 10.7 to 3.4 ms.
//
// The block is written once, times the deconvolution factors, with plain stores: no atomics on
// the grid, and every cell of [-nf1/2, nf1/2)^3 written by exactly one wavefront (no zero pass
// over the grid).  The sums follow the order of the points inside their bins, which the
// counting pass ranks in arrival order (the values an atomic counter returns): float images
// agree between runs to rounding, not bit for bit.
// --------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename R>
struct SpreadMfma;
template <>
struct SpreadMfma<float> {
  typedef f32x4 V4;
  static constexpr int levels = 6;  // most levels per launch: 16 result registers each
  static __device__ __forceinline__ V4 mul(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // row of result register r in lanes 16 k .. 16 k + 15
  static __device__ __forceinline__ int row(int k, int r) { return 4 * k + r; }
};
template <>
struct SpreadMfma<double> {
  typedef f64x4 V4;
  static constexpr int levels = 4;  // 32 result registers each
  static __device__ __forceinline__ V4 mul(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int k, int r) { return k + 4 * r; }
};

// rows of 8 values moved with 16-byte LDS accesses
__device__ __forceinline__ void st_row8(float* dst, const float (&v)[8]) {
  reinterpret_cast<f32x4*>(dst)[0] = f32x4{v[0], v[1], v[2], v[3]};
  reinterpret_cast<f32x4*>(dst)[1] = f32x4{v[4], v[5], v[6], v[7]};
}
__device__ __forceinline__ void st_row8(double* dst, const double (&v)[8]) {
  reinterpret_cast<f64x4*>(dst)[0] = f64x4{v[0], v[1], v[2], v[3]};
  reinterpret_cast<f64x4*>(dst)[1] = f64x4{v[4], v[5], v[6], v[7]};
}

template <typename R, int LG>
struct SpreadBatch {
  static constexpr int VS = LG <= 2 ? LG : LG <= 4 ? 4 : 8;  // levels of a row of values
  R pwx[64][SP_BIN];        // rows from the number of points up to a multiple of 4 are zero
  R pwy[64][SP_BIN];
  R pwz[64][SP_BIN];        // [z % 2][z / 2]
  R pv[64][2][VS];          // re, then im of the levels
  unsigned pend[128];       // points that meet the block, not yet added
  unsigned char tiles[64];  // z pairs that the point of a row reaches
};

// result register r of tile m (s: its levels), deconvolved, into the grid: 16 lanes store
// consecutive re and im.  Cells outside [-nf1/2, nf1/2)^3 are left out.
template <typename R, int LG>
__device__ __forceinline__ void spread_store(const N3SpreadParams<R>& p, const int (&org)[3], int m,
                                             int r, int lane, const R (&s)[LG]) {
  const int row = SpreadMfma<R>::row(lane >> 4, r);
  const int ix = org[0] + ((lane & 15) >> 1), iy = org[1] + (row & 7),
            iz = org[2] + 2 * m + (row >> 3);
  if (ix >= p.nf1[0] || iy >= p.nf1[1] || iz >= p.nf1[2]) return;
  int gx = ix - p.nf1[0] / 2, gy = iy - p.nf1[1] / 2, gz = iz - p.nf1[2] / 2;
  gx += gx < 0 ? p.nf2[0] : 0;
  gy += gy < 0 ? p.nf2[1] : 0;
  gz += gz < 0 ? p.nf2[2] : 0;
  const R f = p.fx[ix] * (p.fy[iy] * p.fz[iz]);
  R* g = reinterpret_cast<R*>(p.grid + ((size_t)gz * p.nf2[1] + gy) * p.nf2[0] + gx) + (lane & 1);
#pragma unroll
  for (int lv = 0; lv < LG; ++lv)
    g[2 * (size_t)(p.lv0 - p.lv_begin + lv) * p.grid_stride] = s[lv] * f;
}

// registers for four wavefronts per SIMD in float up to 4 levels, three above, two in double
template <typename R, int LG>
__global__ __launch_bounds__(64, sizeof(R) == 8 ? 2 : LG <= 4 ? 4 : 3) void n3_spread_kernel(N3SpreadParams<R> p) {
  constexpr int B = SP_BIN, PB = 64;
  typedef SpreadMfma<R> M;
  typedef typename M::V4 V4;
  __shared__ __align__(32) SpreadBatch<R, LG> sb;
  const int w = p.w;
  const int lane = threadIdx.x;
  // Workgroups go to the 8 XCDs in turn (workgroup i to XCD i mod 8).  With xcd_chunk > 0,
  // runs of xcd_chunk consecutive blocks go to one XCD (neighbouring blocks read overlapping
  // point ranges and then share an L2), the runs dealt to the XCDs in turn.
  int bin = static_cast<int>(blockIdx.x);
  if (p.xcd_chunk > 0) {
    const int x = bin % 8, k = bin / 8;
    bin = ((k / p.xcd_chunk) * 8 + x) * p.xcd_chunk + k % p.xcd_chunk;
  }
  if (bin >= p.nbins[0] * p.nbins[1] * p.nbins[2]) return;
  const int bx = bin % p.nbins[0];
  const int by = (bin / p.nbins[0]) % p.nbins[1];
  const int bz = bin / (p.nbins[0] * p.nbins[1]);
  const int org[3] = {bx * B, by * B, bz * B};
  V4 acc[4][LG];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int lv = 0; lv < LG; ++lv) acc[m][lv] = V4{R(0), R(0), R(0), R(0)};
  const unsigned long long t_start = p.prof ? wall_clock64() : 0;
  unsigned long long n_hit = 0;
  const R two_over_w = R(2) / R(w);
  const R beta = R(p.beta);
  // The bins that can reach the block: for each (cy, cz) of the neighbourhood the bins
  // cx = bx - nback .. bx are consecutive in the sorted point array, so the neighbourhood is
  // at most (nback + 1)^2 contiguous ranges; batches run over their concatenation.
  unsigned rbeg[SP_MAXR], rlen[SP_MAXR];
  int nr = 0;
  unsigned total_pts = 0;
  for (int cz_ = max(0, bz - p.nback[2]); cz_ <= bz; ++cz_)
    for (int cy_ = max(0, by - p.nback[1]); cy_ <= by; ++cy_) {
      const int row = (cz_ * p.nbins[1] + cy_) * p.nbins[0];
      const int lo = row + max(0, bx - p.nback[0]), hi = row + bx;
      rbeg[nr] = p.bin_start[lo];
      rlen[nr] = p.bin_start[hi] + p.bin_count[hi] - rbeg[nr];
      total_pts += rlen[nr];
      ++nr;
    }
  const unsigned n_batches = (total_pts + PB - 1) / PB;
  // operand rows and columns of the lane: A row i = lane % 16 is y = i % 8, z = 2 m + i / 8,
  // B column j = lane % 16 is x = j / 2, re or im = j % 2; both take point q0 + lane / 16
  const int i16 = lane & 15, kq = lane >> 4;

  // the first `total` (at most 64) pending points added to the sums
  auto add_pending = [&](int total) {
    const bool hit = lane < total;
    N3Point pt;
    cplx<R> vals[LG];
    int rel[3] = {0, 0, 0};
    if (hit) {
      const unsigned v = sb.pend[lane];
      pt = p.pts[v];
      const cplx<R>* pv = p.vals + (size_t)v * p.n_levels_total + p.lv0;
#pragma unroll
      for (int lv = 0; lv < LG; ++lv) vals[lv] = pv[lv];
#pragma unroll
      for (int d = 0; d < 3; ++d) rel[d] = pt.l0[d] - org[d];
    }
    // rows in the order of the points' first z: four neighbours then share most z pairs
    int slot = lane;
    {
      unsigned long long left = __ballot(hit);
      const unsigned long long below = (1ull << lane) - 1ull;
      int base = 0;
      for (int z = 1 - w; z < B && left; ++z) {
        const unsigned long long same = __ballot(hit && rel[2] == z);
        if (hit && rel[2] == z) slot = base + __popcll(same & below);
        base += __popcll(same);
        left &= ~same;
      }
    }
    if (hit) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        // column c is support offset o = c - rel of the point, at (o - fr) 2 / w: the
        // argument stepped from c = 0, the support test 0 <= o < w as one unsigned compare
        const R x0 = (R(-rel[d]) - R(pt.fr[d])) * two_over_w;
        R row[B];
#pragma unroll
        for (int c = 0; c < B; ++c)
          row[d < 2 ? c : (c & 1) * 4 + c / 2] =
              static_cast<unsigned>(c - rel[d]) < static_cast<unsigned>(w)
                  ? es_kernel<R>(x0 + R(c) * two_over_w, beta)
                  : R(0);
        st_row8(d == 0 ? sb.pwx[slot] : d == 1 ? sb.pwy[slot] : sb.pwz[slot], row);
        __builtin_amdgcn_sched_barrier(0);  // one row held at a time
      }
      const int z0 = max(rel[2], 0) >> 1, z1 = min(rel[2] + w - 1, B - 1) >> 1;
      sb.tiles[slot] = static_cast<unsigned char>((2 << z1) - (1 << z0));
      const R pr = R(pt.ph[0]), pim = R(pt.ph[1]);  // multiplicity included
#pragma unroll
      for (int lv = 0; lv < LG; ++lv) {
        sb.pv[slot][0][lv] = vals[lv].re * pr - vals[lv].im * pim;
        sb.pv[slot][1][lv] = vals[lv].re * pim + vals[lv].im * pr;
      }
    }
    if (lane >= total && lane < ((total + 3) & ~3)) {
      const R zero[B] = {R(0), R(0), R(0), R(0), R(0), R(0), R(0), R(0)};
      st_row8(sb.pwx[lane], zero);
      st_row8(sb.pwy[lane], zero);
      st_row8(sb.pwz[lane], zero);
      sb.tiles[lane] = 0;
#pragma unroll
      for (int lv = 0; lv < LG; ++lv) sb.pv[lane][0][lv] = sb.pv[lane][1][lv] = R(0);
    }
    wave_sync();
    unsigned tiles = reinterpret_cast<const unsigned*>(sb.tiles)[lane & 15];  // four rows
    tiles |= tiles >> 16;
    tiles |= tiles >> 8;
    n_hit += total;
    for (int q0 = 0; q0 < total; q0 += 4) {
      const int q = q0 + kq;
      const unsigned act = __builtin_amdgcn_readlane(tiles, q0 >> 2);
      const R wy = sb.pwy[q][i16 & 7], wx = sb.pwx[q][i16 >> 1];
      const V4 wz = *reinterpret_cast<const V4*>(&sb.pwz[q][4 * (i16 >> 3)]);
      R bv[LG];
#pragma unroll
      for (int lv = 0; lv < LG; ++lv) bv[lv] = sb.pv[q][i16 & 1][lv] * wx;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (!(act >> m & 1u)) continue;
        const R a = wy * wz[m];
#pragma unroll
        for (int lv = 0; lv < LG; ++lv)
          acc[m][lv] = M::mul(a, bv[lv], acc[m][lv]);
      }
    }
    wave_sync();  // rows consumed
  };

  int n_pend = 0;
  for (unsigned bi = blockIdx.y; bi < n_batches; bi += gridDim.y) {
    const unsigned b0 = bi * PB;
    const int nb = min<unsigned>(PB, total_pts - b0);
    bool hit = false;
    unsigned v = b0 + lane;
    if (lane < nb) {
      int r = 0;
      while (v >= rlen[r]) v -= rlen[r++];
      v += rbeg[r];
      hit = true;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int rel = p.pts[v].l0[d] - org[d];
        hit = hit && rel < B && rel + w > 0;
      }
    }
    const unsigned long long mask = __ballot(hit);
    if (hit) sb.pend[n_pend + __popcll(mask & ((1ull << lane) - 1ull))] = v;
    n_pend += __popcll(mask);
    wave_sync();
    if (n_pend >= PB) {
      add_pending(PB);
      n_pend -= PB;
      if (lane < n_pend) {
        const unsigned t = sb.pend[PB + lane];
        sb.pend[lane] = t;
      }
      wave_sync();
    }
  }
  if (n_pend > 0) add_pending(n_pend);
  if (p.prof && lane == 0 && blockIdx.y == 0) {
    unsigned long long* pr = p.prof + (size_t)bin * 4;
    pr[0] = t_start;
    pr[1] = wall_clock64();
    pr[2] = total_pts;
    pr[3] = n_hit;  // hits of the first share
  }
  if (gridDim.y > 1) {  // a share's sums: [block][share][tile][result register][level][lane]
    R* part = p.part + ((size_t)bin * gridDim.y + blockIdx.y) * (16 * LG * 64) + lane;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int lv = 0; lv < LG; ++lv) part[((m * 4 + r) * LG + lv) * 64] = acc[m][lv][r];
    return;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      R s[LG];
#pragma unroll
      for (int lv = 0; lv < LG; ++lv) s[lv] = acc[m][lv][r];
      spread_store<R, LG>(p, org, m, r, lane, s);
      __builtin_amdgcn_sched_barrier(0);  // no addresses of later stores held meanwhile
    }
}

// sums of the shares of a block (blockIdx.x), in their order: wavefront and blockIdx.y take
// result register and tile
template <typename R, int LG>
__global__ __launch_bounds__(256) void n3_spread_sum_kernel(N3SpreadParams<R> p) {
  const int bin = blockIdx.x, m = blockIdx.y, lane = threadIdx.x & 63, r = threadIdx.x >> 6;
  const int org[3] = {bin % p.nbins[0] * SP_BIN, bin / p.nbins[0] % p.nbins[1] * SP_BIN,
                      bin / (p.nbins[0] * p.nbins[1]) * SP_BIN};
  const R* part = p.part + (size_t)bin * p.shares * (16 * LG * 64) + (m * 4 + r) * LG * 64 + lane;
  R s[LG];
#pragma unroll
  for (int lv = 0; lv < LG; ++lv) s[lv] = R(0);
  for (int k = 0; k < p.shares; ++k)
#pragma unroll
    for (int lv = 0; lv < LG; ++lv) s[lv] += part[(size_t)k * (16 * LG * 64) + lv * 64];
  spread_store<R, LG>(p, org, m, r, lane, s);
}

// --------------------------------------------------------------------------------------
// Stockham FFT in LDS (sign +): `nl` lines of length n, line stride ld, radices r[].
// Returns the buffer holding the result.
// --------------------------------------------------------------------------------------
// exp(+2 pi i m / N) for the constant twiddles of the composite radices (m is a
// compile-time constant after unrolling, so the selection folds away).
template <typename R, int N>
__device__ __forceinline__ cplx<R> root_const(int m) {
  constexpr double C8 = 0.923879532511286756128, S8 = 0.382683432365089771728,
                   H2 = 0.707106781186547524401, H3 = 0.866025403784438646764;
  double c = 1, s = 0;
  if constexpr (N == 16) {
    constexpr double tc[10] = {1, C8, H2, S8, 0, -S8, -H2, -C8, -1, -C8};
    constexpr double ts[10] = {0, S8, H2, C8, 1, C8, H2, S8, 0, -S8};
    c = tc[m];
    s = ts[m];
  } else if constexpr (N == 9) {
    constexpr double tc[5] = {1, 0.766044443118978035202, 0.173648177666930348852, -0.5,
                              -0.939692620785908384054};
    constexpr double ts[5] = {0, 0.642787609686539326323, 0.984807753012208059367, H3,
                              0.342020143325668733044};
    c = tc[m];
    s = ts[m];
  } else if constexpr (N == 8) {
    constexpr double tc[4] = {1, H2, 0, -H2};
    constexpr double ts[4] = {0, H2, 1, H2};
    c = tc[m];
    s = ts[m];
  } else if constexpr (N == 10) {
    constexpr double C = 0.809016994374947424102, D = 0.309016994374947424102,
                     E = 0.587785252292473129169, F = 0.951056516295153572116;
    constexpr double tc[5] = {1, C, D, -D, -C};
    constexpr double ts[5] = {0, E, F, F, E};
    c = tc[m];
    s = ts[m];
  } else if constexpr (N == 12) {
    constexpr double tc[7] = {1, H3, 0.5, 0, -0.5, -H3, -1};
    constexpr double ts[7] = {0, 0.5, H3, 1, H3, 0.5, 0};
    c = tc[m];
    s = ts[m];
  } else if constexpr (N == 15) {
    constexpr double tc[9] = {1, 0.913545457642600895502, 0.669130606358858213826,
                              0.309016994374947424102, -0.104528463267653471400, -0.5,
                              -0.809016994374947424102, -0.978147600733805637929,
                              -0.978147600733805637929};
    constexpr double ts[9] = {0, 0.406736643075800207754, 0.743144825477394235015,
                              0.951056516295153572116, 0.994521895368273336923, H3,
                              0.587785252292473129169, 0.207911690817759337102,
                              -0.207911690817759337102};
    c = tc[m];
    s = ts[m];
  } else {
    static_assert(N == 6, "roots of the composite radices");
    constexpr double tc[3] = {1, 0.5, -0.5};
    constexpr double ts[3] = {0, H3, H3};
    c = tc[m];
    s = ts[m];
  }
  return mk<R>(static_cast<R>(c), static_cast<R>(s));
}

template <typename R, int RAD>
__device__ __forceinline__ void dft_small(cplx<R>* v);

// DFT of length N = P Q (sign +) in registers, Cooley-Tukey: input j = Q j1 + j2, output
// k = k1 + P k2, X[k] = sum_j2 w_N^(j2 k1) w_Q^(j2 k2) sum_j1 x[Q j1 + j2] w_P^(j1 k1).
template <typename R, int P, int Q>
__device__ __forceinline__ void dft_ct(cplx<R>* v) {
  constexpr int N = P * Q;
  cplx<R> f[N];
#pragma unroll
  for (int j2 = 0; j2 < Q; ++j2) {
    cplx<R> t[P];
#pragma unroll
    for (int j1 = 0; j1 < P; ++j1) t[j1] = v[Q * j1 + j2];
    dft_small<R, P>(t);
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      const int m = (j2 * k1) % N;
      f[j2 * P + k1] = m == 0 ? t[k1] : t[k1] * root_const<R, N>(m);
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < P; ++k1) {
    cplx<R> t[Q];
#pragma unroll
    for (int j2 = 0; j2 < Q; ++j2) t[j2] = f[j2 * P + k1];
    dft_small<R, Q>(t);
#pragma unroll
    for (int k2 = 0; k2 < Q; ++k2) v[k1 + P * k2] = t[k2];
  }
}

// Small DFTs with sign +, constant roots.
template <typename R, int RAD>
__device__ __forceinline__ void dft_small(cplx<R>* v) {
  if constexpr (RAD == 1) {
  } else if constexpr (RAD == 2) {
    const cplx<R> a = v[0], b = v[1];
    v[0] = a + b;
    v[1] = a - b;
  } else if constexpr (RAD == 4) {
    const cplx<R> a = v[0], b = v[1], c = v[2], d = v[3];
    const cplx<R> s0 = a + c, s1 = a - c, s2 = b + d, s3 = b - d;
    const cplx<R> is3 = mk<R>(-s3.im, s3.re);  // +i * s3
    v[0] = s0 + s2;
    v[1] = s1 + is3;
    v[2] = s0 - s2;
    v[3] = s1 - is3;
  } else if constexpr (RAD == 3) {
    // w = exp(+2 pi i / 3): y1,2 = a - (b + c)/2 +- i sqrt(3)/2 (b - c)
    const R h = R(0.86602540378443864676);
    const cplx<R> a = v[0], t1 = v[1] + v[2], t2 = v[1] - v[2];
    const cplx<R> m = mk<R>(a.re - R(0.5) * t1.re, a.im - R(0.5) * t1.im);
    const cplx<R> q = mk<R>(-h * t2.im, h * t2.re);
    v[0] = a + t1;
    v[1] = m + q;
    v[2] = m - q;
  } else if constexpr (RAD == 6) {
    dft_ct<R, 2, 3>(v);
  } else if constexpr (RAD == 8) {
    dft_ct<R, 2, 4>(v);
  } else if constexpr (RAD == 9) {
    dft_ct<R, 3, 3>(v);
  } else if constexpr (RAD == 10) {
    dft_ct<R, 2, 5>(v);
  } else if constexpr (RAD == 12) {
    dft_ct<R, 3, 4>(v);
  } else if constexpr (RAD == 15) {
    dft_ct<R, 3, 5>(v);
  } else if constexpr (RAD == 16) {
    dft_ct<R, 4, 4>(v);
  } else {
    static_assert(RAD == 5, "radix 2, 3, 4, 5, 6, 8, 9, 10, 12, 15 or 16");
    // radix 5, roots w^k = exp(+2 pi i k / 5) = c_k + i s_k with w^4 = conj(w), w^3 =
    // conj(w^2): with t1 = x1 + x4, t2 = x2 + x3, t3 = x1 - x4, t4 = x2 - x3,
    //   y1, y4 = x0 + c1 t1 + c2 t2 +- i (s1 t3 + s2 t4)
    //   y2, y3 = x0 + c2 t1 + c1 t2 +- i (s2 t3 - s1 t4)
    // (36 real operations instead of the 80 of the direct sums)
    const R c1 = R(0.30901699437494742410), c2 = R(-0.80901699437494742410);
    const R s1 = R(0.95105651629515357212), s2 = R(0.58778525229247312917);
    const cplx<R> x0 = v[0];
    const cplx<R> t1 = v[1] + v[4], t2 = v[2] + v[3], t3 = v[1] - v[4], t4 = v[2] - v[3];
    const cplx<R> a1 = mk<R>(x0.re + c1 * t1.re + c2 * t2.re, x0.im + c1 * t1.im + c2 * t2.im);
    const cplx<R> a2 = mk<R>(x0.re + c2 * t1.re + c1 * t2.re, x0.im + c2 * t1.im + c1 * t2.im);
    const cplx<R> b1 = mk<R>(s1 * t3.re + s2 * t4.re, s1 * t3.im + s2 * t4.im);
    const cplx<R> b2 = mk<R>(s2 * t3.re - s1 * t4.re, s2 * t3.im - s1 * t4.im);
    v[0] = x0 + t1 + t2;
    v[1] = mk<R>(a1.re - b1.im, a1.im + b1.re);
    v[4] = mk<R>(a1.re + b1.im, a1.im - b1.re);
    v[2] = mk<R>(a2.re - b2.im, a2.im + b2.re);
    v[3] = mk<R>(a2.re + b2.im, a2.im - b2.re);
  }
}

// exp(+2 pi i t / n) from two LDS tables: t1[t mod 64] * t2[t / 64]
template <typename R>
struct Twid {
  const cplx<R>* t1;
  const cplx<R>* t2;
  __device__ __forceinline__ cplx<R> operator()(int t) const { return t1[t & 63] * t2[t >> 6]; }
};

// table layout in global memory: [64] fine entries, then [ceil(n / 64)] coarse entries
__host__ __device__ __forceinline__ int twid_len(int n) { return 64 + (n + 63) / 64; }

template <typename R>
__device__ __forceinline__ Twid<R> load_twid(const cplx<R>* __restrict__ g, int n, cplx<R>* lds,
                                             int tid, int nt) {
  const int len = twid_len(n);
  for (int i = tid; i < len; i += nt) lds[i] = g[i];
  return Twid<R>{lds, lds + 64};
}

// x / d for 0 <= x < 2^31 from the multiplier and shift of d (N3Radix)
__device__ __forceinline__ int fast_div(int x, unsigned m, int s) {
  return static_cast<int>((__umulhi(static_cast<unsigned>(x), m) + static_cast<unsigned>(x)) >> s);
}

// One Stockham stage of radix RAD over nl lines (stride ld) of length n; (nb_m, nb_s) and
// (ns_m, ns_s) divide by n / RAD and by ns.  FIRST: the first stage (ns = 1), whose
// twiddles are all 1 (k = 0), so none are formed or applied.  TAB: the twiddles w^(k r) of
// this stage are read from its table (entry (r - 1) ns + k, build_stage_tab) instead of
// being formed from the two-level table.  ONE: a single line (nl = 1), no line index.
template <typename R, int RAD, bool FIRST, bool TAB, bool ONE>
__device__ __forceinline__ void fft_stage(const cplx<R>* in, cplx<R>* out, int n, int nl, int ld,
                                          int ns, const Twid<R>& tw, const cplx<R>* stab,
                                          int tid, int nt, unsigned nb_m, int nb_s,
                                          unsigned ns_m, int ns_s) {
  const int nb = n / RAD;
  for (int t = tid; t < (ONE ? nb : nl * nb); t += nt) {
    const int line = ONE ? 0 : fast_div(t, nb_m, nb_s), j = ONE ? t : t - line * nb;
    const cplx<R>* src = ONE ? in + j : in + (size_t)line * ld + j;
    cplx<R>* dst = ONE ? out : out + (size_t)line * ld;
    cplx<R> v[RAD];
    if constexpr (FIRST) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[r] = src[r * nb];
      dft_small<R, RAD>(v);
      dst += j * RAD;
#pragma unroll
      for (int r = 0; r < RAD; ++r) dst[r] = v[r];
      continue;
    }
    const int jq = fast_div(j, ns_m, ns_s);
    const int k = j - jq * ns;
    v[0] = src[0];
    if constexpr (TAB) {
      const cplx<R>* tk = stab + k;  // consecutive lanes read consecutive entries
#pragma unroll
      for (int r = 1; r < RAD; ++r) v[r] = src[r * nb] * tk[(r - 1) * ns];
    } else {
      // twiddles w^r, w = exp(2 pi i k tstride / n): w, w^4 and w^8 from the table, the
      // others as products at most two deep (k r tstride < n for r < RAD)
      const int tstride = n / (ns * RAD);  // twiddle k r / (ns RAD) of the full length
      const int t1 = k * tstride;
      cplx<R> wp[RAD];
      if constexpr (RAD > 1) wp[1] = tw(t1);
      if constexpr (RAD > 2) wp[2] = wp[1] * wp[1];
      if constexpr (RAD > 3) wp[3] = wp[2] * wp[1];
      if constexpr (RAD > 4) {
        wp[4] = tw(4 * t1);
#pragma unroll
        for (int r = 5; r < RAD && r < 8; ++r) wp[r] = wp[4] * wp[r - 4];
      }
      if constexpr (RAD > 8) {
        wp[8] = tw(8 * t1);
#pragma unroll
        for (int r = 9; r < RAD; ++r) wp[r] = wp[8] * wp[r - 8];
      }
#pragma unroll
      for (int r = 1; r < RAD; ++r) v[r] = src[r * nb] * wp[r];
    }
    dft_small<R, RAD>(v);
    dst += jq * ns * RAD + k;
#pragma unroll
    for (int r = 0; r < RAD; ++r) dst[r * ns] = v[r];
  }
}

// Twiddle tables of the stages after the first, one after another: stage st (span ns, radix
// RAD) holds RAD - 1 rows of ns entries, entry (r - 1) ns + k = exp(2 pi i k r tstride / n)
// with tstride = n / (ns RAD) (k r tstride < n); n - r[0] entries in all.
__host__ __device__ __forceinline__ int stage_tab_len(int n, const N3Radix& rad) {
  return rad.count > 1 ? n - rad.r[0] : 0;
}
template <typename R>
__device__ void build_stage_tab(cplx<R>* tab, int n, const N3Radix& rad, const Twid<R>& tw,
                                int tid, int nt) {
  int ns = rad.r[0], off = 0;
  for (int st = 1; st < rad.count; ++st) {
    const int RAD = rad.r[st], rm = RAD - 1, cnt = ns * rm;
    const int tstride = n / (ns * RAD);
    for (int e = tid; e < cnt; e += nt) {
      const int r = e / ns + 1, k = e - (r - 1) * ns;
      tab[off + e] = tw(k * r * tstride);
    }
    off += cnt;
    ns *= RAD;
  }
}

template <typename R, int MAXR, bool FIRST, bool TAB, bool ONE>
__device__ __forceinline__ void fft_stage_radix(int R_, const cplx<R>* in, cplx<R>* out, int n,
                                                int nl, int ld, int ns, const N3Radix& rad, int st,
                                                const Twid<R>& tw, const cplx<R>* stab, int tid,
                                                int nt) {
#define STAGE(RR) fft_stage<R, RR, FIRST, TAB, ONE>(in, out, n, nl, ld, ns, tw, stab, tid, nt, \
                                               rad.nb_m[st], rad.nb_s[st], rad.ns_m[st], rad.ns_s[st])
  switch (R_) {
    case 2: STAGE(2); break;
    case 3: STAGE(3); break;
    case 4: STAGE(4); break;
    case 6:
      if constexpr (MAXR >= 6) STAGE(6);
      break;
    case 8:
      if constexpr (MAXR >= 8) STAGE(8);
      break;
    case 9:
      if constexpr (MAXR >= 9) STAGE(9);
      break;
    case 16:
      if constexpr (MAXR >= 16) STAGE(16);
      break;
    default: STAGE(5); break;
  }
#undef STAGE
}

// Stockham stages in LDS; returns the buffer holding the result.  MAXR: the largest radix
// compiled in (5: radices 2-5 only, which keeps the kernel's register and scalar-register
// footprint small; 16: also the composite radices 6, 8, 9, 16); the launchers pick it from
// the plan.
template <typename R, int MAXR, bool TAB, bool ONE>
__device__ cplx<R>* lds_fft(cplx<R>* a, cplx<R>* b, int n, int nl, int ld, const N3Radix& rad,
                            const Twid<R>& tw, const cplx<R>* stab, int tid, int nt) {
  int ns = 1;
  cplx<R>* in = a;
  cplx<R>* out = b;
  for (int st = 0; st < rad.count; ++st) {
    const int R_ = rad.r[st];
    if (st == 0) {
      fft_stage_radix<R, MAXR, true, false, ONE>(R_, in, out, n, nl, ld, ns, rad, st, tw, stab, tid, nt);
    } else {
      fft_stage_radix<R, MAXR, false, TAB, ONE>(R_, in, out, n, nl, ld, ns, rad, st, tw, stab, tid, nt);
      if (TAB) stab += ns * (R_ - 1);
    }
    __syncthreads();
    ns *= R_;
    cplx<R>* tmp = in;
    in = out;
    out = tmp;
  }
  return in;
}

// position of index a inside window [start, start + count) of an axis of length n
__device__ __forceinline__ bool in_window(int a, N3Window wd, int n) {
  int d = a - wd.start;
  d += d < 0 ? n : 0;
  return d < wd.count;
}

// Elements per thread of one FFT item: items hold at most 4096 elements (the launchers
// check), so 8 per thread of an FFT_NT = 512 workgroup.
constexpr int FFT_PF = 8;

// Contiguous axis (x): `nl` lines per workgroup (lines (level, z, y) of the windows).  The
// next group's inputs are fetched into registers while the current group is transformed.
// TAB: the stages' twiddle tables are built in LDS once per workgroup (build_stage_tab).
// ONE: one line per group (nl = 1): no line index per element, and the stores run over the
// output window only.
template <typename R, int MAXR, bool TAB, bool ONE>
__global__ __launch_bounds__(FFT_NT) void fft_lines_kernel(N3LineParams<R> p, int nl) {
  extern __shared__ __align__(16) unsigned char fsh[];
  __shared__ long long lbase[2][16];
  const int n = p.n;
  const int tid = threadIdx.x;
  cplx<R>* a = reinterpret_cast<cplx<R>*>(fsh);
  cplx<R>* b = a + (size_t)nl * n;
  const Twid<R> tw = load_twid<R>(p.tw, n, b + (size_t)nl * n, tid, FFT_NT);
  cplx<R>* stab = b + (size_t)nl * n + twid_len(n);
  if (TAB) {
    __syncthreads();  // the two-level table is in LDS
    build_stage_tab<R>(stab, n, p.rad, tw, tid, FFT_NT);
  }
  const long long n_lines = (long long)p.n_levels * p.zw.count * p.yw.count;
  const long long n_groups = (n_lines + nl - 1) / nl;
  auto set_bases = [&](long long grp, int buf) {
    const long long line0 = grp * nl;
    const int nlg = static_cast<int>(min<long long>(nl, n_lines - line0));
    if (tid < nlg) {
      const long long line = line0 + tid;
      const int yo = static_cast<int>(line % p.yw.count);
      const long long r = line / p.yw.count;
      const int zo = static_cast<int>(r % p.zw.count);
      const int lv = static_cast<int>(r / p.zw.count);
      int y = p.yw.start + yo, z = p.zw.start + zo;
      y -= y >= p.ny ? p.ny : 0;
      z -= z >= p.nz ? p.nz : 0;
      lbase[buf][tid] = (long long)lv * p.grid_stride + ((long long)z * p.ny + y) * n;
    }
  };
  auto fetch = [&](long long grp, int buf, cplx<R>* regs) {
    const int nlg = static_cast<int>(min<long long>(nl, n_lines - grp * nl));
    if (ONE) {
      const cplx<R>* g = p.grid + lbase[buf][0];
#pragma unroll
      for (int k = 0; k < FFT_PF; ++k) {
        const int i = tid + k * FFT_NT;
        if (i < n) regs[k] = in_window(i, p.in, n) ? g[i] : mk<R>(0, 0);
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < FFT_PF; ++k) {
      const int i = tid + k * FFT_NT;
      if (i < nlg * n) {
        const int li = fast_div(i, p.rad.n_m, p.rad.n_s), x = i - li * n;
        regs[k] = in_window(x, p.in, n) ? p.grid[lbase[buf][li] + x] : mk<R>(0, 0);
      }
    }
  };
  long long grp = blockIdx.x;
  if (grp >= n_groups) return;
  cplx<R> cur[FFT_PF], nxt[FFT_PF];
  int cb = 0;
  set_bases(grp, cb);
  __syncthreads();
  fetch(grp, cb, cur);
  for (; grp < n_groups; grp += gridDim.x) {
    const int nlg = static_cast<int>(min<long long>(nl, n_lines - grp * nl));
    const long long gn = grp + gridDim.x;
#pragma unroll
    for (int k = 0; k < FFT_PF; ++k) {
      const int i = tid + k * FFT_NT;
      if (i < nlg * n) a[i] = cur[k];
    }
    if (gn < n_groups) set_bases(gn, cb ^ 1);
    __syncthreads();
    if (gn < n_groups) fetch(gn, cb ^ 1, nxt);  // in flight during the transform
    cplx<R>* res = lds_fft<R, MAXR, TAB, ONE>(a, b, n, nlg, n, p.rad, tw, stab, tid, FFT_NT);
    if (ONE) {
      cplx<R>* g = p.grid + lbase[cb][0];
      for (int e = tid; e < p.out.count; e += FFT_NT) {
        int k = p.out.start + e;  // start < n, count <= n
        k -= k >= n ? n : 0;
        g[k] = res[k];
      }
    } else {
      for (int i = tid; i < nlg * n; i += FFT_NT) {
        const int li = fast_div(i, p.rad.n_m, p.rad.n_s), k = i - li * n;
        if (in_window(k, p.out, n)) p.grid[lbase[cb][li] + k] = res[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < FFT_PF; ++k) cur[k] = nxt[k];
    cb ^= 1;
  }
}

// Strided axis: transforms of length m for TW consecutive x positions at once; element i of
// sub-transform `sub` at axis index sub * sub_stride + i * estride.  The LDS line stride is
// odd so that the TW lines of a load fall into different banks.  (Latency is hidden by
// occupancy: a register prefetch of the next item costs more waves than it saves.)
template <typename R, int MAXR>
__global__ __launch_bounds__(FFT_NT) void fft_pass_kernel(N3PassParams<R> p, int tw_shift) {
  extern __shared__ __align__(16) unsigned char fsh[];
  const int TW = 1 << tw_shift;  // x positions per item (power of two)
  const int ld = p.m | 1;
  cplx<R>* a = reinterpret_cast<cplx<R>*>(fsh);
  cplx<R>* b = a + TW * ld;
  cplx<R>* tws = b + TW * ld;
  const Twid<R> tw = load_twid<R>(p.tw, p.m, tws, threadIdx.x, blockDim.x);
  // second table (two-pass twiddles) right after the first; unused when p.twiddle == 0
  cplx<R>* tws2 = tws + twid_len(p.m);
  if (p.twiddle) load_twid<R>(p.tw2, static_cast<int>(p.ntot), tws2, threadIdx.x, blockDim.x);
  const Twid<R> tw2{tws2, tws2 + 64};
  const int n_xt = (p.xw.count + TW - 1) >> tw_shift;
  // the launcher checks that the item count fits in 31 bits
  const int n_items = n_xt * p.n_sub * p.other.count * p.n_levels;
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int q1 = fast_div(item, p.xt_m, p.xt_s);
    const int xt = item - q1 * n_xt;
    const int q2 = fast_div(q1, p.sub_m, p.sub_s);
    const int sub = q1 - q2 * p.n_sub;
    const int lv = fast_div(q2, p.oc_m, p.oc_s);
    const int o = q2 - lv * p.other.count;
    int oo = p.other.start + o;
    oo -= oo >= p.no ? p.no : 0;
    if (p.operm_n2 > 1) {
      const int q = fast_div(oo, p.op_m, p.op_s);
      oo = (oo - q * p.operm_n1) * p.operm_n2 + q;
    }
    cplx<R>* base = p.grid + (size_t)lv * p.grid_stride + (size_t)oo * p.outer_stride;
    for (int t = threadIdx.x; t < (p.m << tw_shift); t += blockDim.x) {
      const int xi = t & (TW - 1), i = t >> tw_shift;
      const int j = (xt << tw_shift) + xi;
      cplx<R> v = mk<R>(0, 0);
      if (j < p.xw.count) {
        int x = p.xw.start + j;
        x -= x >= p.nx ? p.nx : 0;
        const int ai = static_cast<int>(sub * p.sub_stride + i * p.estride);
        if (!p.in_check || in_window(ai, p.in, p.nax))
          v = base[(long long)ai * p.axis_stride + x];
      }
      a[xi * ld + i] = v;
    }
    __syncthreads();
    cplx<R>* res = lds_fft<R, MAXR, false, false>(a, b, p.m, TW, ld, p.rad, tw, nullptr, threadIdx.x,
                                           blockDim.x);
    for (int t = threadIdx.x; t < (p.m << tw_shift); t += blockDim.x) {
      const int xi = t & (TW - 1), k = t >> tw_shift;
      const int j = (xt << tw_shift) + xi;
      if (j >= p.xw.count) continue;
      if (p.out_check && !in_window(sub * p.fa + k * p.fb, p.out, p.nax)) continue;
      int x = p.xw.start + j;
      x -= x >= p.nx ? p.nx : 0;
      cplx<R> v = res[xi * ld + k];
      if (p.twiddle) v = v * tw2(sub * k);  // sub < n2, k < n1: sub k < ntot
      const int ai = static_cast<int>(sub * p.sub_stride + k * p.estride);
      base[(long long)ai * p.axis_stride + x] = v;
    }
    __syncthreads();
  }
}

// Strided axis, m = M1 M2 with both factors radices of dft_small: each transform in two
// register stages with one LDS exchange (X[k1 + M1 k2] = sum_c2 w_M2^(c2 k2) w_m^(c2 k1)
// sum_j1 x[c2 + M2 j1] w_M1^(j1 k1)).  Stage 1: thread (x position, c2) loads x[c2 + M2 j1],
// j1 < M1, straight from global memory, transforms them, applies w_m^(c2 k1) and stores row
// k1 M2 + c2 of its line in LDS; stage 2: thread (x position, k1) reads the M2 values of row
// k1, transforms them and stores outputs k1 + M1 k2.  Lanes run over consecutive x
// positions, so global accesses are contiguous and the odd LDS line stride spreads a
// wavefront's accesses over the banks.  Same items, windows, pass twiddle and output
// permutation as fft_pass_kernel.
template <typename R, int M1, int M2>
__global__ __launch_bounds__(FFT_NT) void fft_pass_rr_kernel(N3PassParams<R> p, int tw_shift) {
  extern __shared__ __align__(16) unsigned char fsh[];
  constexpr int M = M1 * M2;
  constexpr int LD = M | 1;
  const int TW = 1 << tw_shift;
  cplx<R>* a = reinterpret_cast<cplx<R>*>(fsh);  // [TW][LD]
  cplx<R>* twm = a + TW * LD;                     // exp(+2 pi i t / M), t < M
  cplx<R>* tws2 = twm + M;                        // two-level table of ntot (pass twiddle)
  const int tid = threadIdx.x;
  for (int t = tid; t < M; t += FFT_NT) twm[t] = p.tw[t & 63] * p.tw[64 + (t >> 6)];
  if (p.twiddle) load_twid<R>(p.tw2, static_cast<int>(p.ntot), tws2, tid, FFT_NT);
  const Twid<R> tw2{tws2, tws2 + 64};
  __syncthreads();
  const int n_xt = (p.xw.count + TW - 1) >> tw_shift;
  const int n_items = n_xt * p.n_sub * p.other.count * p.n_levels;
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int q1 = fast_div(item, p.xt_m, p.xt_s);
    const int xt = item - q1 * n_xt;
    const int q2 = fast_div(q1, p.sub_m, p.sub_s);
    const int sub = q1 - q2 * p.n_sub;
    const int lv = fast_div(q2, p.oc_m, p.oc_s);
    const int o = q2 - lv * p.other.count;
    int oo = p.other.start + o;
    oo -= oo >= p.no ? p.no : 0;
    if (p.operm_n2 > 1) {
      const int q = fast_div(oo, p.op_m, p.op_s);
      oo = (oo - q * p.operm_n1) * p.operm_n2 + q;
    }
    cplx<R>* base = p.grid + (size_t)lv * p.grid_stride + (size_t)oo * p.outer_stride;
    const long long sub_off = (long long)sub * p.sub_stride;
    for (int u = tid; u < (M2 << tw_shift); u += FFT_NT) {
      const int xi = u & (TW - 1), c2 = u >> tw_shift;
      const int j = (xt << tw_shift) + xi;
      cplx<R> v[M1];
      if (j < p.xw.count) {
        int x = p.xw.start + j;
        x -= x >= p.nx ? p.nx : 0;
#pragma unroll
        for (int j1 = 0; j1 < M1; ++j1) {
          const int ai = static_cast<int>(sub_off + (long long)(c2 + M2 * j1) * p.estride);
          v[j1] = (!p.in_check || in_window(ai, p.in, p.nax))
                      ? base[(long long)ai * p.axis_stride + x]
                      : mk<R>(0, 0);
        }
      } else {
#pragma unroll
        for (int j1 = 0; j1 < M1; ++j1) v[j1] = mk<R>(0, 0);
      }
      dft_small<R, M1>(v);
      cplx<R>* row = a + xi * LD + c2;
      row[0] = v[0];
#pragma unroll
      for (int k1 = 1; k1 < M1; ++k1) row[k1 * M2] = c2 == 0 ? v[k1] : v[k1] * twm[c2 * k1];
    }
    __syncthreads();
    for (int u = tid; u < (M1 << tw_shift); u += FFT_NT) {
      const int xi = u & (TW - 1), k1 = u >> tw_shift;
      const int j = (xt << tw_shift) + xi;
      if (j >= p.xw.count) continue;
      int x = p.xw.start + j;
      x -= x >= p.nx ? p.nx : 0;
      cplx<R> v[M2];
      const cplx<R>* row = a + xi * LD + k1 * M2;
#pragma unroll
      for (int c2 = 0; c2 < M2; ++c2) v[c2] = row[c2];
      dft_small<R, M2>(v);
#pragma unroll
      for (int k2 = 0; k2 < M2; ++k2) {
        const int k = k1 + M1 * k2;
        if (p.out_check && !in_window(sub * p.fa + k * p.fb, p.out, p.nax)) continue;
        cplx<R> w = v[k2];
        if (p.twiddle) w = w * tw2(sub * k);  // sub < n2, k < n1: sub k < ntot
        const int ai = static_cast<int>(sub_off + (long long)k * p.estride);
        base[(long long)ai * p.axis_stride + x] = w;
      }
    }
    __syncthreads();
  }
}

// Strided axis of n = n1 n2 points in one pass (the two passes' transforms, windows and output
// order): 2^tw_shift x positions per workgroup, their lines in LDS between up to four stages of
// radix r[s] in place, X[K], K = f0 + r0 (f1 + r1 (f2 + ...)), at f0 S0 + f1 S1 + ... with
// S_s = n / (r0 ... r_s).  The first stage loads from global memory, inside the input window,
// and the last one stores the frequencies of the output window, so the unpruned middle of the
// two passes, twice the windows' size each way, stays in the CU.
// Workgroup i of a round runs on XCD i mod 8 and the tiles of a round are dealt to the XCDs in
// runs: neighbouring tiles share 128-byte lines (a tile of 4 positions has 32 bytes of each).
// Bound by LDS exchanges and the transforms' arithmetic between barriers, behind them HBM.  500
// samples of 256 antennas, y axis of 3456 points, 4 levels: 3.7 ms and 7.9 GB (4.3 ms with 512
// threads) against 3.9 + 3.0 ms and 23 GB in two passes.
// NAT: contiguous axis (x lines, a position is a line): consecutive lanes take consecutive
// elements of one line, and the frequencies are stored in their own order.
template <typename R, int NT, int RAD, bool FIRST, bool LAST, bool NAT>
__device__ __forceinline__ void axis_stage(const N3AxisParams<R>& p, int s, cplx<R>* lds, const Twid<R>& tw,
                                           cplx<R>* base, int xt, int tid) {
  const int tws = p.tw_shift, TW = 1 << tws, per = p.n / RAD;
  const int S = p.span[s], items = per << tws;
  for (int u = tid; u < items; u += NT) {
    const int xi = NAT ? fast_div(u, p.per_m[s], p.per_s[s]) : u & (TW - 1);
    const int t = NAT ? u - xi * per : u >> tws;
    int K = 0, rest = t, at = 0;  // LAST: frequency of output 0 and the position it comes from
    if constexpr (LAST && NAT) {
      K = t;
      for (int q = 0; q < s; ++q) {
        const int f = fast_div(rest, p.rd_m[q], p.rd_s[q]);
        at += (rest - f * p.r[q]) * p.span[q];
        rest = f;
      }
    }
    const int hi = LAST ? t : FIRST ? 0 : fast_div(t, p.sp_m[s], p.sp_s[s]);
    const int lo = LAST ? 0 : t - hi * S;
    cplx<R>* line = lds + xi * p.ld + (LAST && NAT ? at : hi * (RAD * S) + lo);
    const int j = (xt << tws) + xi;
    int xp = p.xw.start + j;
    xp -= xp >= p.nx ? p.nx : 0;
    const long long x = NAT ? (long long)xp * p.n : xp;
    cplx<R> v[RAD];
    if constexpr (FIRST) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const int ai = lo + r * S;
        v[r] = j < p.xw.count && in_window(ai, p.in, p.n) ? base[(long long)ai * p.axis_stride + x]
                                                          : mk<R>(0, 0);
      }
    } else {
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[r] = line[r * S];
    }
    dft_small<R, RAD>(v);
    if constexpr (LAST) {
      if (j >= p.xw.count) continue;
      if constexpr (NAT) {
#pragma unroll
        for (int r = 0; r < RAD; ++r)
          if (in_window(K + r * p.weight[s], p.out, p.n)) base[x + K + r * p.weight[s]] = v[r];
        continue;
      }
      // digits of the position hi RAD
      rest = hi * RAD;
      for (int q = 0; q < s; ++q) {
        const int f = fast_div(rest, p.sp_m[q], p.sp_s[q]);
        rest -= f * p.span[q];
        K += f * p.weight[q];
      }
      const int q0 = fast_div(K, p.n1_m, p.n1_s), row = (K - q0 * p.n1) * p.n2 + q0;
#pragma unroll
      for (int r = 0; r < RAD; ++r)
        if (in_window(K + r * p.weight[s], p.out, p.n))
          base[(long long)(row + r * p.last_step) * p.axis_stride + x] = v[r];
    } else {
      const int t1 = lo * p.weight[s];  // w_(RAD S)^lo = w_n^t1
      cplx<R> wp[RAD];
      wp[1] = tw(t1);
      if constexpr (RAD > 2) wp[2] = wp[1] * wp[1];
      if constexpr (RAD > 3) wp[3] = wp[2] * wp[1];
      if constexpr (RAD > 4) {
        wp[4] = tw(4 * t1);
#pragma unroll
        for (int r = 5; r < RAD && r < 8; ++r) wp[r] = wp[4] * wp[r - 4];
      }
      if constexpr (RAD > 8) {
        wp[8] = tw(8 * t1);
#pragma unroll
        for (int r = 9; r < RAD; ++r) wp[r] = wp[8] * wp[r - 8];
      }
      line[0] = v[0];
#pragma unroll
      for (int r = 1; r < RAD; ++r) line[r * S] = v[r] * wp[r];
    }
  }
}

template <typename R, int NT, bool FIRST, bool LAST, bool NAT>
__device__ __forceinline__ void axis_radix(const N3AxisParams<R>& p, int s, cplx<R>* lds, const Twid<R>& tw,
                                           cplx<R>* base, int xt, int tid) {
  switch (p.r[s]) {
    case 2: axis_stage<R, NT, 2, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 3: axis_stage<R, NT, 3, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 4: axis_stage<R, NT, 4, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 5: axis_stage<R, NT, 5, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 6: axis_stage<R, NT, 6, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 8: axis_stage<R, NT, 8, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 9: axis_stage<R, NT, 9, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 10: axis_stage<R, NT, 10, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 12: axis_stage<R, NT, 12, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    case 15: axis_stage<R, NT, 15, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
    default: axis_stage<R, NT, 16, FIRST, LAST, NAT>(p, s, lds, tw, base, xt, tid); break;
  }
}

template <typename R, int NT, bool NAT>
__global__ __launch_bounds__(NT) void fft_axis_kernel(N3AxisParams<R> p) {
  extern __shared__ __align__(16) unsigned char fsh[];
  cplx<R>* lds = reinterpret_cast<cplx<R>*>(fsh);
  const int tid = threadIdx.x;
  const Twid<R> tw = load_twid<R>(p.tw, p.n, lds + ((size_t)p.ld << p.tw_shift), tid, NT);
  __syncthreads();
  const int n_xt = (p.xw.count + (1 << p.tw_shift) - 1) >> p.tw_shift;
  const int n_items = n_xt * p.other.count * p.n_levels;
  const int at = gridDim.x % 8 == 0 ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  for (int item = at; item < n_items; item += gridDim.x) {
    const int q1 = fast_div(item, p.xt_m, p.xt_s);
    const int xt = item - q1 * n_xt;
    const int lv = fast_div(q1, p.oc_m, p.oc_s);
    int oo = p.other.start + q1 - lv * p.other.count;
    oo -= oo >= p.no ? p.no : 0;
    if (p.operm_n2 > 1) {
      const int q = fast_div(oo, p.op_m, p.op_s);
      oo = (oo - q * p.operm_n1) * p.operm_n2 + q;
    }
    cplx<R>* base = p.grid + (size_t)lv * p.grid_stride + (size_t)oo * p.outer_stride;
    axis_radix<R, NT, true, false, NAT>(p, 0, lds, tw, base, xt, tid);
    for (int s = 1; s < p.stages - 1; ++s) {
      __syncthreads();
      axis_radix<R, NT, false, false, NAT>(p, s, lds, tw, base, xt, tid);
    }
    __syncthreads();
    axis_radix<R, NT, false, true, NAT>(p, p.stages - 1, lds, tw, base, xt, tid);
    __syncthreads();  // lines read before the next tile's first stage
  }
}

// --------------------------------------------------------------------------------------
// Interpolation at the pixels, correction, real part accumulated into the images.
// --------------------------------------------------------------------------------------
// The kernel width is a template argument so that the per-axis weights and indices stay in
// registers (a run-time width puts them in scratch memory, read in the innermost loop).
template <typename R, typename TI, int W>
__global__ __launch_bounds__(256) void n3_interp_kernel(N3InterpParams<R> p) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= p.n_pix) return;
  constexpr int w = W;
  R wx[W], wy[W], wz[W];
  int kx[W], ky[W], kz[W];
  double corr = 1.0, cphase = 0.0;
  const double xq[3] = {p.lmn[q], p.lmn[p.n_pix + q], p.lmn[2 * (size_t)p.n_pix + q]};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double s = p.gam[d] * (xq[d] - p.D[d]);
    const double a2 = p.h1[d] * s / p.h2[d];
    const int k0 = static_cast<int>(ceil(a2 - 0.5 * w));
    R* wd = d == 0 ? wx : (d == 1 ? wy : wz);
    int* kd = d == 0 ? kx : (d == 1 ? ky : kz);
    // frequency k = (k0 + o) mod nf2 and, for two-pass axes (stored at (k mod n1) n2 +
    // k / n1), its digits (k mod n1, k / n1): one division each for o = 0, then stepped
    // with the wrap-around at nf2 = n1 n2
    const int nf = p.nf2[d], n1 = p.n1[d], n2 = p.n2[d];
    int k = k0 % nf;
    if (k < 0) k += nf;
    int kq = k / n1, kr = k - kq * n1;
#pragma unroll
    for (int o = 0; o < w; ++o) {
      wd[o] = es_kernel<R>(static_cast<R>((k0 + o - a2) * 2.0 / w), R(p.beta2));
      kd[o] = n2 > 1 ? kr * n2 + kq : k;
      ++k;
      ++kr;
      if (kr == n1) {
        kr = 0;
        ++kq;
      }
      if (k == nf) k = kr = kq = 0;
    }
    const double alpha1 = 0.5 * p.w1 * p.h1[d];
    corr *= p.h1[d] * p.h2[d] / (alpha1 * ft_lookup(p.ft, p.n_ft, p.ft_inv_delta, s * alpha1));
    cphase += p.C[d] * xq[d];
  }
  const double turns = cphase * 0.15915494309189535;
  double cs, cc;
  sincospi(2.0 * (turns - rint(turns)), &cs, &cc);
  for (int lv = 0; lv < p.n_levels; ++lv) {
    const cplx<R>* g = p.grid + (size_t)lv * p.grid_stride;
    R sr = 0, si = 0;
#pragma unroll 1
    for (int oz = 0; oz < w; ++oz) {
#pragma unroll 1
      for (int oy = 0; oy < w; ++oy) {
        const cplx<R>* row = g + ((size_t)kz[oz] * p.nf2[1] + ky[oy]) * p.nf2[0];
        const R wyz = wy[oy] * wz[oz];
        R rr = 0, ri = 0;
#pragma unroll
        for (int ox = 0; ox < w; ++ox) {
          const cplx<R> v = row[kx[ox]];
          rr += wx[ox] * v.re;
          ri += wx[ox] * v.im;
        }
        sr += wyz * rr;
        si += wyz * ri;
      }
    }
    // Re( exp(i C.x) * corr * (sr + i si) )
    const double re = corr * (cc * static_cast<double>(sr) - cs * static_cast<double>(si));
    TI* img = static_cast<TI*>(p.img) + (size_t)lv * p.img_ld;
    img[q] += static_cast<TI>(re * p.scale);
  }
}

template <typename R>
__global__ void zero_kernel(R* p, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    p[i] = R(0);
}

// Per-sample min/max of the positions of the rows used (positions / wavelength).
__global__ void pos_range_kernel(const double* pos, long long pos_stride, int apad,
                                 const int* n_rows, int n_rows_const, double* out) {
  const int s = blockIdx.x;
  const int n = n_rows ? n_rows[s] : n_rows_const;
  __shared__ double mn[3][256], mx[3][256];
  for (int d = 0; d < 3; ++d) {
    double lo = 1e300, hi = -1e300;
    for (int a = threadIdx.x; a < n; a += blockDim.x) {
      const double v = pos[(size_t)s * pos_stride + d * apad + a];
      lo = fmin(lo, v);
      hi = fmax(hi, v);
    }
    mn[d][threadIdx.x] = lo;
    mx[d][threadIdx.x] = hi;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int d = threadIdx.x;
    double lo = 1e300, hi = -1e300;
    for (int i = 0; i < (int)blockDim.x; ++i) {
      lo = fmin(lo, mn[d][i]);
      hi = fmax(hi, mx[d][i]);
    }
    out[s * 6 + d] = lo;
    out[s * 6 + 3 + d] = hi;
  }
}

// --------------------------------------------------------------------------------------
// Direct sum: img_l(x_q) += Re sum_j v_lj exp(i u_j . x_q)  (src/host/kernels/nuft_sum.cpp:9-31)
// over the points of a source (a pair whose mirror is its conjugate stands for both), one
// phase for all levels of the launch.  A thread owns a pixel; 256 slots at a time are turned
// into points, compacted into LDS and read by all threads of the workgroup.  float64 phase
// reduced to one turn; R = float: float32 cos/sin, sums of at most 256 points added to the
// running float32 sum.
// Bound: vector ALU, one cos/sin pair (35 instructions with its phase) and two
// multiply-adds per level for each point and pixel.  Where the pixels give too few workgroups
// the slots are split as well (direct_chunks); the parts are summed in a fixed order.
// 8 samples of 55 antennas, 128^2 pixels, 2 images: 0.19 ms against 16 launches of 0.33 ms (one
// sample and image each, every entry of the antisymmetric uvw, 64 workgroups).
// --------------------------------------------------------------------------------------
template <typename R, int LG>
__global__ __launch_bounds__(256) void direct_sum_kernel(N3DirectParams<R> p) {
  __shared__ double su[3][256];
  __shared__ cplx<R> sv[256][LG];
  __shared__ int cnt[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = blockIdx.x * 256 + tid;
  const bool live = q < p.n_pix;
  // direction cosines in turns per unit u
  constexpr double INV_2PI = 0.15915494309189533577;
  const double x = live ? p.lmn[q] * INV_2PI : 0.0;
  const double y = live ? p.lmn[p.n_pix + q] * INV_2PI : 0.0;
  const double z = live ? p.lmn[2 * (size_t)p.n_pix + q] * INV_2PI : 0.0;
  const long long sps = p.src.slots_per_sample();
  const long long per = ((p.n_slots + p.chunks - 1) / p.chunks + 255) / 256 * 256;
  const long long b0 = blockIdx.y * per, b1 = min(p.n_slots, b0 + per);
  R acc[LG];
#pragma unroll
  for (int l = 0; l < LG; ++l) acc[l] = R(0);
  for (long long base = b0; base < b1; base += 256) {
    const long long slot = base + tid;
    SlotPoint sp;
    bool hit = false;
    int s = 0;
    if (slot < b1) {
      s = static_cast<int>(slot / sps);
      hit = slot_point(p.src, s, slot - (long long)s * sps, sp);
    }
    const unsigned long long mask = __ballot(hit);
    if (lane == 0) cnt[wave] = __popcll(mask);
    __syncthreads();  // the previous points are no longer read
    int k = __popcll(mask & ((1ull << lane) - 1ull)), m = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      k += w < wave ? cnt[w] : 0;
      m += cnt[w];
    }
    if (hit) {
#pragma unroll
      for (int d = 0; d < 3; ++d) su[d][k] = sp.u[d];
      const cplx<R>* v = p.vv + ((size_t)s * p.n_levels_total + p.lv0) * p.vv_stride + sp.src;
      const R mr = R(sp.mult), mi = sp.conj ? -mr : mr;
#pragma unroll
      for (int l = 0; l < LG; ++l) {
        cplx<R> c = mk<R>(0, 0);
        if (l < p.n_levels) c = v[(size_t)l * p.vv_stride];
        sv[k][l] = mk<R>(c.re * mr, c.im * mi);
      }
    }
    __syncthreads();
    R sum[LG];
#pragma unroll
    for (int l = 0; l < LG; ++l) sum[l] = R(0);
#pragma unroll 2
    for (int j = 0; j < m; ++j) {
      const double t = fma(x, su[0][j], fma(y, su[1][j], z * su[2][j]));
      R c, sn;
      if constexpr (sizeof(R) == 8)
        sincospi(2.0 * (t - rint(t)), &sn, &c);
      else
        cossin_turn(static_cast<float>(t - rint(t)), c, sn);
#pragma unroll
      for (int l = 0; l < LG; ++l) sum[l] += sv[j][l].re * c - sv[j][l].im * sn;
    }
#pragma unroll
    for (int l = 0; l < LG; ++l) acc[l] += sum[l];
  }
  if (!live) return;
#pragma unroll
  for (int l = 0; l < LG; ++l) {
    if (l >= p.n_levels) break;
    if (p.chunks > 1)
      p.part[((size_t)blockIdx.y * p.n_levels + l) * p.n_pix + q] = acc[l];
    else
      p.img[(size_t)(p.lv0 + l) * p.n_pix + q] += acc[l];
  }
}

template <typename R>
__global__ __launch_bounds__(256) void direct_reduce_kernel(N3DirectParams<R> p) {
  const int q = blockIdx.x * 256 + threadIdx.x, l = blockIdx.y;
  if (q >= p.n_pix) return;
  R s = R(0);
  for (int k = 0; k < p.chunks; ++k) s += p.part[((size_t)k * p.n_levels + l) * p.n_pix + q];
  p.img[(size_t)(p.lv0 + l) * p.n_pix + q] += s;
}

// VV_l = Z diag(w_l) Z^H for every (sample, level); Z rows = antennas used (ld ldz).  The
// vector-ALU form, used for float32 eigenvectors (float64 ones take vv_levels_mfma_kernel).
template <typename R, typename TO>
__global__ __launch_bounds__(256) void vv_levels_kernel(N3VVParams<R> p) {
  // 64 x 64 output tile per workgroup (tiles on or below the diagonal), eigenvectors taken
  // VK at a time through LDS; thread (tx, ty) accumulates rows i0 + tx + 16 u and columns
  // j0 + ty + 16 v (u, v < 4), so LDS reads are consecutive over tx and broadcast over ty
  constexpr int VT = 64, VK = 16;
  __shared__ cplx<R> ti[VK][VT + 1];  // Z[i0 + r, e] d_e
  __shared__ cplx<R> tj[VK][VT + 1];  // Z[j0 + c, e]
  const int sl = blockIdx.z;
  const int s = sl / p.n_levels, lv = sl % p.n_levels;
  const int n = p.n_rows ? p.n_rows[s] : p.n_rows_const;
  const int i0 = blockIdx.x * VT, j0 = blockIdx.y * VT;
  if (i0 >= n || j0 > i0) return;  // only tiles touching the lower triangle
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const cplx<R>* Z = p.z + (size_t)s * p.stride_z;
  const R* dw = p.wd + ((size_t)s * p.n_levels + lv) * p.n_cols;
  cplx<R> acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = mk<R>(0, 0);
  for (int e0 = 0; e0 < p.n_cols; e0 += VK) {
    // eigenvectors outside the level carry weight 0: skip chunks without any (uniform)
    const int ew = e0 + (tid & (VK - 1));
    const R dt = ew < p.n_cols ? dw[ew] : R(0);
    if (!__syncthreads_or(dt != R(0))) continue;
#pragma unroll
    for (int q = 0; q < VK * VT / 256; ++q) {
      const int idx = tid + 256 * q;
      const int k = idx / VT, r = idx % VT, e = e0 + k;
      const bool ok = e < p.n_cols;
      const R de = ok ? dw[e] : R(0);
      ti[k][r] = (ok && i0 + r < n) ? Z[(i0 + r) + (size_t)e * p.ldz] * de : mk<R>(0, 0);
      tj[k][r] = (ok && j0 + r < n) ? Z[(j0 + r) + (size_t)e * p.ldz] : mk<R>(0, 0);
    }
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < VK; ++k) {
      cplx<R> a[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] = ti[k][tx + 16 * u];
#pragma unroll
      for (int v = 0; v < 4; ++v) b[v] = tj[k][ty + 16 * v];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] = acc[u][v] + mulc(a[u], b[v]);
    }
    __syncthreads();
  }
  cplx<TO>* out = reinterpret_cast<cplx<TO>*>(p.vv) + (size_t)sl * p.vv_stride;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = i0 + tx + 16 * u, j = j0 + ty + 16 * v;
      if (i < n && j < n && i >= j) out[i + (size_t)p.ld_vv * j] = cvt<TO>(acc[u][v]);
    }
}

// vv_levels_kernel in float64 on v_mfma_f64_16x16x4f64 with the operands loaded straight from
// global memory (no LDS, no barriers).  Workgroup = (sample, level, 64 x 64 tile on or below
// the diagonal); wavefront = 32 x 32 quadrant as 2 x 2 blocks of 16 x 16.  The products form
// D[j][i] = sum_e conj(Z[j, e]) (w_e Z[i, e]) = VV[i][j] (A operand: lane l holds row j =
// l % 16, eigenvector l / 16; B operand: eigenvector l / 16, row i = l % 16; result register r:
// j = l / 16 + 4 r, i = l % 16), so one store writes 16 consecutive rows i of a column j.  Only
// the eigenvectors from the level's first to its last nonzero weight are visited, four per
// step, with the next step's operands loaded before the current step's products.  Workgroups
// are numbered so that the tiles and levels of one sample run on one XCD (workgroup x runs on
// XCD x mod 8), which keeps the sample's Z in that XCD's L2.  Held to 128 registers (four
// wavefronts per SIMD; the 2 x 2 blocks' sums stay in vector registers, no spills).
template <typename TO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void
vv_levels_mfma_kernel(N3VVParams<double> p, int n_tiles, int per_xcd, int n_units) {
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  const int unit = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (unit >= n_units) return;
  const int t = unit % n_tiles, sl = unit / n_tiles;
  const int s = sl / p.n_levels, lv = sl % p.n_levels;
  int ti = 0;
  while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
  const int tj = t - ti * (ti + 1) / 2;
  const int n = p.n_rows ? p.n_rows[s] : p.n_rows_const;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ib = 64 * ti + 32 * (wave & 1), jb = 64 * tj + 32 * (wave >> 1);
  // quadrant outside the matrix or strictly above the diagonal (every i < every j)
  if (ib >= n || jb >= n || jb > ib + 31) return;
  const double* dw = p.wd + ((size_t)s * p.n_levels + lv) * p.n_cols;
  int lo = p.n_cols, hi = -1;
  for (int e = lane; e < p.n_cols; e += 64)
    if (dw[e] != 0.0) {
      lo = e < lo ? e : lo;
      hi = e;
    }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const int ol = __shfl_xor(lo, m), oh = __shfl_xor(hi, m);
    lo = ol < lo ? ol : lo;
    hi = oh > hi ? oh : hi;
  }
  const cplx<double>* Z = p.z + (size_t)s * p.stride_z;
  const int lr = lane & 15, lk = lane >> 4;
  const int jr[2] = {jb + lr, jb + 16 + lr}, ir[2] = {ib + lr, ib + 16 + lr};
  f64x4 dr[2][2], di[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      dr[a][b] = f64x4{0, 0, 0, 0};
      di[a][b] = f64x4{0, 0, 0, 0};
    }
  // P = Z[j, e] (rows j of the two column blocks), Q = w_e Z[i, e] (rows i of the two row
  // blocks) for the eigenvector e = k + l / 16 of this lane; zero outside [lo, hi] and n.
  auto load = [&](int k, cplx<double>* P, cplx<double>* Q) {
    const int e = k + lk;
    const bool ok = e <= hi;
    const double w = ok ? dw[e] : 0.0;
    const cplx<double>* col = Z + (size_t)(ok ? e : 0) * p.ldz;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      P[b] = (ok && jr[b] < n) ? col[jr[b]] : mk<double>(0, 0);
      const cplx<double> z = (ok && ir[b] < n) ? col[ir[b]] : mk<double>(0, 0);
      Q[b] = mk<double>(z.re * w, z.im * w);
    }
  };
  if (lo <= hi) {
    cplx<double> P[2], Q[2];
    load(lo & ~3, P, Q);
    for (int k = lo & ~3; k <= hi; k += 4) {
      cplx<double> Pn[2], Qn[2];
      load(k + 4, Pn, Qn);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          // re: Pr Qr + Pi Qi; im: Pr Qi - Pi Qr
          dr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].re, Q[b].re, dr[a][b], 0, 0, 0);
          dr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].im, Q[b].im, dr[a][b], 0, 0, 0);
          di[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].re, Q[b].im, di[a][b], 0, 0, 0);
          di[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-P[a].im, Q[b].re, di[a][b], 0, 0, 0);
        }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        P[b] = Pn[b];
        Q[b] = Qn[b];
      }
    }
  }
  cplx<TO>* out = reinterpret_cast<cplx<TO>*>(p.vv) + (size_t)sl * p.vv_stride;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = jb + 16 * a + lk + 4 * r, i = ib + 16 * b + lr;
        if (i < n && j < n && i >= j)
          out[i + (size_t)p.ld_vv * j] = mk<TO>(static_cast<TO>(dr[a][b][r]), static_cast<TO>(di[a][b][r]));
      }
}

// Trace of VV_l for every (sample, level) into the unused upper-triangle slot (0, 1).
template <typename TO>
__global__ __launch_bounds__(256) void vv_trace_kernel(int n_levels, const int* n_rows,
                                                       int n_rows_const, cplx<TO>* vv,
                                                       long long vv_stride, long long ld_vv) {
  __shared__ double red[4];
  const int sl = blockIdx.x;
  const int s = sl / n_levels;
  const int n = n_rows ? n_rows[s] : n_rows_const;
  cplx<TO>* m = vv + (size_t)sl * vv_stride;
  double re = 0, im = 0;
  for (int a = threadIdx.x; a < n; a += 256) {
    const cplx<TO> c = m[a + ld_vv * a];
    re += static_cast<double>(c.re);
    im += static_cast<double>(c.im);
  }
  re = block_sum<256>(re, red);
  im = block_sum<256>(im, red);
  if (threadIdx.x == 0) m[ld_vv] = mk<TO>(static_cast<TO>(re), static_cast<TO>(im));
}

}  // namespace

// --------------------------------------------------------------------------------------
// launchers
// --------------------------------------------------------------------------------------
void launch_pos_range(int n_samples, const double* pos, long long pos_stride, int apad,
                      const int* n_rows, int n_rows_const, double* out, hipStream_t st) {
  if (n_samples <= 0) return;
  pos_range_kernel<<<n_samples, 256, 0, st>>>(pos, pos_stride, apad, n_rows, n_rows_const, out);
  check_launch("pos_range_kernel");
}

template <typename R>
void launch_zero(R* p, long long n, hipStream_t st) {
  if (n <= 0) return;
  const long long blocks = std::min<long long>((n + 255) / 256, 1 << 16);
  zero_kernel<R><<<static_cast<unsigned>(blocks), 256, 0, st>>>(p, n);
  check_launch("zero_kernel");
}
template void launch_zero<float>(float*, long long, hipStream_t);
template void launch_zero<double>(double*, long long, hipStream_t);
template void launch_zero<unsigned>(unsigned*, long long, hipStream_t);

void launch_n3_points(const N3PointsParams& p, int n_samples, hipStream_t st) {
  if (n_samples <= 0 || p.n_list <= 0) return;
  if (!p.slot_list && p.n_list != p.src.slots_per_sample() * n_samples)
    fail(BIPP_INTERNAL_ERROR, "NUFFT point slots do not match the batch");
  n3_points_kernel<<<static_cast<unsigned>((p.n_list + 255) / 256), 256, 0, st>>>(p);
  check_launch("n3_points_kernel");
}

void launch_uvw_antisym(const N3Source& src, int n_samples, unsigned char* out, hipStream_t st) {
  if (n_samples <= 0) return;
  uvw_antisym_kernel<<<n_samples, 256, 0, st>>>(src, out);
  check_launch("uvw_antisym_kernel");
}

// Workgroups per item: about 2048 workgroups over all items (8 per CU), at least 1024 slots
// each, at most the 64 partial ranges that one wavefront reduces.
int slot_range_parts(int n_items, long long n_slots) {
  if (n_items <= 0) return 1;
  const long long by_grid = (2048 + n_items - 1) / n_items, by_work = n_slots / n_items / 1024;
  return static_cast<int>(std::max<long long>(1, std::min<long long>(64, std::min(by_grid, by_work))));
}

void launch_slot_range(const N3Source& src, int n_items, const unsigned long long* list,
                       const unsigned* begin, const unsigned* count, int parts, double* part,
                       double* out, hipStream_t st) {
  if (n_items <= 0) return;
  if (parts < 1 || parts > 64) fail(BIPP_INTERNAL_ERROR, "slot range parts");
  slot_range_kernel<<<dim3(n_items, parts), 256, 0, st>>>(src, list, begin, count,
                                                          parts > 1 ? part : out);
  check_launch("slot_range_kernel");
  if (parts == 1) return;
  slot_range_reduce_kernel<<<n_items, 64, 0, st>>>(part, parts, out);
  check_launch("slot_range_reduce_kernel");
}

void launch_n3_partition(const N3PartParams& p, hipStream_t st) {
  const long long n = p.src.slots_per_sample() * p.n_samples;
  if (n <= 0) return;
  const long long per = 256LL * PART_PER;
  n3_partition_kernel<<<static_cast<unsigned>((n + per - 1) / per), 256, 0, st>>>(
      p, p.dims[0] * p.dims[1] * p.dims[2]);
  check_launch("n3_partition_kernel");
}

void launch_n3_group_scatter(long long n_slots, int n_groups, const int* group_of,
                             const unsigned* group_start, unsigned* group_fill,
                             unsigned long long* list, hipStream_t st) {
  if (n_slots <= 0) return;
  const long long per = 256LL * PART_PER;
  n3_group_scatter_kernel<<<static_cast<unsigned>((n_slots + per - 1) / per), 256, 0, st>>>(
      n_slots, n_groups, group_of, group_start, group_fill, list);
  check_launch("n3_group_scatter_kernel");
}

void launch_scan(const unsigned* in, unsigned* out, unsigned* tmp, int n, hipStream_t st) {
  if (n <= 0) return;
  const int nb = (n + 1023) / 1024;
  if (nb > 1024 * 1024) fail(BIPP_INVALID_PARAMETER_ERROR, "too many NUFFT bins");
  unsigned* sums = tmp;
  unsigned* offs = tmp + nb;
  scan_block_kernel<<<nb, 1024, 0, st>>>(in, out, sums, n);
  check_launch("scan_block_kernel");
  if (nb > 1) {
    unsigned* sums2 = offs + nb;
    launch_scan(sums, offs, sums2, nb, st);
    scan_add_kernel<<<nb, 1024, 0, st>>>(out, offs, n);
    check_launch("scan_add_kernel");
  }
}


namespace {
template <typename R, int LG>
void spread_blocks(const N3SpreadParams<R>& p, unsigned blocks, unsigned grid, hipStream_t st) {
  if constexpr (LG > SpreadMfma<R>::levels) {
    fail(BIPP_INTERNAL_ERROR, "NUFFT spread level count");
  } else {
    n3_spread_kernel<R, LG><<<dim3(grid, p.shares), 64, 0, st>>>(p);
    check_launch("n3_spread_kernel");
    if (p.shares > 1) {
      n3_spread_sum_kernel<R, LG><<<dim3(blocks, 4), 256, 0, st>>>(p);
      check_launch("n3_spread_sum_kernel");
    }
  }
}
}  // namespace

int n3_spread_shares(long long n_blocks, const int (&nback)[3], long long n_points) {
  // Few blocks: their points shared until about 4096 wavefronts (four per SIMD) run or a share
  // gets fewer than 4 batches of points on average; its sums cost a write and a read of 16 to
  // 24 KiB.  50 samples of 60 antennas in double precision: 395 us with up to 2048, 220 + 30 us
  // (the sum) with 4096, 201 + 39 us with 8192; 40 samples of 96 antennas in float, 4096
  // blocks and more: 97 us without shares, 84 + 72 us with 8192.
  const long long reach = n_points * (nback[0] + 1) * (nback[1] + 1) * (nback[2] + 1);
  const long long most = reach / (n_blocks * 256);
  return static_cast<int>(std::max(1LL, std::min({(4096 + n_blocks - 1) / n_blocks, most, 256LL})));
}

template <typename R>
size_t n3_spread_part_elems(long long n_blocks, int shares, int levels) {
  return (size_t)n_blocks * shares * 1024 * std::min(levels, SpreadMfma<R>::levels);
}
template size_t n3_spread_part_elems<float>(long long, int, int);
template size_t n3_spread_part_elems<double>(long long, int, int);

template <typename R>
void launch_n3_spread(const N3SpreadParams<R>& p_all, hipStream_t st) {
  const long long n_blocks = (long long)p_all.nbins[0] * p_all.nbins[1] * p_all.nbins[2];
  if (n_blocks <= 0) return;
  if (n_blocks > 0x7fffffffLL) fail(BIPP_INVALID_PARAMETER_ERROR, "too many NUFFT spread blocks");
  if (p_all.w < 1 || p_all.w > SP_WMAX) fail(BIPP_INVALID_PARAMETER_ERROR, "NUFFT kernel width above 16");
  for (int d = 0; d < 3; ++d)
    if (p_all.bin_size[d] != SP_BIN || (long long)p_all.nbins[d] * SP_BIN < p_all.nf1[d] ||
        p_all.nback[d] < 0 || p_all.nback[d] > 2)
      fail(BIPP_INTERNAL_ERROR, "NUFFT spread blocks do not cover the grid");
  if (p_all.lv_begin < 0 || p_all.lv_end > p_all.n_levels_total || p_all.lv_begin >= p_all.lv_end)
    fail(BIPP_INTERNAL_ERROR, "NUFFT spread level range");
  if (p_all.shares < 1 || (p_all.shares > 1 && !p_all.part))
    fail(BIPP_INTERNAL_ERROR, "NUFFT spread shares");
  // the levels in launches of equal size, at most as many as a kernel keeps sums for
  constexpr int most = SpreadMfma<R>::levels;
  const int n_all = p_all.lv_end - p_all.lv_begin;
  const int launches = (n_all + most - 1) / most;
  const int per = (n_all + launches - 1) / launches;
  for (int lv0 = p_all.lv_begin; lv0 < p_all.lv_end; lv0 += per) {
    N3SpreadParams<R> p = p_all;
    p.lv0 = lv0;
    p.n_levels = std::min(per, p_all.lv_end - lv0);
    // with the XCD order (see the kernel), a multiple of 8 chunks of workgroups; the extra
    // ones exit
    const long long unit = p.xcd_chunk > 0 ? 8LL * p.xcd_chunk : 1;
    const long long grid = (n_blocks + unit - 1) / unit * unit;
    const unsigned nb = static_cast<unsigned>(n_blocks), ng = static_cast<unsigned>(grid);
    switch (p.n_levels) {
      case 1: spread_blocks<R, 1>(p, nb, ng, st); break;
      case 2: spread_blocks<R, 2>(p, nb, ng, st); break;
      case 3: spread_blocks<R, 3>(p, nb, ng, st); break;
      case 4: spread_blocks<R, 4>(p, nb, ng, st); break;
      case 5: spread_blocks<R, 5>(p, nb, ng, st); break;
      default: spread_blocks<R, 6>(p, nb, ng, st); break;
    }
  }
}
template void launch_n3_spread<float>(const N3SpreadParams<float>&, hipStream_t);
template void launch_n3_spread<double>(const N3SpreadParams<double>&, hipStream_t);

namespace {
bool window_ok(const N3Window& w, int n) {
  return n > 0 && w.start >= 0 && w.start < n && w.count >= 0 && w.count <= n;
}
inline int max_radix(const N3Radix& r) {
  int m = 0;
  for (int i = 0; i < r.count; ++i) m = std::max(m, r.r[i]);
  return m;
}
}  // namespace

template <typename R>
bool launch_fft_xlines(const N3LineParams<R>& q, hipStream_t st);

template <typename R>
void launch_fft_lines(const N3LineParams<R>& p, hipStream_t st) {
  const long long n_lines = (long long)p.n_levels * p.zw.count * p.yw.count;
  if (n_lines <= 0) return;
  if (launch_fft_xlines(p, st)) return;
  if (!window_ok(p.yw, p.ny) || !window_ok(p.zw, p.nz) || !window_ok(p.in, p.n) ||
      !window_ok(p.out, p.n))
    fail(BIPP_INTERNAL_ERROR, "FFT line windows out of range");
  // several short lines per workgroup so that every stage keeps most lanes busy
  const int nl = std::max(1, std::min(16, 2048 / p.n));
  if ((long long)nl * p.n > FFT_NT * FFT_PF) fail(BIPP_INTERNAL_ERROR, "FFT line group too long");
  const size_t sh0 = sizeof(cplx<R>) * (2 * (size_t)p.n * nl + twid_len(p.n));
  // 1 KiB of the 160 KiB stays for the kernel's static line bases
  if (sh0 > 159 * 1024) fail(BIPP_INTERNAL_ERROR, "FFT line exceeds LDS");
  // the stages' twiddle tables where two workgroups still fit a CU
  const size_t sh_tab = sh0 + sizeof(cplx<R>) * stage_tab_len(p.n, p.rad);
  const bool tab = sh_tab <= 79 * 1024;
  const size_t sh = tab ? sh_tab : sh0;
  const long long groups = (n_lines + nl - 1) / nl;
  const unsigned blocks = static_cast<unsigned>(std::min<long long>(groups, 32768));
  auto go = [&](auto kernel, bool& attr_set) {
    if (!attr_set) {
      BIPP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024));
      attr_set = true;
    }
    kernel<<<blocks, FFT_NT, sh, st>>>(p, nl);
  };
  // [max radix > 5][stage tables][one line per group]
  static bool attr[2][2][2] = {};
  const bool r16 = max_radix(p.rad) > 5, one = nl == 1;
  if (r16 && tab && one) go(&fft_lines_kernel<R, 16, true, true>, attr[1][1][1]);
  else if (r16 && tab) go(&fft_lines_kernel<R, 16, true, false>, attr[1][1][0]);
  else if (r16 && one) go(&fft_lines_kernel<R, 16, false, true>, attr[1][0][1]);
  else if (r16) go(&fft_lines_kernel<R, 16, false, false>, attr[1][0][0]);
  else if (tab && one) go(&fft_lines_kernel<R, 5, true, true>, attr[0][1][1]);
  else if (tab) go(&fft_lines_kernel<R, 5, true, false>, attr[0][1][0]);
  else if (one) go(&fft_lines_kernel<R, 5, false, true>, attr[0][0][1]);
  else go(&fft_lines_kernel<R, 5, false, false>, attr[0][0][0]);
  check_launch("fft_lines_kernel");
}
template void launch_fft_lines<float>(const N3LineParams<float>&, hipStream_t);
template void launch_fft_lines<double>(const N3LineParams<double>&, hipStream_t);

// The two-stage register pass for m = M1 M2: x positions per item a power of two in
// [16, 2^tw_shift_max] with the line block at most 80 KiB of LDS (two workgroups per CU).
template <typename R, int M1, int M2>
void go_pass_rr(const N3PassParams<R>& p, hipStream_t st) {
  constexpr int M = M1 * M2, LD = M | 1;
  const int tw_cap = p.tw_shift_max >= 4 && p.tw_shift_max <= 7 ? p.tw_shift_max : 6;
  int tw_shift = 4;
  while (tw_shift < tw_cap && (size_t)LD * (2u << tw_shift) * sizeof(cplx<R>) <= 80 * 1024)
    ++tw_shift;
  const int TW = 1 << tw_shift;
  const long long items =
      (long long)((p.xw.count + TW - 1) / TW) * p.n_sub * p.other.count * p.n_levels;
  if (items <= 0) return;
  if (items > 0x7fffffffLL) fail(BIPP_INVALID_PARAMETER_ERROR, "NUFFT grid too large for one pass");
  N3PassParams<R> q = p;
  n3_div_magic((p.xw.count + TW - 1) / TW, q.xt_m, q.xt_s);
  n3_div_magic(p.n_sub, q.sub_m, q.sub_s);
  n3_div_magic(p.other.count, q.oc_m, q.oc_s);
  n3_div_magic(p.operm_n2 > 1 ? p.operm_n1 : 1, q.op_m, q.op_s);
  const size_t sh = sizeof(cplx<R>) * ((size_t)TW * LD + M +
                                       (p.twiddle ? twid_len(static_cast<int>(p.ntot)) : 0));
  if (sh > 96 * 1024) fail(BIPP_INTERNAL_ERROR, "FFT pass exceeds LDS");
  static bool attr = false;
  if (!attr) {
    BIPP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&fft_pass_rr_kernel<R, M1, M2>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
    attr = true;
  }
  const unsigned blocks = static_cast<unsigned>(std::min<long long>(items, 32768));
  fft_pass_rr_kernel<R, M1, M2><<<blocks, FFT_NT, sh, st>>>(q, tw_shift);
}

// factor pairs compiled for the register pass (M1 >= M2, M1 M2 <= 128)
#define BIPP_RR_PAIRS(X)                                                                     \
  X(2, 1) X(2, 2) X(3, 1) X(3, 2) X(3, 3) X(4, 1) X(4, 2) X(4, 3) X(4, 4) X(5, 1) X(5, 2)   \
  X(5, 3) X(5, 4) X(5, 5) X(6, 1) X(6, 2) X(6, 3) X(6, 4) X(6, 5) X(6, 6) X(8, 1) X(8, 2)   \
  X(8, 3) X(8, 4) X(8, 5) X(8, 6) X(8, 8) X(9, 1) X(9, 2) X(9, 3) X(9, 4) X(9, 5) X(9, 6)   \
  X(9, 8) X(9, 9) X(10, 5) X(10, 6) X(10, 9) X(10, 10) X(12, 9) X(12, 10) X(15, 5) X(16, 1) X(16, 2) X(16, 3) X(16, 4) X(16, 5) X(16, 6) X(16, 8)

template <typename R>
bool launch_fft_pass_rr(const N3PassParams<R>& p, hipStream_t st) {
  const int m1 = p.rr_m1, m2 = p.m / std::max(1, p.rr_m1);
  if (m1 * m2 != p.m) return false;
#define BIPP_RR_CASE(A, B)              \
  if (m1 == A && m2 == B) {             \
    go_pass_rr<R, A, B>(p, st);         \
    return true;                        \
  }
  BIPP_RR_PAIRS(BIPP_RR_CASE)
#undef BIPP_RR_CASE
  return false;
}

bool fft_rr_factors(int m, int& m1, int& m2) {
#define BIPP_RR_FIND(A, B)   \
  if (A * B == m) {          \
    m1 = A;                  \
    m2 = B;                  \
    found = true;            \
  }
  bool found = false;
  BIPP_RR_PAIRS(BIPP_RR_FIND)  // the last match: the largest first factor
#undef BIPP_RR_FIND
  return found;
}

// x positions per workgroup of the one-pass form as a power of two, or -1.  Up to 16 where two
// workgroups of 512 threads fit a CU, down to 2 with one of 1024 (rows of 16 bytes in float, the
// rest of a line is its neighbours' on the same XCD); two positions are still faster than two
// passes (the 512-antenna case's axes of 6000 to 6912 points 10.0 to 7.3 ms), 8 positions in half
// a CU's LDS than in all of it (121 against 126 us at 40 samples of 96 antennas).
int fft_axis_shift(int n, size_t elem) {
  for (int k = 4; k >= 1; --k)
    if (elem * ((size_t)(n + 32) << k) <= (k >= 3 ? 76 : 152) * 1024) return k;
  return -1;
}

// radices of a contiguous axis: at most four, the fewest, the most even of those
bool fft_line_radices(int n, int (&f)[4]) {
  constexpr int rad[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
  int best = 5, best_max = 17, cur[4];
  auto go = [&](auto&& self, int m, int k, int top) -> void {
    if (m == 1) {
      if (k < best || (k == best && cur[0] < best_max)) {
        best = k;
        best_max = cur[0];
        for (int i = 0; i < 4; ++i) f[i] = i < k ? cur[i] : 1;
      }
      return;
    }
    if (k == 4 || k >= best) return;
    for (int r : rad)
      if (r <= top && m % r == 0) {
        cur[k] = r;
        self(self, m / r, k + 1, r);
      }
  };
  go(go, n, 0, 16);
  return best >= 2 && best <= 4;
}

// The LDS limit is a property of the kernel, so its flag belongs to the instantiation (the kernels
// of the two workgroup sizes have one function type), and is set once the runtime took the limit.
template <typename R, int NT, bool NAT>
void start_fft_axis(const N3AxisParams<R>& p, long long items, size_t sh, hipStream_t st) {
  static std::atomic<bool> attr{false};
  if (!attr) {
    BIPP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&fft_axis_kernel<R, NT, NAT>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024));
    attr = true;
  }
  // a round is one tile per resident workgroup
  const long long round = sh <= 39 * 1024 ? 1024 : sh <= 52 * 1024 ? 768 : sh <= 79 * 1024 ? 512 : 256;
  fft_axis_kernel<R, NT, NAT><<<static_cast<unsigned>(std::min(items, round)), NT, sh, st>>>(p);
}

template <typename R, bool NAT>
bool go_fft_axis(N3AxisParams<R> p, const int (&f)[4], hipStream_t st) {
  if (!window_ok(p.xw, p.nx) || !window_ok(p.other, p.no) || !window_ok(p.in, p.n) ||
      !window_ok(p.out, p.n))
    fail(BIPP_INTERNAL_ERROR, "FFT pass windows out of range");
  p.stages = 0;
  int done = 1;
  for (int k = 0; k < 4; ++k) {
    if (f[k] == 1) continue;
    const int s = p.stages++;
    p.r[s] = f[k];
    p.weight[s] = done;
    done *= f[k];
    p.span[s] = p.n / done;
    n3_div_magic(p.span[s], p.sp_m[s], p.sp_s[s]);
    n3_div_magic(p.n / f[k], p.per_m[s], p.per_s[s]);
    n3_div_magic(f[k], p.rd_m[s], p.rd_s[s]);
  }
  if (!NAT) p.last_step = p.weight[p.stages - 1] / p.n1;
  n3_div_magic(NAT ? 1 : p.n1, p.n1_m, p.n1_s);
  // line stride 32 / positions modulo 32 elements: a row of positions in different banks
  const int want = 32 >> p.tw_shift;
  p.ld = NAT ? p.n : p.n + ((want - p.n) % 32 + 32) % 32;
  const int TW = 1 << p.tw_shift;
  const long long items = (long long)((p.xw.count + TW - 1) / TW) * p.other.count * p.n_levels;
  if (items <= 0) return true;
  if (items > 0x7fffffffLL) fail(BIPP_INVALID_PARAMETER_ERROR, "NUFFT grid too large for one pass");
  n3_div_magic((p.xw.count + TW - 1) / TW, p.xt_m, p.xt_s);
  n3_div_magic(p.other.count, p.oc_m, p.oc_s);
  n3_div_magic(p.operm_n2 > 1 ? p.operm_n1 : 1, p.op_m, p.op_s);
  const size_t sh = sizeof(cplx<R>) * (((size_t)p.ld << p.tw_shift) + twid_len(p.n));
  // x lines (at most 4096 elements per tile) stay below 79 KiB
  if (sh > (NAT ? 79 : 159) * 1024) fail(BIPP_INTERNAL_ERROR, "FFT pass exceeds LDS");
  if (NAT || sh <= 79 * 1024)
    start_fft_axis<R, 512, NAT>(p, items, sh, st);
  else if constexpr (!NAT)
    start_fft_axis<R, 1024, false>(p, items, sh, st);
  check_launch("fft_axis_kernel");
  return true;
}

bool fft_axis_radices(int n, int n1, int n2, int (&f)[4]) {
  return n2 >= 2 && (long long)n1 * n2 == n && fft_rr_factors(n1, f[0], f[1]) && fft_rr_factors(n2, f[2], f[3]);
}
bool fft_axis_form(int n, int n1, int n2, size_t elem) {
  int f[4];
  return fft_axis_radices(n, n1, n2, f) && fft_axis_shift(n, elem) >= 0;
}

template <typename R>
bool launch_fft_axis(const N3AxisParams<R>& p_in, hipStream_t st) {
  N3AxisParams<R> p = p_in;
  int f[4];
  if (!fft_axis_radices(p.n, p.n1, p.n2, f)) return false;
  p.tw_shift = fft_axis_shift(p.n, sizeof(cplx<R>));
  return p.tw_shift >= 0 && go_fft_axis<R, false>(p, f, st);
}

// x lines by the same stages, up to 2048 points: two lines and more per workgroup, one buffer
// instead of two.  Above, fft_lines_kernel's prefetch and twiddle tables are as good or better
// (FFT of 64-antenna samples, x and y of 1800 points: 13.7 to 10.6 ms with this form, 768 points
// 3.1 to 2.1, 240 points 0.49 to 0.39; 2160 points 18.9 and 18.5 in float, 51.9 and 53.4 in
// double; 3240 points 3.27 against 3.80 for the lines alone, 6000 5.98 against 7.42).
constexpr int FFT_XLINES_MAX = 2048;
bool fft_xlines_form(int n) {
  int f[4];
  return n <= FFT_XLINES_MAX && fft_line_radices(n, f);
}

template <typename R>
bool launch_fft_xlines(const N3LineParams<R>& q, hipStream_t st) {
  N3AxisParams<R> p{};
  int f[4];
  if (q.n > FFT_XLINES_MAX || !fft_line_radices(q.n, f)) return false;
  p.grid = q.grid;
  p.grid_stride = q.grid_stride;
  p.n_levels = q.n_levels;
  p.nx = q.ny;
  p.xw = q.yw;
  p.no = q.nz;
  p.other = q.zw;
  p.operm_n1 = p.operm_n2 = 1;
  p.outer_stride = (long long)q.n * q.ny;
  p.axis_stride = 1;
  p.n = q.n;
  p.in = q.in;
  p.out = q.out;
  p.tw = q.tw;
  while (p.tw_shift < 4 && (q.n << (p.tw_shift + 1)) <= 4096) ++p.tw_shift;
  return go_fft_axis<R, true>(p, f, st);
}
template bool launch_fft_axis<float>(const N3AxisParams<float>&, hipStream_t);
template bool launch_fft_axis<double>(const N3AxisParams<double>&, hipStream_t);

template <typename R>
void launch_fft_pass(const N3PassParams<R>& p_in, hipStream_t st) {
  N3PassParams<R> p = p_in;
  if (!window_ok(p.xw, p.nx) || !window_ok(p.other, p.no) || !window_ok(p.in, p.nax) ||
      !window_ok(p.out, p.nax) || (long long)p.m * p.n_sub != p.nax ||
      (p.twiddle && p.ntot != p.nax))
    fail(BIPP_INTERNAL_ERROR, "FFT pass windows out of range");
  // x positions per item: a power of two in [16, 64] with about 4096 elements per item
  const int ld = p.m | 1;
  const int tw_cap = p.tw_shift_max >= 4 && p.tw_shift_max <= 6 ? p.tw_shift_max : 6;
  int tw_shift = 4;
  while (tw_shift < tw_cap && (ld << (tw_shift + 1)) <= 4096) ++tw_shift;
  const int TW = 1 << tw_shift;
  if ((long long)p.m * TW > FFT_NT * FFT_PF) fail(BIPP_INTERNAL_ERROR, "FFT pass item too large");
  const long long items =
      (long long)((p.xw.count + TW - 1) / TW) * p.n_sub * p.other.count * p.n_levels;
  if (items <= 0) return;
  if (items > 0x7fffffffLL) fail(BIPP_INVALID_PARAMETER_ERROR, "NUFFT grid too large for one pass");
  if (p.operm_n2 > 1 && p.operm_n1 < 1) fail(BIPP_INTERNAL_ERROR, "FFT pass permutation");
  n3_div_magic((p.xw.count + TW - 1) / TW, p.xt_m, p.xt_s);
  n3_div_magic(p.n_sub, p.sub_m, p.sub_s);
  n3_div_magic(p.other.count, p.oc_m, p.oc_s);
  n3_div_magic(p.operm_n2 > 1 ? p.operm_n1 : 1, p.op_m, p.op_s);
  const size_t sh = sizeof(cplx<R>) * (2 * (size_t)TW * ld + twid_len(p.m) +
                                       (p.twiddle ? twid_len(static_cast<int>(p.ntot)) : 0));
  if (sh > 160 * 1024) fail(BIPP_INTERNAL_ERROR, "FFT pass exceeds LDS");
  const unsigned blocks = static_cast<unsigned>(std::min<long long>(items, 32768));
  auto go = [&](auto kernel, bool& attr_set) {
    if (!attr_set) {
      BIPP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
      attr_set = true;
    }
    kernel<<<blocks, FFT_NT, sh, st>>>(p, tw_shift);
  };
  if (p.rr_m1 > 0) {
    if (!launch_fft_pass_rr(p, st)) fail(BIPP_INTERNAL_ERROR, "FFT pass factors not compiled");
    check_launch("fft_pass_rr_kernel");
    return;
  }
  static bool attr5 = false, attr16 = false;
  if (max_radix(p.rad) > 5)
    go(&fft_pass_kernel<R, 16>, attr16);
  else
    go(&fft_pass_kernel<R, 5>, attr5);
  check_launch("fft_pass_kernel");
}
template void launch_fft_pass<float>(const N3PassParams<float>&, hipStream_t);
template void launch_fft_pass<double>(const N3PassParams<double>&, hipStream_t);

template <typename R, typename TI>
void launch_n3_interp(const N3InterpParams<R>& p, hipStream_t st) {
  if (p.n_pix <= 0) return;
  const dim3 grid(ceil_div(p.n_pix, 256)), block(256);
  switch (p.w2) {
#define BIPP_INTERP_W(W) \
  case W: n3_interp_kernel<R, TI, W><<<grid, block, 0, st>>>(p); break;
    BIPP_INTERP_W(2) BIPP_INTERP_W(3) BIPP_INTERP_W(4) BIPP_INTERP_W(5) BIPP_INTERP_W(6)
    BIPP_INTERP_W(7) BIPP_INTERP_W(8) BIPP_INTERP_W(9) BIPP_INTERP_W(10) BIPP_INTERP_W(11)
    BIPP_INTERP_W(12) BIPP_INTERP_W(13) BIPP_INTERP_W(14) BIPP_INTERP_W(15) BIPP_INTERP_W(16)
#undef BIPP_INTERP_W
    default: fail(BIPP_INVALID_PARAMETER_ERROR, "NUFFT kernel width outside [2, 16]");
  }
  check_launch("n3_interp_kernel");
}
template void launch_n3_interp<float, float>(const N3InterpParams<float>&, hipStream_t);
template void launch_n3_interp<double, double>(const N3InterpParams<double>&, hipStream_t);

// Workgroups per pixel block: about eight per CU over all blocks, at least 512 slots each.
int direct_chunks(long long n_slots, int n_pix, int n_cu) {
  const long long blocks = ceil_div(n_pix, 256);
  return static_cast<int>(std::max<long long>(1, std::min((8LL * n_cu) / std::max(1LL, blocks), n_slots / 512)));
}

template <typename R>
void launch_direct_sum(const N3DirectParams<R>& p, hipStream_t st) {
  if (p.n_pix <= 0 || p.n_slots <= 0 || p.n_levels <= 0) return;
  if (p.n_levels > 8 || p.chunks < 1 || p.chunks > 65535) fail(BIPP_INTERNAL_ERROR, "direct sum arguments");
  const dim3 grid(ceil_div(p.n_pix, 256), p.chunks);
  if (p.n_levels == 1)
    direct_sum_kernel<R, 1><<<grid, 256, 0, st>>>(p);
  else if (p.n_levels == 2)
    direct_sum_kernel<R, 2><<<grid, 256, 0, st>>>(p);
  else if (p.n_levels <= 4)
    direct_sum_kernel<R, 4><<<grid, 256, 0, st>>>(p);
  else
    direct_sum_kernel<R, 8><<<grid, 256, 0, st>>>(p);
  check_launch("direct_sum_kernel");
  if (p.chunks == 1) return;
  direct_reduce_kernel<R><<<dim3(ceil_div(p.n_pix, 256), p.n_levels), 256, 0, st>>>(p);
  check_launch("direct_reduce_kernel");
}
template void launch_direct_sum<float>(const N3DirectParams<float>&, hipStream_t);
template void launch_direct_sum<double>(const N3DirectParams<double>&, hipStream_t);

template <typename TO>
void launch_vv_trace(int n_samples, int n_levels, const int* n_rows, int n_rows_const, void* vv,
                     long long vv_stride, long long ld_vv, hipStream_t st) {
  if (n_samples <= 0 || n_levels <= 0) return;
  if (ld_vv < 2) fail(BIPP_INTERNAL_ERROR, "trace slot needs at least two rows");
  vv_trace_kernel<TO><<<n_samples * n_levels, 256, 0, st>>>(
      n_levels, n_rows, n_rows_const, static_cast<cplx<TO>*>(vv), vv_stride, ld_vv);
  check_launch("vv_trace_kernel");
}
template void launch_vv_trace<float>(int, int, const int*, int, void*, long long, long long,
                                     hipStream_t);
template void launch_vv_trace<double>(int, int, const int*, int, void*, long long, long long,
                                      hipStream_t);

template <typename R, typename TO>
void launch_vv_levels(const N3VVParams<R>& p, int n_samples, int n_rows_max, hipStream_t st) {
  if (n_samples <= 0 || n_rows_max <= 0) return;
  if constexpr (std::is_same<R, double>::value) {
    const long long nt = ceil_div(n_rows_max, 64), n_tiles = nt * (nt + 1) / 2;
    const long long n_units = n_tiles * n_samples * p.n_levels;
    const long long per_xcd = (n_units + 7) / 8;
    if (8 * per_xcd > 0x7fffffffLL) fail(BIPP_INVALID_PARAMETER_ERROR, "too many VV tiles for one launch");
    vv_levels_mfma_kernel<TO><<<static_cast<unsigned>(8 * per_xcd), 256, 0, st>>>(
        p, static_cast<int>(n_tiles), static_cast<int>(per_xcd), static_cast<int>(n_units));
    check_launch("vv_levels_mfma_kernel");
  } else {
    dim3 grid(ceil_div(n_rows_max, 64), ceil_div(n_rows_max, 64), n_samples * p.n_levels);
    vv_levels_kernel<R, TO><<<grid, 256, 0, st>>>(p);
    check_launch("vv_levels_kernel");
  }
}
template void launch_vv_levels<double, float>(const N3VVParams<double>&, int, int, hipStream_t);
template void launch_vv_levels<double, double>(const N3VVParams<double>&, int, int, hipStream_t);
template void launch_vv_levels<float, float>(const N3VVParams<float>&, int, int, hipStream_t);
template void launch_vv_levels<float, double>(const N3VVParams<float>&, int, int, hipStream_t);

}  // namespace bippamd
