// Phase-split form of the batched generalized eigensolver (float64): one launch per phase over
// all samples of a batch instead of one workgroup per sample for all phases.
//
// The persistent kernel (eig_kernel) gives a sample one CU, so a batch of fewer samples than
// CUs leaves the rest of the chip idle and a sample takes its single-CU time: 55 ms for twelve
// 400..512-antenna samples, 64 ms for 96 of them (tridiagonalisation 23, back-transform 17,
// whitening 3.9, un-whitening 3.0, load 1.3 ms per sample).  Here the dense phases run on tiles
// or column groups of every sample, and the tridiagonalisation, whose column steps depend on
// each other, takes one launch per column with several workgroups per sample.  The divide and
// conquer keeps a workgroup per sample (the phase of eig_kernel).
//
// Buffers (leading dimension nmax): p.z_out[sample] holds the reduced S, then C, then the
// reflectors and T factors, and in the end the eigenvectors; p.ws_l[job] G, then W = L^-1;
// p.ws_a[job] scratch (W S, the divide and conquer's arrays, the back-transformed vectors);
// p.ws_z[job] the eigenvectors of the tridiagonal.  job: position in p.order.
#pragma once

// Job and unit of a workgroup when the `per_job` units of a job are to run on one XCD (workgroup
// x runs on XCD x mod 8): a job's operands then stay in that XCD's L2.  Each XCD takes an eighth
// of the units in the order of jobs 0, 8, 16, .., 1, 9, ..: jobs come largest first, so in their own
// order the first XCD would get the largest (96 jobs of 400..512 beams: 30.7 against 29.0 ms).
struct SplitUnit {
  int job, unit;
};
__device__ __forceinline__ SplitUnit split_unit(int per_job, int n_jobs) {
  const int n_units = per_job * n_jobs, per_xcd = (n_units + 7) / 8;
  const int u = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || u >= n_units) return {-1, 0};
  const int q = u / per_job, full = n_jobs & 7, len = n_jobs >> 3;  // `full` sequences of len + 1
  const int q1 = q - full * (len + 1);
  const int job = q1 < 0 ? q % (len + 1) * 8 + q / (len + 1) : q1 % len * 8 + full + q1 / len;
  return {job, u % per_job};
}
inline unsigned split_grid(int per_job, int n_jobs) {
  return static_cast<unsigned>(8 * ((static_cast<long long>(per_job) * n_jobs + 7) / 8));
}

// The reduced pencil: S (full) into z_out, G into ws_l.  Workgroup: 16 columns of one job.
template <typename TIn>
__global__ __launch_bounds__(256) void split_load_kernel(EigParams<double> p) {
  const int job = blockIdx.y, sid = p.order[job], n = p.n_red[sid];
  const int j1 = min(n, static_cast<int>(blockIdx.x) * 16 + 16);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int* idx = p.idx + (size_t)sid * p.idx_stride;
  const cplx<TIn>* S = reinterpret_cast<const cplx<TIn>*>(p.s) + (size_t)sid * p.stride_s;
  const double* xyz = p.xyz + (size_t)sid * p.stride_xyz;
  const cplx<double>* Gin = p.g_in ? p.g_in + (size_t)sid * p.stride_g : nullptr;
  cplx<double>* A = p.z_out + (size_t)sid * p.stride_z;
  cplx<double>* L = p.ws_l + (size_t)job * p.ws_stride;
  const double wl = p.wl[sid];
  for (int j = blockIdx.x * 16 + wave; j < j1; j += 4) {
    const int bj = idx[j];
    for (int i = lane; i < n; i += 64) {
      const int bi = idx[i];
      cplx<TIn> sv = (bi >= bj) ? S[bi + (size_t)bj * p.lds] : conj(S[bj + (size_t)bi * p.lds]);
      cplx<double> a = cvt<double>(sv);
      if (i == j) a.im = 0;
      A[i + (size_t)j * p.ldz] = a;
      cplx<double> g;
      if (Gin) {
        g = Gin[i + (size_t)j * p.ld_g];
      } else if (i == j) {
        g = mk<double>(p.gram_prefactor, 0);
      } else {
        const double dx = xyz[bi] - xyz[bj], dy = xyz[bi + p.ldxyz] - xyz[bj + p.ldxyz],
                     dz = xyz[bi + 2 * p.ldxyz] - xyz[bj + 2 * p.ldxyz];
        const double x = 2.0 * sqrt(dx * dx + dy * dy + dz * dz) / wl;
        const double sc = x != 0.0 ? sinpi(x) / (3.14159265358979323846 * x) : 1.0;
        g = mk<double>(p.gram_prefactor * sc, 0);
      }
      L[i + (size_t)j * p.ws_ld] = g;
    }
  }
}

// W = L^-1 of G = L L^H in place (scratch ws_a): the steps of chol_inverse, the diagonal blocks
// on a workgroup per job, the products on one per tile; bound by the chain of diagonal blocks
// (0.47 ms) and, at many jobs, the trailing matrix's traffic.  96 jobs of 400..512 beams 3.75 to
// 1.96 ms, 12 jobs 3.4 to 0.99 ms against one workgroup per job for all steps.
constexpr int SCH_NT = 256, SCH_DIAG_NT = 512;

// diagonal block of column j0; info and, where there is nothing to solve, the eigenvalues
__global__ __launch_bounds__(SCH_DIAG_NT) void split_chol_diag_kernel(EigParams<double> p, int j0) {
  const int job = blockIdx.x, sid = p.order[job], n = p.n_red[sid], tid = threadIdx.x;
  __shared__ CiShared<double> sh;
  if (j0 == 0 ? n <= 0 : (j0 >= n || p.info[sid])) {  // uniform
    if (j0 == 0) {
      for (int j = tid; j < p.nmax; j += SCH_DIAG_NT) p.d_out[(size_t)sid * p.stride_d + j] = 0;
      if (tid == 0) p.info[sid] = 0;
    }
    return;
  }
  WgTeam tm{tid};
  const int bad = chol_diagonal<double, SCH_DIAG_NT>(tm, n, j0, global_ptr(p.ws_l + (size_t)job * p.ws_stride),
                                                p.ws_ld, sh);
  // leading minor bad + 1 of G is not positive definite: ?hegv reports info = n + bad + 1
  if (bad >= 0)
    for (int j = tid; j < p.nmax; j += SCH_DIAG_NT) p.d_out[(size_t)sid * p.stride_d + j] = 0;
  if (tid == 0 && (bad >= 0 || j0 == 0)) p.info[sid] = bad >= 0 ? n + bad + 1 : 0;
}

// one tile of a product per workgroup: STEP 0 the panel below diagonal block j0, 1 the trailing
// matrix, 2 and 3 T and W21 of the pairs of blocks of size j0 (unit: pair, tile)
template <int STEP>
__global__ __launch_bounds__(SCH_NT) void split_chol_tile_kernel(EigParams<double> p, int j0, int per_job,
                                                                 int tiles) {
  const SplitUnit u = split_unit(per_job, p.n_jobs);
  if (u.job < 0) return;
  const int sid = p.order[u.job], n = p.n_red[sid];
  if (n <= 0 || p.info[sid]) return;
  __shared__ CiShared<double> sh;
  WgTeam tm{static_cast<int>(threadIdx.x)};
  BIPP_GLOBAL cplx<double>* L = global_ptr(p.ws_l + (size_t)u.job * p.ws_stride);
  BIPP_GLOBAL cplx<double>* T = global_ptr(p.ws_a + (size_t)u.job * p.ws_stride);
  constexpr int ONE = 1 << 30;  // no second tile
  if (STEP == 0) chol_panel<double, SCH_NT>(tm, n, j0, L, p.ws_ld, sh, u.unit, ONE);
  if (STEP == 1) chol_trailing<double, SCH_NT>(tm, n, j0, L, p.ws_ld, sh, u.unit, ONE);
  if (STEP >= 2) {
    const int b0 = u.unit / tiles * 2 * j0;
    if (b0 + j0 >= n) return;
    if (STEP == 2) chol_pair_t<double, SCH_NT>(tm, n, j0, b0, L, p.ws_ld, T, p.ws_ld, sh, u.unit % tiles, ONE);
    if (STEP == 3) chol_pair_w<double, SCH_NT>(tm, n, j0, b0, L, p.ws_ld, T, p.ws_ld, sh, u.unit % tiles, ONE);
  }
}

inline void launch_split_chol(const EigParams<double>& p, int n_max, hipStream_t stream) {
  const int jobs = p.n_jobs;
  for (int j0 = 0; j0 < std::max(n_max, 1); j0 += CI_CB) {
    split_chol_diag_kernel<<<jobs, SCH_DIAG_NT, 0, stream>>>(p, j0);
    const int rows = n_max - j0 - CI_CB, t = rows > 0 ? ceil_div(rows, CI_T) : 0;
    if (t == 0) continue;
    split_chol_tile_kernel<0><<<split_grid(t, jobs), SCH_NT, 0, stream>>>(p, j0, t, t);
    const int tt = t * (t + 1) / 2;
    split_chol_tile_kernel<1><<<split_grid(tt, jobs), SCH_NT, 0, stream>>>(p, j0, tt, tt);
  }
  for (int s = CI_CB; s < n_max; s *= 2) {
    const int pairs = ceil_div(n_max - s, 2 * s), side = ceil_div(s, CI_T), tiles = side * side;
    split_chol_tile_kernel<2><<<split_grid(pairs * tiles, jobs), SCH_NT, 0, stream>>>(p, s, pairs * tiles, tiles);
    split_chol_tile_kernel<3><<<split_grid(pairs * tiles, jobs), SCH_NT, 0, stream>>>(p, s, pairs * tiles, tiles);
  }
  check_launch("split_chol_kernel");
}

// Dense products on 64 x 64 tiles, a wavefront per 32 x 32 quadrant (2 x 2 blocks of
// v_mfma_f64_16x16x4f64, four per complex product), operands straight from global memory with
// the next four k in flight: an MFMA takes 64 cycles, so a CU reads 16 bytes per cycle, a
// quarter of what its L1 delivers, and neither LDS nor barriers are needed.  D[j][i] is
// formed (A operand: rows j, B operand: rows i), so stores write 16 consecutive rows.
//   MODE 0: ws_a = W S       = sum_{k <= i} W[i,k] conj(S[j,k])          (S Hermitian)
//   MODE 1: z_out = ws_a W^H = sum_{k <= j} X[i,k] conj(W[j,k]), lower triangle, real diagonal
//   MODE 2: z_out = W^H ws_a = sum_{k >= i} conj(W[k,i]) X[k,j]
template <int MODE>
__global__ __launch_bounds__(256) void split_gemm_kernel(EigParams<double> p, int tiles_side) {
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  const int n_tiles = MODE == 1 ? tiles_side * (tiles_side + 1) / 2 : tiles_side * tiles_side;
  const SplitUnit u = split_unit(n_tiles, p.n_jobs);
  if (u.job < 0) return;
  const int sid = p.order[u.job], n = p.n_red[sid];
  if (p.info[sid] != 0) return;
  int ti, tj;
  if (MODE == 1) {
    ti = 0;
    while ((ti + 1) * (ti + 2) / 2 <= u.unit) ++ti;
    tj = u.unit - ti * (ti + 1) / 2;
  } else {
    ti = u.unit % tiles_side;
    tj = u.unit / tiles_side;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ib = 64 * ti + 32 * (wave & 1), jb = 64 * tj + 32 * (wave >> 1);
  if (ib >= n || jb >= n || (MODE == 1 && jb > ib + 31)) return;
  const int ld = p.ws_ld;
  const cplx<double>* W = p.ws_l + (size_t)u.job * p.ws_stride;
  cplx<double>* X = p.ws_a + (size_t)u.job * p.ws_stride;
  cplx<double>* A = p.z_out + (size_t)sid * p.stride_z;
  const int lr = lane & 15, lk = lane >> 4;
  const int jr[2] = {jb + lr, jb + 16 + lr}, ir[2] = {ib + lr, ib + 16 + lr};
  const int k1 = MODE == 0 ? min(n, ib + 32) : (MODE == 1 ? min(n, jb + 32) : n);
  f64x4 dr[2][2], di[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      dr[a][b] = f64x4{0, 0, 0, 0};
      di[a][b] = f64x4{0, 0, 0, 0};
    }
  // Operands of step k for this lane's k + lk.  Rows past n read row n - 1 (their results are not
  // stored).  MASK: k past k1 and, in the triangular operand, elements of the other triangle
  // give zero; the steps between need no test, so their loads are a uniform base plus a fixed
  // lane offset (with a test and a 64-bit address per load the vector ALU took 10
  // instructions per MFMA, which the float64 MFMA does not overlap: 1.54 against 1.21 ms for 96
  // products of 400..512 rows).
  const unsigned uld = ld;
  unsigned oj[2], oi[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const unsigned j = min(jr[b], n - 1), i = min(ir[b], n - 1);
    oj[b] = MODE == 2 ? lk + j * uld : j + lk * uld;
    oi[b] = MODE == 2 ? lk + i * uld : i + lk * uld;
  }
  auto load = [&](auto mask, int k, cplx<double>* P, cplx<double>* Q) __attribute__((always_inline)) {
    const cplx<double>* bp = (MODE == 0 ? A : (MODE == 1 ? W : X)) + (MODE == 2 ? (size_t)k : (size_t)k * uld);
    const cplx<double>* bq = (MODE == 1 ? X : W) + (MODE == 2 ? (size_t)k : (size_t)k * uld);
    const int e = k + lk;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (!decltype(mask)::value) {
        P[b] = bp[oj[b]];
        Q[b] = bq[oi[b]];
        continue;
      }
      P[b] = Q[b] = mk<double>(0, 0);
      if (e < k1) {
        if (MODE != 1 || e <= jr[b]) P[b] = bp[oj[b]];
        if (MODE == 1 || (MODE == 0 ? e <= ir[b] : e >= ir[b])) Q[b] = bq[oi[b]];
      }
    }
  };
  auto mul = [&](const cplx<double>* P, const cplx<double>* Q) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const double np = -P[a].im;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // conj(P) Q: re Pr Qr + Pi Qi, im Pr Qi - Pi Qr (MODE 2: P conj(Q), the conjugate)
        dr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].re, Q[b].re, dr[a][b], 0, 0, 0);
        dr[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].im, Q[b].im, dr[a][b], 0, 0, 0);
        di[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[a].re, Q[b].im, di[a][b], 0, 0, 0);
        di[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(np, Q[b].re, di[a][b], 0, 0, 0);
      }
    }
  };
  auto run = [&](auto mask, int ka, int kb) __attribute__((always_inline)) {
    if (ka >= kb) return;
    cplx<double> P[2][2], Q[2][2];
    load(mask, ka, P[0], Q[0]);
    for (int k = ka; k < kb; k += 8) {
      if (k + 4 < kb) load(mask, k + 4, P[1], Q[1]);
      mul(P[0], Q[0]);
      if (k + 4 >= kb) break;
      if (k + 8 < kb) load(mask, k + 8, P[0], Q[0]);
      mul(P[1], Q[1]);
    }
  };
  constexpr std::true_type MASKED{};
  constexpr std::false_type PLAIN{};
  if (MODE == 2) {
    const int k2 = n & ~3;
    run(MASKED, ib, min(n, ib + 32));
    run(PLAIN, ib + 32, k2);
    if (k2 >= ib + 32) run(MASKED, k2, n);
  } else {
    const int kd = MODE == 0 ? ib : jb;  // the triangular operand's diagonal blocks begin
    run(PLAIN, 0, kd);
    run(MASKED, kd, k1);
  }
  cplx<double>* out = MODE == 0 ? X : A;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = jb + 16 * a + lk + 4 * r, i = ir[b];
        if (i >= n || j >= n || (MODE == 1 && i < j)) continue;
        double im = MODE == 2 ? -di[a][b][r] : di[a][b][r];
        if (MODE == 1 && i == j) im = 0;
        out[i + (size_t)j * ld] = mk<double>(dr[a][b][r], im);
      }
}

// --------------------------------------------------------------------------------------
// Tridiagonalisation (zhetd2 order, lower triangle): the first n - TRI_TAIL columns with one
// launch per column c, the trailing matrix that is left in the registers of one workgroup per
// sample (split_tail_kernel).
//
// State between launches: the reflectors v, tau of the last TRI_LAG columns and their w, and
// y = A v_{c-1} over the trailing matrix as per-workgroup row sums plus the column sums.  Launch c
//   - forms w_{c-1} from y, v_{c-1}, tau_{c-1}, the updated column c and its reflector v_c (every
//     workgroup of the sample for itself, from the same operands in the same order, so all
//     hold the same bits; workgroup 0 records d_c, e_c, v_c, tau_c, w_{c-1} and puts v_{c-1} into
//     its column of A);
//   - applies the P pending updates A -= v w^H + w v^H to its columns of the trailing matrix and
//     adds their part of A v_c from the updated lower triangle.  The updated elements are
//     stored in every TRI_LAG-th launch only; the others repeat them from the same operands.
//   - at c = n - TRI_TAIL forms no reflector and stores what is pending.
// Bound: the launches follow each other (a prologue of two workgroup sums and the round trip
// through the last-level cache per launch), then, for many samples, the last-level cache (the
// trailing triangle read once per column and written once per TRI_LAG).  Lanes hold 16 rows x 4
// columns, so a column's sum takes four lane moves for four columns at once, and row sums over
// the columns of a wavefront stay in registers.  Column tiles of 4 are dealt to the sample's
// wavefronts in turn, which keeps them balanced while the trailing matrix shrinks.
// Measured, batches of 400..512 beams: 96 samples 28.3 to 24.8 ms, 12 samples 15.4 to 14.1 ms against
// launches for all columns that store every time; over the first 256 columns of 96 samples a
// storing launch takes 43 us on average, one that does not 30 us, the tail kernel 1.84 ms.  (Longer
// lags could save a sixth of a launch at most and take the LDS of the second workgroup.)
// --------------------------------------------------------------------------------------
constexpr int TRI_N = 512;   // largest reduced size
constexpr int TRI_GMAX = 8;  // workgroups per sample of a launch
constexpr int TRI_TAIL = 256;  // columns left to split_tail_kernel
constexpr int TRI_LAG = 2;   // columns per store of the trailing matrix
constexpr int TRI_RING = TRI_LAG + 1;

struct TriWork {
  cplx<double>* v;     // [job][TRI_RING][nmax], column c in slot c mod TRI_RING
  cplx<double>* w;     // [job][TRI_RING][nmax]
  cplx<double>* tau;   // [job][2]
  cplx<double>* col;   // [job][2][nmax] column sums
  cplx<double>* row;   // [job][2][TRI_GMAX][nmax] row sums of each workgroup
  double* de;          // [job][nmax][2] diagonal, subdiagonal
  int* perm;           // [job][nmax]
};

template <int NW, int P>
struct TriShared {
  cplx<double> v[P ? P : 1][TRI_N], w[P ? P : 1][TRI_N];  // pending updates, newest first
  cplx<double> vn[TRI_N];
  cplx<double> xw[NW][TRI_N];  // a wavefront's row sums
  double red[2][2 * NW];
  cplx<double> yc, alpha, vc[P ? P : 1], wc[P ? P : 1];  // row c of y and of the older updates
};

// sums of a and b over the workgroup in a fixed order; one barrier (slots alternate)
template <int NW>
__device__ __forceinline__ void tri_sum2(double& a, double& b, double* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  a = wave_total(a);
  b = wave_total(b);
  if (lane == 0) {
    red[wave] = a;
    red[NW + wave] = b;
  }
  __syncthreads();
  a = 0;
  b = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    a += red[w];
    b += red[NW + w];
  }
}

// NCT: column tiles of a wavefront taken together (a tile's row operands are read once)
// P: pending updates, those of columns c - 1 .. c - P
template <int NT, int NCT, int P>
__global__ __launch_bounds__(NT) void tri_column_kernel(EigParams<double> p, TriWork tw, int c) {
  constexpr int NW = NT / 64, RPT = TRI_N / NT;
  __shared__ TriShared<NW, P> sh;
  const int job = blockIdx.y, g = blockIdx.x, G = gridDim.x;
  const int sid = p.order[job], n = p.n_red[sid];
  const int last = n - TRI_TAIL;  // the column that hands over
  if (c > last || last <= 0 || p.info[sid] != 0) return;  // uniform
  const bool hand = c == last, keep = hand || P == TRI_LAG;  // keep: store the updated elements
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ld = p.ldz, nmax = p.nmax;
  cplx<double>* A = p.z_out + (size_t)sid * p.stride_z;
  const int cur = c & 1, prv = cur ^ 1;
  const size_t j2 = (size_t)job * 2;
  const size_t jr = (size_t)job * TRI_RING;
  auto slot = [&](int col) { return (jr + col % TRI_RING) * nmax; };

  const int i0 = hand ? c : c + 1;
  const int lr = lane & 15, lc = lane >> 4;
  const int W = G * NW, gw = g * NW + wave;
  const int ct_end = (n + 3) >> 2, rt_end = (n + 15) >> 4;
  constexpr int RU = 8 / NCT;  // row tiles loaded together: eight elements in flight per lane
  int ct = i0 >> 2;
  ct += (gw - ct % W + W) % W;  // first tile at or after column i0 that is this wavefront's
  int jc[NCT];
  auto tiles = [&]() {
#pragma unroll
    for (int u = 0; u < NCT; ++u) {
      const int j = 4 * (ct + u * W) + lc;
      jc[u] = j >= i0 && j < n ? j : n;  // n: no such column (every row test fails)
    }
  };
  cplx<double> x[RU][NCT], xn[RU][NCT];
  auto load = [&](int rt, cplx<double>(&o)[RU][NCT]) {
#pragma unroll
    for (int k = 0; k < RU; ++k)
#pragma unroll
      for (int u = 0; u < NCT; ++u) {
        const int r = 16 * (rt + k) + lr;
        o[k][u] = mk<double>(0, 0);
        if (r < n && r >= jc[u]) o[k][u] = A[r + (size_t)jc[u] * ld];
      }
  };
  // the first elements of the pass are in flight during the prologue
  tiles();
  load(ct >> 2, x);

  // ---- w_{c-1}, column c, its reflector; a thread holds rows tid + NT q ----------------
  cplx<double> a[RPT], v[P ? P : 1][RPT], w[P ? P : 1][RPT], y[RPT], tau = mk<double>(0, 0);
  bool live[RPT];
#pragma unroll
  for (int q = 0; q < RPT; ++q) {
    const int i = tid + NT * q;
    live[q] = i >= c && i < n;
    a[q] = y[q] = mk<double>(0, 0);
#pragma unroll
    for (int k = 0; k < (P ? P : 1); ++k) v[k][q] = w[k][q] = mk<double>(0, 0);
    if (live[q]) {
      if (!hand) a[q] = A[i + (size_t)c * ld];  // (at the handover its owner is storing to it)
#pragma unroll
      for (int k = 0; k < P; ++k) {
        v[k][q] = tw.v[slot(c - 1 - k) + i];
        if (k > 0) w[k][q] = tw.w[slot(c - 1 - k) + i];
      }
      if (P > 0) {
        y[q] = tw.col[(j2 + prv) * nmax + i];
        for (int k = 0; k < G; ++k) y[q] = y[q] + tw.row[((j2 + prv) * TRI_GMAX + k) * nmax + i];
      }
      if (i == c) {
        sh.yc = y[q];
#pragma unroll
        for (int k = 1; k < P; ++k) sh.vc[k] = v[k][q], sh.wc[k] = w[k][q];
      }
    }
  }
  if (P > 0) {
    tau = tw.tau[j2 + prv];
    double pr = 0, pi = 0;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      w[0][q] = tau * y[q];
      const cplx<double> dt = cmul_conj_a(w[0][q], v[0][q]);
      pr += dt.re;
      pi += dt.im;
    }
    tri_sum2<NW>(pr, pi, sh.red[0]);
    const cplx<double> alpha2 = tau * mk<double>(-0.5 * pr, -0.5 * pi);
    const cplx<double> wc = tau * sh.yc + alpha2;  // row c, where v_{c-1} is 1
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      w[0][q] = w[0][q] + alpha2 * v[0][q];
      if (!live[q]) continue;
#pragma unroll
      for (int k = P - 1; k > 0; --k) a[q] = a[q] - (v[k][q] * conj(sh.wc[k]) + w[k][q] * conj(sh.vc[k]));
      a[q] = a[q] - (v[0][q] * conj(wc) + w[0][q]);
    }
  }
  double part = 0, unused = 0;
#pragma unroll
  for (int q = 0; q < RPT; ++q) {
    const int i = tid + NT * q;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      sh.v[k][i] = v[k][q];
      sh.w[k][i] = w[k][q];
    }
    if (i == c + 1) sh.alpha = a[q];
    if (live[q] && i >= c + 2) part += abs2(a[q]);
  }
  tri_sum2<NW>(part, unused, sh.red[1]);
  if (g == 0) {
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
      const int i = tid + NT * q;
      if (!live[q]) continue;
      if (P > 0) {
        tw.w[slot(c - 1) + i] = w[0][q];
        if (i > c)
          A[i + (size_t)(c - 1) * ld] = v[0][q];
        else
          A[(c - 1) + (size_t)(c - 1) * ld] = tau;  // the diagonal slot keeps tau
      }
      if (i == c && !hand) tw.de[((size_t)job * nmax + c) * 2] = a[q].re;
    }
  }
  const cplx<double> alpha = sh.alpha;
  cplx<double> tn, scal;
  double beta;
  if (part == 0.0 && alpha.im == 0.0) {
    tn = mk<double>(0, 0);
    beta = alpha.re;
    scal = mk<double>(0, 0);
  } else {
    const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + part);
    beta = alpha.re >= 0.0 ? -nrm : nrm;
    tn = mk<double>((beta - alpha.re) / beta, -alpha.im / beta);
    scal = crecip(mk<double>(alpha.re - beta, alpha.im));
  }
#pragma unroll
  for (int q = 0; q < RPT; ++q) {
    const int i = tid + NT * q;
    cplx<double> vn = mk<double>(i == c + 1 ? 1.0 : 0.0, 0);
    if (live[q] && i >= c + 2) vn = a[q] * scal;
    sh.vn[i] = vn;
    if (g == 0) {
      if (live[q] && i > c) tw.v[slot(c) + i] = vn;
      if (i == c) {
        tw.tau[j2 + cur] = tn;
        tw.de[((size_t)job * nmax + c) * 2 + 1] = beta;
      }
    }
  }
  // ---- pass over this wavefront's column tiles ------------------------------------------
  for (int r = (i0 & ~63) + lane; r < n; r += 64) sh.xw[wave][r] = mk<double>(0, 0);
  __syncthreads();
  bool first = true;
  for (; ct < ct_end; ct += NCT * W) {
    if (!first) {
      tiles();
      load(ct >> 2, x);
    }
    first = false;
    cplx<double> cv[P ? P : 1][NCT], cw[P ? P : 1][NCT], cn[NCT], cs[NCT];
#pragma unroll
    for (int u = 0; u < NCT; ++u) {
      const int jj = min(jc[u], TRI_N - 1);
#pragma unroll
      for (int q = 0; q < P; ++q) {
        cv[q][u] = conj(sh.v[q][jj]);
        cw[q][u] = conj(sh.w[q][jj]);
      }
      cn[u] = sh.vn[jj];
      cs[u] = mk<double>(0, 0);
    }
    for (int rt = ct >> 2; rt < rt_end; rt += RU) {
      if (rt + RU < rt_end) load(rt + RU, xn);
#pragma unroll
      for (int k = 0; k < RU; ++k) {
        const int r = 16 * (rt + k) + lr;
        if (16 * (rt + k) >= n) break;  // uniform
        const int rr = min(r, TRI_N - 1);
        const cplx<double> ni = sh.vn[rr];
        cplx<double> vi[P ? P : 1], wi[P ? P : 1];
#pragma unroll
        for (int q = 0; q < P; ++q) vi[q] = sh.v[q][rr], wi[q] = sh.w[q][rr];
        cplx<double> acc = mk<double>(0, 0);
#pragma unroll
        for (int u = 0; u < NCT; ++u) {
          if (r < n && r >= jc[u]) {
            cplx<double> e = x[k][u];
#pragma unroll
            for (int q = P - 1; q >= 0; --q) e = sub_mul2(e, vi[q], cw[q][u], wi[q], cv[q][u]);
            if (keep) A[r + (size_t)jc[u] * ld] = e;
            acc = add_mul(acc, e, cn[u]);
            if (r > jc[u]) cs[u] = add_mul_conj(cs[u], e, ni);
          }
        }
        const double t = rows_total(acc.re, acc.im);
        if (!(lc & 1) && r < n) {
          double* o = reinterpret_cast<double*>(&sh.xw[wave][r]) + (lc >> 1);
          *o += t;
        }
      }
#pragma unroll
      for (int k = 0; k < RU; ++k)
#pragma unroll
        for (int u = 0; u < NCT; ++u) x[k][u] = xn[k][u];
    }
#pragma unroll
    for (int u = 0; u < NCT; ++u) {
      const cplx<double> s = mk<double>(sum16(cs[u].re), sum16(cs[u].im));
      if (lr == 0 && jc[u] < n) tw.col[(j2 + cur) * nmax + jc[u]] = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < RPT; ++q) {
    const int i = tid + NT * q;
    if (i < i0 || i >= n) continue;
    cplx<double> s = sh.xw[0][i];
#pragma unroll
    for (int k = 1; k < NW; ++k) s = s + sh.xw[k][i];
    tw.row[((j2 + cur) * TRI_GMAX + g) * nmax + i] = s;
  }
}

// The trailing matrix from column n - TRI_TAIL on (all of a smaller one).  Workgroup per job.
__global__ __launch_bounds__(EigCfg<TRI_TAIL>::NT) void split_tail_kernel(EigParams<double> p, TriWork tw) {
  EigShared<double, TRI_TAIL>& sh = eig_sh<double, TRI_TAIL, 1>;
  const int job = blockIdx.x, sid = p.order[job], n = p.n_red[sid], ld = p.ldz;
  if (n <= 0 || p.info[sid] != 0) return;
  const int c0 = max(0, n - TRI_TAIL), m = n - c0;
  cplx<double>* A = p.z_out + (size_t)sid * p.stride_z + c0 + (size_t)c0 * ld;
  if (m > 1) {
    tridiag_resident<TRI_TAIL, 1>(m, A, ld, nullptr);
  } else {
    if (threadIdx.x == 0) {
      sh.de[0].x = A[0].re;
      sh.de[0].y = 0;
      A[0] = mk<double>(0, 0);
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < m; i += EigCfg<TRI_TAIL>::NT) {
    tw.de[((size_t)job * p.nmax + c0 + i) * 2] = sh.de[i].x;
    tw.de[((size_t)job * p.nmax + c0 + i) * 2 + 1] = sh.de[i].y;
  }
}

// Eigenpairs of the tridiagonal (dc_phase, scratch ws_a), ascending order: eigenvalues to
// d_out, the column order to perm.  Workgroup per job.
template <int NMAX>
__global__ __launch_bounds__(EigCfg<NMAX>::NT) void split_dc_kernel(EigParams<double> p, TriWork tw) {
  EigShared<double, NMAX>& sh = eig_sh<double, NMAX, 1>;
  constexpr int NT_ = EigCfg<NMAX>::NT;
  const int job = blockIdx.x, sid = p.order[job], n = p.n_red[sid], tid = threadIdx.x;
  if (n <= 0 || p.info[sid] != 0) return;
  for (int i = tid; i < n; i += NT_) {
    sh.de[i].x = tw.de[((size_t)job * p.nmax + i) * 2];
    sh.de[i].y = tw.de[((size_t)job * p.nmax + i) * 2 + 1];
  }
  __syncthreads();
  dc_phase<double, NMAX, 1>(n, p.ws_z + (size_t)job * p.ws_stride, p.ws_ld,
                         reinterpret_cast<double*>(p.ws_a + (size_t)job * p.ws_stride), nullptr);
  rank_order<double, NMAX>(n, sh);
  for (int j = tid; j < p.nmax; j += NT_) {
    p.d_out[(size_t)sid * p.stride_d + j] = j < n ? sh.de[sh.perm[j]].x : 0.0;
    if (j < n) tw.perm[(size_t)job * p.nmax + j] = sh.perm[j];
  }
}

// --------------------------------------------------------------------------------------
// Back-transform ws_a = Q Z[:, perm] in compact-WY blocks of 16 reflectors on
// v_mfma_f64_16x16x4f64 (the scheme and layouts of back_transform_mfma), over workgroups of
// 16 eigenvector columns: four wavefronts take alternate 16-row blocks of them (in registers
// for the whole phase) and exchange one partial product per reflector block through LDS.  The
// reflectors come straight from A (they are read by every column group of the sample, all
// on one XCD); an MFMA takes 64 cycles, so their loads cost a CU 16 bytes per cycle.
// --------------------------------------------------------------------------------------
// v_{cs + q} at row i (1 at its unit entry, 0 above it and for cs + q < 0)
__device__ __forceinline__ cplx<double> wy_elem(const cplx<double>* A, int ld, int n, int col, int i) {
  if (col < 0 || i <= col || i >= n) return mk<double>(0, 0);
  return i == col + 1 ? mk<double>(1, 0) : A[i + (size_t)col * ld];
}

// T factor of one block of reflectors into the strict upper triangle of A: entry (p, q),
// p <= q, at A[cs + p, cs + q + 1].
__global__ __launch_bounds__(256) void split_tfac_kernel(EigParams<double> p) {
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  __shared__ double red[4][64][8];
  __shared__ cplx<double> gm[16][16], t[16][16], tau[16];
  const int b = blockIdx.x, sid = p.order[blockIdx.y], n = p.n_red[sid];
  const int nblk = (n - 1 + 15) / 16;
  if (b >= nblk || p.info[sid] != 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lk = lane >> 4;
  cplx<double>* A = p.z_out + (size_t)sid * p.stride_z;
  const int ld = p.ldz, cs = n - 2 - 16 * b - 15;
  const int rb0 = (max(cs, 0) + 1) / 16, rb1 = (n + 15) / 16;
  f64x4 gr = {0, 0, 0, 0}, gi = {0, 0, 0, 0};
  for (int rb = rb0 + wave; rb < rb1; rb += 4)
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const cplx<double> v = wy_elem(A, ld, n, cs + lr, rb * 16 + 4 * s4 + lk);
      gr = __builtin_amdgcn_mfma_f64_16x16x4f64(v.re, v.re, gr, 0, 0, 0);
      gr = __builtin_amdgcn_mfma_f64_16x16x4f64(v.im, v.im, gr, 0, 0, 0);
      gi = __builtin_amdgcn_mfma_f64_16x16x4f64(v.re, v.im, gi, 0, 0, 0);
      gi = __builtin_amdgcn_mfma_f64_16x16x4f64(-v.im, v.re, gi, 0, 0, 0);
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    red[wave][lane][r] = gr[r];
    red[wave][lane][4 + r] = gi[r];
  }
  if (tid < 16) tau[tid] = cs + tid >= 0 ? A[(cs + tid) + (size_t)(cs + tid) * ld] : mk<double>(0, 0);
  __syncthreads();
  if (wave != 0) return;  // no workgroup barrier below
#pragma unroll
  for (int r = 0; r < 4; ++r)
    gm[lk + 4 * r][lr] = mk<double>(
        (red[0][lane][r] + red[1][lane][r]) + (red[2][lane][r] + red[3][lane][r]),
        (red[0][lane][4 + r] + red[1][lane][4 + r]) + (red[2][lane][4 + r] + red[3][lane][4 + r]));
  wave_sync();
  for (int i = 0; i < 16; ++i) {
    if (lane < 16) {
      cplx<double> val = mk<double>(0, 0);
      if (lane == i) {
        val = tau[i];
      } else if (lane < i) {
        cplx<double> acc = mk<double>(0, 0);
        for (int q = lane; q < i; ++q) acc = acc + t[lane][q] * gm[q][i];
        val = mk<double>(0, 0) - tau[i] * acc;
      }
      t[lane][i] = val;
    }
    wave_sync();
  }
  for (int e = lane; e < 256; e += 64) {
    const int pr = e / 16, q = e % 16;
    if (pr <= q && cs + pr >= 0) A[(cs + pr) + (size_t)(cs + q + 1) * ld] = t[pr][q];
  }
}

template <int NMAX>
__global__ __launch_bounds__(256) void split_bt_kernel(EigParams<double> p, TriWork tw, int groups) {
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  constexpr int NWV = 4, RBW = NMAX / 16 / NWV;
  __shared__ double red[2][NWV][64][8];
  const SplitUnit u = split_unit(groups, p.n_jobs);
  if (u.job < 0) return;
  const int sid = p.order[u.job], n = p.n_red[sid];
  if (16 * u.unit >= n || p.info[sid] != 0) return;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ld = p.ldz;
  const cplx<double>* A = p.z_out + (size_t)sid * p.stride_z;
  const double* Z = p.ws_z + (size_t)u.job * p.ws_stride;
  cplx<double>* X = p.ws_a + (size_t)u.job * p.ws_stride;
  const int col = 16 * u.unit + lr;
  const int pc = col < n ? tw.perm[(size_t)u.job * p.nmax + col] : 0;
  const f64x4 z4 = {0, 0, 0, 0};
  f64x4 xr[RBW], xi[RBW];  // row block wave + 4 t, register r: row lk + 4 r
#pragma unroll
  for (int t = 0; t < RBW; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (wave + NWV * t) * 16 + lk + 4 * r;
      xr[t][r] = row < n && col < n ? Z[row + (size_t)pc * ld] : 0.0;
    }
    xi[t] = z4;
  }
  const int nblk = (n - 1 + 15) / 16;
  for (int b = 0; b < nblk; ++b) {
    const int cs = n - 2 - 16 * b - 15, rb0 = (max(cs, 0) + 1) / 16;
    f64x4 wr = z4, wi = z4;
#pragma unroll
    for (int t = 0; t < RBW; ++t) {
      const int rb = wave + NWV * t;
      if (rb < rb0 || 16 * rb >= n) continue;  // uniform over the wavefront
      cplx<double> v[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) v[s4] = wy_elem(A, ld, n, cs + lr, rb * 16 + 4 * s4 + lk);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        wr = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s4].re, xr[t][s4], wr, 0, 0, 0);
        wi = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s4].re, xi[t][s4], wi, 0, 0, 0);
        wr = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s4].im, xi[t][s4], wr, 0, 0, 0);
        wi = __builtin_amdgcn_mfma_f64_16x16x4f64(-v[s4].im, xr[t][s4], wi, 0, 0, 0);
      }
    }
    cplx<double> tv[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const int q = 4 * s4 + lk;
      tv[s4] = lr <= q && cs + lr >= 0 ? A[(cs + lr) + (size_t)(cs + q + 1) * ld] : mk<double>(0, 0);
    }
    double(*rd)[64][8] = red[b & 1];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      rd[wave][lane][r] = wr[r];
      rd[wave][lane][4 + r] = wi[r];
    }
    // one barrier per block: the other buffer is next written after the next barrier
    __syncthreads();
    f64x4 w1r, w1i, w2r = z4, w2i = z4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      w1r[r] = (rd[0][lane][r] + rd[1][lane][r]) + (rd[2][lane][r] + rd[3][lane][r]);
      w1i[r] = (rd[0][lane][4 + r] + rd[1][lane][4 + r]) + (rd[2][lane][4 + r] + rd[3][lane][4 + r]);
    }
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      w2r = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[s4].re, w1r[s4], w2r, 0, 0, 0);
      w2i = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[s4].re, w1i[s4], w2i, 0, 0, 0);
      w2r = __builtin_amdgcn_mfma_f64_16x16x4f64(-tv[s4].im, w1i[s4], w2r, 0, 0, 0);
      w2i = __builtin_amdgcn_mfma_f64_16x16x4f64(tv[s4].im, w1r[s4], w2i, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < RBW; ++t) {
      const int rb = wave + NWV * t;
      if (rb < rb0 || 16 * rb >= n) continue;  // uniform over the wavefront
      cplx<double> v[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) v[s4] = wy_elem(A, ld, n, cs + 4 * s4 + lk, rb * 16 + lr);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        xr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-v[s4].re, w2r[s4], xr[t], 0, 0, 0);
        xi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-v[s4].re, w2i[s4], xi[t], 0, 0, 0);
        xr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[s4].im, w2i[s4], xr[t], 0, 0, 0);
        xi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-v[s4].im, w2r[s4], xi[t], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < RBW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (wave + NWV * t) * 16 + lk + 4 * r;
      if (row < n && col < n) X[row + (size_t)col * ld] = mk<double>(xr[t][r], xi[t][r]);
    }
}
