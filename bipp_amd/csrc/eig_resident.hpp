// Householder tridiagonalisation with the trailing matrix in registers (float64, at most 256
// beams): the phase of eig_kernel that takes the place of tridiag_phase there.
//
// tridiag_phase reads and writes the trailing lower triangle once per column; with every CU
// at work that is the last-level cache's rate (89 MB per 256-beam sample, 5.9 TB/s over the
// chip), and a sample alone waits for each pass's loads instead.  Here the lower triangle is
// dealt to the workgroup's registers in tiles of 16 rows x 4 columns (a lane holds row
// 16 rt + lane % 16 of column 4 ct + lane / 16; wavefront w holds column tiles ct = w + NW u).
// Up to 128 beams all of it fits (40 or 144 registers per lane); at 256 beams the 160 last
// columns (120 registers) and 32 more in LDS (96 KB) stay for the whole phase and the first 64
// are streamed while they live, a sixth of the traffic.  The matrix is aligned with the last index (index g = i + NMAX -
// n), so a smaller sample streams less or nothing.
//
// The tiles also cut the work beside the products: a column's sum over its rows takes four
// lane moves for four columns at once, and a row tile's operands are read from LDS once for
// all columns of the wavefront.
// Measured, per sample with every CU at work: 256 beams 4.42 to 1.98 ms, 218 on average 2.95 to
// 1.38 ms; one sample alone: 96 beams 0.67 to 0.32 ms, 37 beams 0.155 to 0.081 ms.  (32 columns
// in LDS instead of streamed: 1.98 against 2.10 ms at 256 beams.)
#pragma once

template <int NMAX>
struct TriRes {
  static constexpr int NW = EigCfg<NMAX>::NW, RT = NMAX / 16, U = NMAX / 4 / NW;
  // column tiles per wavefront: [0, US) streamed, [US, U0) in LDS, [U0, U) in registers
  static constexpr int US = NMAX >= 256 ? 2 : 0, U0 = NMAX >= 256 ? 3 : 0;
  // first row tile at or below the diagonal of the wavefronts' u-th column tiles
  static constexpr int first(int u) { return NW * u / 4; }
  static constexpr int base(int u) {
    int b = 0;
    for (int q = U0; q < u; ++q) b += RT - first(q);
    return b;
  }
  static constexpr int SLOTS = base(U);
  static_assert(U0 == US || (U0 == US + 1 && (RT - first(US)) * 64 * NW == tri_lds_elems<double>(NMAX)),
                "one column tile per wavefront in LDS");
};
enum { TRI_REG = 0, TRI_LDS = 1, TRI_STREAM = 2 };  // where a sweep's tiles are

// x - (a b + c d), acc + x y and acc + conj(x) y as chains of fused multiply-adds (8, 4 and 4;
// the operators give half as many more instructions)
__device__ __forceinline__ cplx<double> sub_mul2(cplx<double> x, cplx<double> a, cplx<double> b,
                                                 cplx<double> c, cplx<double> d) {
  return mk<double>(fma(-a.re, b.re, fma(a.im, b.im, fma(-c.re, d.re, fma(c.im, d.im, x.re)))),
                    fma(-a.re, b.im, fma(-a.im, b.re, fma(-c.re, d.im, fma(-c.im, d.re, x.im)))));
}
__device__ __forceinline__ cplx<double> add_mul(cplx<double> acc, cplx<double> x, cplx<double> y) {
  return mk<double>(fma(x.re, y.re, fma(-x.im, y.im, acc.re)),
                    fma(x.re, y.im, fma(x.im, y.re, acc.im)));
}
__device__ __forceinline__ cplx<double> add_mul_conj(cplx<double> acc, cplx<double> x, cplx<double> y) {
  return mk<double>(fma(x.re, y.re, fma(x.im, y.im, acc.re)),
                    fma(x.re, y.im, fma(-x.im, y.re, acc.im)));
}

// One sweep over column tiles [UA, UB) of every wavefront: the pending update A -= v w^H + w v^H,
// then their part of A vn (row sums added to sh.xw[wave], column sums to sh.xc) and, where it
// is among them, column g0 of the updated matrix into sh.cx.  The tiles are X (TRI_REG), sh.tt
// (TRI_LDS) or come through M, the next row tile loaded during the current one (TRI_STREAM).
template <int NMAX, int UA, int UB, int WHERE>
__device__ __forceinline__ void tri_sweep(int g0, int off, const BufMat<double>& M,
                                          cplx<double> (&X)[TriRes<NMAX>::SLOTS],
                                          const cplx<double>* v, const cplx<double>* vn,
                                          EigShared<double, NMAX>& sh) {
  using T = TriRes<NMAX>;
  constexpr int N = UB - UA;
  constexpr bool STREAM = WHERE == TRI_STREAM;
  const int lane = threadIdx.x & 63, lr = lane & 15, lc = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (4 * (wave + T::NW * (UB - 1)) + 3 < g0) return;  // the last tile is dead: uniform
  int j[N];
  unsigned o0[N];  // buffer offset of row tile 0 (STREAM); past the end for a dead column
  bool act[N], dump[N];
  cplx<double> cv[N], cw[N], cn[N], cs[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int ct = wave + T::NW * (UA + k);
    j[k] = 4 * ct + lc;
    act[k] = 4 * ct + 3 >= g0;
    dump[k] = ct == (g0 >> 2);
    if (STREAM) o0[k] = j[k] >= g0 ? static_cast<unsigned>(16 * (lr - off + (j[k] - off) * M.ld)) : BufMat<double>::OOB;
    cv[k] = conj(v[j[k]]);
    cw[k] = conj(sh.w[j[k]]);
    cn[k] = vn[j[k]];
    cs[k] = mk<double>(0, 0);
  }
  // rows above the diagonal can only be in a column tile's first two row tiles
  auto diag = [](int k, int rt) { return rt <= T::first(UA + k) + 1; };
  auto at = [&](int k, int rt) __attribute__((always_inline)) {
    const unsigned o = o0[k] + 256u * rt;
    return diag(k, rt) && 16 * rt + lr < j[k] ? BufMat<double>::OOB : o;
  };
  constexpr int RT0 = T::first(UA) & ~1;
  cplx<double> cur[N], nxt[N];
  auto load = [&](int rt) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (rt >= T::first(UA + k)) nxt[k] = M.load(at(k, rt));
  };
  bool fetched = false;  // STREAM: the next row tile is in nxt
#pragma unroll
  for (int rp = RT0; rp < T::RT; rp += 2) {
    if (16 * rp + 31 < g0) continue;  // uniform
    cplx<double> acc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int rt = rp + h, r = 16 * rt + lr;
      if (STREAM) {
        if (!fetched) load(rt);
        fetched = true;
#pragma unroll
        for (int k = 0; k < N; ++k) cur[k] = nxt[k];
        if (rt + 1 < T::RT) load(rt + 1);
      }
      const cplx<double> vi = v[r], wi = sh.w[r], ni = vn[r];
      acc[h] = mk<double>(0, 0);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (rt < T::first(UA + k)) continue;  // static
        if (!act[k]) continue;                // uniform
        cplx<double>& xs =
            STREAM ? cur[k]
                   : (WHERE == TRI_LDS ? sh.tt[((rt - T::first(UA)) * T::NW + wave) * 64 + lane]
                                       : X[WHERE != TRI_REG ? 0 : T::base(UA + k) + rt - T::first(UA + k)]);
        cplx<double> x = sub_mul2(xs, vi, cw[k], wi, cv[k]);
        if (STREAM)
          M.store(at(k, rt), x);
        else
          xs = x;
        if (dump[k]) {
          if (lc == (g0 & 3)) sh.cx[r] = x;
        }
        // columns before g0 have vn = 0 and their column sums are not read
        cplx<double> xo = x;
        if (diag(k, rt)) {
          x = r >= j[k] ? x : mk<double>(0, 0);
          xo = r > j[k] ? x : mk<double>(0, 0);
        }
        acc[h] = add_mul(acc[h], x, cn[k]);
        cs[k] = add_mul_conj(cs[k], xo, ni);
      }
    }
    // lane row lc holds (Re, Im)[lc / 2] of row tile rp + lc % 2
    double* o = reinterpret_cast<double*>(&sh.xw[wave][16 * (rp + (lc & 1)) + lr]) + (lc >> 1);
    *o += rows_total2(acc[0], acc[1]);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    if (!act[k]) continue;
    const cplx<double> s = mk<double>(sum16(cs[k].re), sum16(cs[k].im));
    if (lr == 0) sh.xc[j[k]] = s;
  }
}

// d and e into sh.de, the reflectors below the subdiagonal of A with tau in the diagonal slots
// (0 for the last column), as tridiag_phase leaves them; n >= 2.  Out of line: its registers
// are allocated apart from the other phases.
template <int NMAX, int USE = 0>
__device__ __noinline__ void tridiag_resident(int n, cplx<double>* __restrict__ A, int ld,
                                              unsigned long long* prof) {
  using T = TriRes<NMAX>;
  n = uniform(n);
  ld = uniform(ld);
  A = uniform(A);
  prof = uniform(prof);
  EigShared<double, NMAX>& sh = eig_sh<double, NMAX, USE>;
  static_assert(EigCfg<NMAX>::NT >= NMAX, "one row per thread");
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lc = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const BufMat<double> M(A, ld, n);
  const int off = NMAX - n;
  WgTeam tm{tid, prof};  // step timing: 0 w, column update and reflector, 1 pass
  tm.mark(-1);
  cplx<double> X[T::SLOTS];
#pragma unroll
  for (int u = T::U0; u < T::U; ++u)
#pragma unroll
    for (int rt = T::first(u); rt < T::RT; ++rt) {
      const int r = 16 * rt + lr, j = 4 * (wave + T::NW * u) + lc;
      X[T::base(u) + rt - T::first(u)] =
          M.load(r >= j && j >= off ? M.off(r - off, j - off) : BufMat<double>::OOB);
    }
  if constexpr (T::U0 > T::US)
    for (int rt = T::first(T::US); rt < T::RT; ++rt) {
      const int r = 16 * rt + lr, j = 4 * (wave + T::NW * T::US) + lc;
      sh.tt[((rt - T::first(T::US)) * T::NW + wave) * 64 + lane] =
          M.load(r >= j && j >= off ? M.off(r - off, j - off) : BufMat<double>::OOB);
    }
  cplx<double>* v = sh.v;     // reflector of the pending update
  cplx<double>* vn = sh.vn;   // reflector of the current column
  const int g = tid;          // this thread's row
  if (g < NMAX) {
    sh.cx[g] = M.load(g >= off ? M.off(g - off, 0) : BufMat<double>::OOB);
    v[g] = mk<double>(0, 0);
    sh.w[g] = mk<double>(0, 0);
  }
  cplx<double> tau = mk<double>(0, 0);
  __syncthreads();
  for (int c = 0; c < n; ++c) {
    const int gc = off + c;
    const bool live = g >= gc && g < NMAX;
    // ---- w_{c-1} from y = A v_{c-1}, column c with its update, reflector c ----------------
    cplx<double> a = mk<double>(0, 0), vi = a, w = a;
    if (live) a = sh.cx[g];
    if (c > 0) {
      cplx<double> y = mk<double>(0, 0);
      if (live) {
        vi = v[g];
        y = sh.xc[g];
#pragma unroll
        for (int q = 0; q < T::NW; ++q) y = y + sh.xw[q][g];
      }
      if (g == gc) sh.scal[2] = y.re, sh.scal[3] = y.im;
      const cplx<double> x = tau * y;
      const cplx<double> dt = cmul_conj_a(x, vi);
      double pr = dt.re, pi = dt.im;
      block_sum2(pr, pi, sh, 0);
      const cplx<double> alpha2 = tau * mk<double>(-0.5 * pr, -0.5 * pi);
      w = x + alpha2 * vi;
      const cplx<double> wc = tau * mk<double>(sh.scal[2], sh.scal[3]) + alpha2;  // row c: v is 1
      if (live) {
        sh.w[g] = w;
        a = a - (vi * conj(wc) + w);
      }
    }
    if (g == gc) sh.de[c].x = a.re;
    if (c == n - 1) break;
    if (g == gc + 1) sh.scal[0] = a.re, sh.scal[1] = a.im;
    double part = live && g >= gc + 2 ? abs2(a) : 0.0, unused = 0;
    block_sum2(part, unused, sh, 1);
    const cplx<double> alpha = mk<double>(sh.scal[0], sh.scal[1]);
    cplx<double> scal;
    double beta;
    if (part == 0.0 && alpha.im == 0.0) {
      tau = mk<double>(0, 0);
      beta = alpha.re;
      scal = mk<double>(0, 0);
    } else {
      const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + part);
      beta = alpha.re >= 0.0 ? -nrm : nrm;
      tau = mk<double>((beta - alpha.re) / beta, -alpha.im / beta);
      scal = crecip(mk<double>(alpha.re - beta, alpha.im));
    }
    if (g < NMAX) {
      cplx<double> q = mk<double>(g == gc + 1 ? 1.0 : 0.0, 0);
      if (live && g >= gc + 2) {
        q = a * scal;
        M.store(M.off(g - off, c), q);
      }
      vn[g] = q;
    }
    if (g == gc) {
      M.store(M.off(c, c), tau);  // the diagonal slot keeps tau
      sh.de[c].y = beta;
    }
    const int g0 = gc + 1;
    for (int r = (g0 & ~31) + lane; r < NMAX; r += 64) sh.xw[wave][r] = mk<double>(0, 0);
    __syncthreads();
    tm.mark(0);
    // ---- pass: pending update of c - 1, y = A v_c, column c + 1 into sh.cx -----------------
    // (at 256 beams in three sweeps, which share the registers beside the resident tiles)
    if constexpr (T::U0 > 0) {
      tri_sweep<NMAX, 0, T::US, TRI_STREAM>(g0, off, M, X, v, vn, sh);
      tri_sweep<NMAX, T::US, T::U0, TRI_LDS>(g0, off, M, X, v, vn, sh);
      tri_sweep<NMAX, T::U0, T::U0 + 2, TRI_REG>(g0, off, M, X, v, vn, sh);
      tri_sweep<NMAX, T::U0 + 2, T::U, TRI_REG>(g0, off, M, X, v, vn, sh);
    } else {
      constexpr int H = T::U / 2;
      tri_sweep<NMAX, 0, H, TRI_REG>(g0, off, M, X, v, vn, sh);
      tri_sweep<NMAX, H, T::U, TRI_REG>(g0, off, M, X, v, vn, sh);
    }
    __syncthreads();
    tm.mark(1);
    cplx<double>* t = v;
    v = vn;
    vn = t;
  }
  if (tid == 0) {
    M.store(M.off(n - 1, n - 1), mk<double>(0, 0));  // no reflector for the last column
    sh.de[n - 1].y = 0;
  }
  __syncthreads();
}
