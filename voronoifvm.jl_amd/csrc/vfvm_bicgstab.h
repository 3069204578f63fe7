// Kernels of the single-system BiCGStab (included by vfvm_linalg.hip, inside its namespace).
//
// The reductions have no kernels of their own: a reducing kernel writes one partial per
// block, and every block of the next kernel that needs the scalars sums those partials in
// the same order and runs the stage on a copy of the solver state (fold_state); block 0
// stores the new state.  The state moves through three slots in an iteration, each kernel
// reading one and writing another, so no block can see a state that another one is writing:
//   slot 0 -> (rho, beta)  -> slot 1 -> (alpha) -> slot 2 -> (omega) -> slot 0
// Small systems are bound by the chain of launches (2 to 5 us each whatever the size), so
// folding the four finalize launches of an iteration away and fusing the vector updates into
// the products is what their time follows: an iteration has 3 launches (point Jacobi), 5 (block
// Jacobi) or 7 (two-colour ILU(0)) instead of 8, 10 and 14.  Measured over whole solves, before
// and after: 33^2 rows with point Jacobi 5.3 and 2.9 ms, 3 x 129^2 with block Jacobi 133 and
// 63 ms, 101^2 with ILU(0) 15.8 and 8.1 ms; 129^3 with ILU(0) in FP32, where memory counts
// (ILU and product 128 us, now 79), 63.4 and 42 ms.
//
// A folding kernel starts with two chains of dependent loads: partials, sums, scalars; and row,
// columns, gathers.  Both are issued before either is waited for, and sums within a wave use
// register moves: 3.5 to 4.2 us a kernel where loads after the scalars took 4.4 to 5 us.

enum { SLOT_RHO = 0, SLOT_BETA = 1, SLOT_ALPHA = 2 };

// Totals of the previous reduction (NR sums of np partials) and the stage on them.  begin()
// issues the loads, so that a kernel's own loads can follow before finish() waits; finish()
// returns the new state, which block 0 stores to `out`.  A finished solve's state is passed on
// unchanged.
template <int STAGE, int NR>
struct Fold {
  static constexpr int WORDS = sizeof(KState) / 4;
  double a[NR];
  uint32_t word;  // thread t holds word t of the state
  __device__ __forceinline__ void begin(const double *__restrict__ part, int np, const KState *__restrict__ in) {
    const int b = threadIdx.x;
#pragma unroll
    for (int q = 0; q < NR; q++) a[q] = b < np ? part[(size_t)q * np + b] : 0.0;
    if (b < WORDS) word = reinterpret_cast<const uint32_t *>(in)[b];
  }
  __device__ __forceinline__ const KState &finish(const double *__restrict__ part, int np, KState *__restrict__ out) {
    __shared__ double red[NR][VB / 64];
    __shared__ KState ks;
    if (threadIdx.x < WORDS) reinterpret_cast<uint32_t *>(&ks)[threadIdx.x] = word;
#pragma unroll 4
    for (int b = threadIdx.x + VB; b < np; b += VB)
#pragma unroll
      for (int q = 0; q < NR; q++) a[q] += part[(size_t)q * np + b];
#pragma unroll
    for (int q = 0; q < NR; q++) {
      a[q] = wave_sum(a[q]);
      if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = a[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double tot[NR];
#pragma unroll
      for (int q = 0; q < NR; q++) {
        tot[q] = 0.0;
#pragma unroll
        for (int w = 0; w < VB / 64; w++) tot[q] += red[q][w];
      }
      if (!ks.done && !(STAGE == STAGE_OMEGA && ks.half)) run_stage<STAGE>(&ks, tot);
    }
    __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x < WORDS)
      reinterpret_cast<uint32_t *>(out)[threadIdx.x] = reinterpret_cast<const uint32_t *>(&ks)[threadIdx.x];
    return ks;
  }
};

template <int NR>
__device__ __forceinline__ void write_partials_at(const double (&v)[NR], double *part, int np, int at) {
  __shared__ double red[NR][VB / 64];
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const double w = wave_sum(v[q]);
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = w;
  }
  __syncthreads();
  if (threadIdx.x < NR) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < VB / 64; w++) t += red[threadIdx.x][w];
    part[(size_t)threadIdx.x * np + at] = t;
  }
}

// s = r - alpha v, rounded alike wherever it is formed
template <class V>
__device__ __forceinline__ V half_step(V r, V v, double alpha) {
  return (V)__builtin_fma(-alpha, (double)v, (double)r);
}
// p = r + beta (p - omega v)
template <class V>
__device__ __forceinline__ V direction(V r, V p, V v, double beta, double omega) {
  return (V)((double)r + beta * ((double)p - omega * (double)v));
}

// z = B y of a node (block Jacobi)
template <int NS, class V>
__device__ __forceinline__ void node_solve(const double (&B)[NS * NS], const V (&y)[NS], V *__restrict__ z) {
#pragma unroll
  for (int i = 0; i < NS; i++) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < NS; j++) acc += B[i * NS + j] * (double)y[j];
    z[i] = (V)acc;
  }
}

// the state after the last queued iteration, to pinned host memory (one block)
__global__ void __launch_bounds__(VB) k_bicg_report(const double *__restrict__ part, int np, const KState *in,
                                                    KState *out) {
  Fold<STAGE_XR, 2> f;
  f.begin(part, np, in);
  f.finish(part, np, out);
}

// The loads of a thread's first row are issued before the scalars are known, so that they and
// the partial sums share one memory latency; later rows (large systems) load at the loop's end.
// stage (INIT or XR), then p = r + beta (p - omega v); NS > 0: also ph = Binv p per node of NS
// rows (n counts nodes then)
template <class V, int STAGE, int NS>
__global__ void __launch_bounds__(VB) k_bicg_p(int64_t n, const V *__restrict__ r, V *__restrict__ p,
                                               const V *__restrict__ v, const double *__restrict__ binv,
                                               V *__restrict__ ph, const double *__restrict__ part, int np,
                                               const KState *in, KState *out) {
  constexpr int M = NS == 0 ? 1 : NS;
  Fold<STAGE, STAGE == STAGE_INIT ? 1 : 2> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  V a[3][M];
  double B[NS == 0 ? 1 : NS * NS];
  auto load = [&]() {
#pragma unroll
    for (int j = 0; j < M; j++) {
      a[0][j] = r[i * M + j];
      a[1][j] = p[i * M + j];
      a[2][j] = v[i * M + j];
    }
    if constexpr (NS > 0)
#pragma unroll
      for (int j = 0; j < NS * NS; j++) B[j] = binv[i * NS * NS + j];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  while (i < n) {
    V y[M];
#pragma unroll
    for (int j = 0; j < M; j++) {
      y[j] = direction(a[0][j], a[1][j], a[2][j], beta, omega);
      p[i * M + j] = y[j];
    }
    if constexpr (NS > 0) node_solve<NS, V>(B, y, ph + i * NS);
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
}

// alpha, then s = r - alpha v (and sh = Binv s); SS: partials of (s, s)
template <class V, int NS, bool SS>
__global__ void __launch_bounds__(VB) k_bicg_s(int64_t n, const V *__restrict__ r, const V *__restrict__ v,
                                               V *__restrict__ s, const double *__restrict__ binv,
                                               V *__restrict__ sh, const double *__restrict__ part, int np,
                                               const KState *in, KState *out, double *__restrict__ part_ss) {
  constexpr int M = NS == 0 ? 1 : NS;
  Fold<STAGE_ALPHA, 1> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  V a[2][M];
  double B[NS == 0 ? 1 : NS * NS];
  auto load = [&]() {
#pragma unroll
    for (int j = 0; j < M; j++) {
      a[0][j] = r[i * M + j];
      a[1][j] = v[i * M + j];
    }
    if constexpr (NS > 0)
#pragma unroll
      for (int j = 0; j < NS * NS; j++) B[j] = binv[i * NS * NS + j];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double alpha = ks.alpha;
  double d = 0.0;
  while (i < n) {
    V y[M];
#pragma unroll
    for (int j = 0; j < M; j++) {
      y[j] = half_step(a[0][j], a[1][j], alpha);
      s[i * M + j] = y[j];
      if (SS) d += (double)y[j] * (double)y[j];
    }
    if constexpr (NS > 0) node_solve<NS, V>(B, y, sh + i * NS);
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
  if constexpr (SS) {
    double vv[1] = {d};
    write_partials_at<1>(vv, part_ss, (int)gridDim.x, (int)blockIdx.x);
  }
}

// omega (STAGE_OMEGA, or STAGE_SOMEGA from (s, t), (t, t), (s, s)), then x += alpha ph + omega
// sh, r = s - omega t; partials of (r0, r), (r, r).  NOS: no preconditioner and no stored s
// (ph = p, sh = s = r - alpha v)
template <class V, class VXo, int STAGE, bool NOS>
__global__ void __launch_bounds__(VB) k_bicg_xr(int64_t n, VXo *__restrict__ x, const V *__restrict__ ph,
                                                const V *__restrict__ sh, const V *__restrict__ s,
                                                const V *__restrict__ v, const V *__restrict__ t,
                                                V *__restrict__ r, const V *__restrict__ r0,
                                                const double *__restrict__ part, int np, const KState *in,
                                                KState *out, double *__restrict__ part_rho) {
  Fold<STAGE, STAGE == STAGE_SOMEGA ? 3 : 2> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  VXo xi;
  V pi, s0, s1, ti, ri;  // s0, s1: r and v (NOS) or s and sh
  auto load = [&]() {
    xi = x[i];
    pi = ph[i];
    s0 = NOS ? r[i] : s[i];
    s1 = NOS ? v[i] : sh[i];
    ti = t[i];
    ri = r0[i];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double alpha = ks.alpha, omega = ks.omega;
  const bool half = ks.half != 0;
  double d0 = 0.0, d1 = 0.0;
  while (i < n) {
    if (half) {
      x[i] = (VXo)((double)xi + alpha * (double)pi);
    } else {
      const V sv = NOS ? half_step(s0, s1, alpha) : s0;
      x[i] = (VXo)((double)xi + alpha * (double)pi + omega * (double)(NOS ? sv : s1));
      const V rv = (V)((double)sv - omega * (double)ti);
      r[i] = rv;
      d0 += (double)ri * (double)rv;
      d1 += (double)rv * (double)rv;
    }
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
  double vv[2] = {d0, d1};
  write_partials_at<2>(vv, part_rho, (int)gridDim.x, (int)blockIdx.x);
}

// One SELL-64 row times values formed from NG gathered vectors.  load() issues the row's first CH
// entries and their gathers together (before the scalars are known); sum() takes the rest.
template <class V, bool NT, class CI, int NG>
struct SellRow {
  static constexpr int CH = 8;
  int32_t q, w;  // position of the row's first entry; entries (uniform in the wave)
  V a[CH];
  V g[NG][CH];
  __device__ __forceinline__ void load(int64_t i, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                       const V *__restrict__ val, const V *__restrict__ y0, const V *__restrict__ y1,
                                       const V *__restrict__ y2) {
    const int sl = __builtin_amdgcn_readfirstlane((int)(i >> 6));
    const int32_t s0 = sptr[sl];
    w = (sptr[sl + 1] - s0) >> 6;
    q = s0 + (int32_t)(i & 63);
    CI c[CH];
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (j < w) {
        c[j] = ldm<NT>(col + (q + 64 * j));
        a[j] = ldm<NT>(val + (q + 64 * j));
      }
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (j < w) {
        const int64_t k = sell_column(c[j], i);
        g[0][j] = y0[k];
        if constexpr (NG > 1) g[1][j] = y1[k];
        if constexpr (NG > 2) g[2][j] = y2[k];
      }
  }
  template <class F>
  __device__ __forceinline__ double sum(int64_t i, const CI *__restrict__ col, const V *__restrict__ val,
                                        const V *__restrict__ y0, const V *__restrict__ y1, const V *__restrict__ y2,
                                        F &&f) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (j < w) acc += (double)a[j] * (double)f(g[0][j], g[NG > 1 ? 1 : 0][j], g[NG > 2 ? 2 : 0][j]);
    for (int j = CH; j < w; j++) {
      const int64_t k = sell_column(ldm<NT>(col + (q + 64 * j)), i);
      acc += (double)ldm<NT>(val + (q + 64 * j)) * (double)f(y0[k], NG > 1 ? y1[k] : (V)0, NG > 2 ? y2[k] : (V)0);
    }
    return acc;
  }
};

// ---- no preconditioner (point Jacobi on the row-scaled operator) ----

// stage, p' = r + beta (p - omega v) and v' = Ahat p' in one launch, p' formed again for every
// gathered column; p, v and p', v' are different buffers.  Partials of (r0, v').
template <class V, int STAGE, bool NT, class CI>
__global__ void __launch_bounds__(VB) k_bicg_pv(int64_t n, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                                const V *__restrict__ val, const V *__restrict__ r,
                                                const V *__restrict__ p, const V *__restrict__ v,
                                                V *__restrict__ pn, V *__restrict__ vn, const V *__restrict__ r0,
                                                const double *__restrict__ part, int np, const KState *in,
                                                KState *out, double *__restrict__ part_alpha) {
  Fold<STAGE, STAGE == STAGE_INIT ? 1 : 2> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  SellRow<V, NT, CI, 3> c;
  V a[4];
  auto load = [&]() {
    c.load(i, sptr, col, val, r, p, v);
    a[0] = r[i];
    a[1] = p[i];
    a[2] = v[i];
    a[3] = r0[i];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  double d = 0.0;
  while (i < n) {
    const V vv = (V)c.sum(i, col, val, r, p, v, [&](V ry, V py, V vy) { return direction(ry, py, vy, beta, omega); });
    pn[i] = direction(a[0], a[1], a[2], beta, omega);
    vn[i] = vv;
    d += (double)a[3] * (double)vv;
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part_alpha, (int)gridDim.x, (int)blockIdx.x);
}

// alpha, then t = Ahat s with s = r - alpha v formed where it is gathered; partials of (s, t),
// (t, t), (s, s)
template <class V, bool NT, class CI>
__global__ void __launch_bounds__(VB) k_bicg_st(int64_t n, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                                const V *__restrict__ val, const V *__restrict__ r,
                                                const V *__restrict__ v, V *__restrict__ t,
                                                const double *__restrict__ part, int np, const KState *in,
                                                KState *out, double *__restrict__ part_omega) {
  Fold<STAGE_ALPHA, 1> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  SellRow<V, NT, CI, 2> c;
  V a[2];
  auto load = [&]() {
    c.load(i, sptr, col, val, r, v, nullptr);
    a[0] = r[i];
    a[1] = v[i];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double alpha = ks.alpha;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  while (i < n) {
    const V tv = (V)c.sum(i, col, val, r, v, nullptr, [&](V ry, V vy, V) { return half_step(ry, vy, alpha); });
    const V sv = half_step(a[0], a[1], alpha);
    t[i] = tv;
    d0 += (double)sv * (double)tv;
    d1 += (double)tv * (double)tv;
    d2 += (double)sv * (double)sv;
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
  double dd[3] = {d0, d1, d2};
  write_partials_at<3>(dd, part_omega, (int)gridDim.x, (int)blockIdx.x);
}

// ---- ILU(0) of a two-colour ordering ----
//
// With the red rows first, the row-scaled operator is [I E; F I] and its ILU(0) factor
//   M = [I 0; F I] [I E; 0 D],  D = diag(1 - diag(F E)),
// since no black-black pair other than the diagonal is in the pattern.  So M^-1 y is
//   z_b = (y_b - F y_r) / D,  z_r = y_r - E z_b,
// and Ahat M^-1 y is y_r on the red rows and z_b + F z_r on the black ones: the product needs
// half of the matrix, the red parts of v and t need no storage (v_r = p_r, t_r = s_r), and an
// application with its product reads three half matrices instead of four.  Vectors are kept in
// colour order (no gathers through a permutation).  M uses the current Jacobian at every
// Newton step: with two colours the factorisation is one pass over F.
template <class V, class CI>
struct RbMat {
  int64_t nr, nb;
  const int32_t *es, *fs;  // slice pointers
  const CI *ec, *fc;       // columns, as 16-bit offsets from the row or as they are
  const V *ev, *fv, *d;    // values; 1 / D
};

template <class V, class CI>
__device__ __forceinline__ double sell_row(int64_t i, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                           const V *__restrict__ val, const V *__restrict__ y) {
  const int64_t sl = i >> 6;
  const int32_t q1 = sptr[sl + 1];
  double acc = 0.0;
#pragma unroll 4
  for (int32_t q = sptr[sl] + (int32_t)(i & 63); q < q1; q += 64)
    acc += (double)val[q] * (double)y[sell_column(col[q], i)];
  return acc;
}

// values of one half in SELL order; BLACK: also 1 / D.  A row without a usable diagonal gets
// NaN, which ends the solve as a breakdown, as a zero pivot does.
template <class V, bool BLACK>
__global__ void __launch_bounds__(VB) k_rb_values(int64_t m, const int32_t *__restrict__ sptr,
                                                  const int32_t *__restrict__ src, const int32_t *__restrict__ tsrc,
                                                  const int32_t *__restrict__ row, const int32_t *__restrict__ colind,
                                                  const int32_t *__restrict__ dofdiag, const double *__restrict__ J,
                                                  const double *__restrict__ rs, V *__restrict__ val,
                                                  V *__restrict__ dinv) {
  const int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  if (i >= m) return;
  const int32_t r = row[i];
  const double s = rs[r], dg = J[dofdiag[r]];
  const bool ok = dg != 0.0 && dg == dg;
  double piv = 1.0;
  const int64_t sl = i >> 6;
  for (int32_t q = sptr[sl] + (int32_t)(i & 63); q < sptr[sl + 1]; q += 64) {
    const int32_t k = src[q];
    const double a = !ok ? __longlong_as_double(0x7ff8000000000000ll) : (k < 0 ? 0.0 : J[k] * s);
    val[q] = (V)a;
    if constexpr (BLACK) {
      const int32_t tk = tsrc[q];
      if (tk >= 0) piv -= a * (J[tk] * rs[colind[k]]);
    }
  }
  if constexpr (BLACK) dinv[i] = ok ? (V)(1.0 / piv) : (V)__longlong_as_double(0x7ff8000000000000ll);
}

// r = r0 = b in colour order, p = v = x = 0; partials of (r, r)
template <class V, class VBin>
__global__ void __launch_bounds__(VB) k_rb_init(int64_t nr, int64_t n, const int32_t *__restrict__ rowr,
                                                const int32_t *__restrict__ rowb, const VBin *__restrict__ b,
                                                V *__restrict__ r, V *__restrict__ r0, V *__restrict__ p,
                                                V *__restrict__ v, V *__restrict__ x, double *__restrict__ part) {
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const V bv = (V)b[i < nr ? rowr[i] : rowb[i - nr]];
    r[i] = bv;
    r0[i] = bv;
    p[i] = (V)0;
    v[i] = (V)0;
    x[i] = (V)0;
    d += (double)bv * (double)bv;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, (int)gridDim.x, (int)blockIdx.x);
}

// out[dof] = x in colour order
template <class V, class VXo>
__global__ void __launch_bounds__(VB) k_rb_out(int64_t nr, int64_t n, const int32_t *__restrict__ rowr,
                                               const int32_t *__restrict__ rowb, const V *__restrict__ x,
                                               VXo *__restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
    out[i < nr ? rowr[i] : rowb[i - nr]] = (VXo)x[i];
}

// black rows, stage: p' = r + beta (p - omega v), z = (p' - F p'_r) / D with p'_r formed from
// the old red p (the red launch writes it)
template <class V, int STAGE, class CI>
__global__ void __launch_bounds__(VB) k_rb_p_black(RbMat<V, CI> A, const V *__restrict__ r, V *__restrict__ p,
                                                   const V *__restrict__ v, V *__restrict__ z,
                                                   const double *__restrict__ part, int np, const KState *in,
                                                   KState *out) {
  Fold<STAGE, STAGE == STAGE_INIT ? 1 : 2> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  SellRow<V, false, CI, 2> c;
  V a[4];
  auto load = [&]() {
    c.load(i, A.fs, A.fc, A.fv, r, p, nullptr);
    a[0] = r[A.nr + i];
    a[1] = p[A.nr + i];
    a[2] = v[A.nr + i];
    a[3] = A.d[i];
  };
  if (i < A.nb) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  while (i < A.nb) {
    const double acc = c.sum(i, A.fc, A.fv, r, p, nullptr, [&](V ry, V py, V) { return direction(ry, py, py, beta, omega); });
    const V pn = direction(a[0], a[1], a[2], beta, omega);
    p[A.nr + i] = pn;
    z[A.nr + i] = (V)(((double)pn - acc) * (double)a[3]);
    i += (int64_t)gridDim.x * VB;
    if (i < A.nb) load();
  }
}

// red rows (v = p there): p' and z = p' - E z_b; partial of (r0, v) = (r0, p') on the red rows
template <class V, class CI>
__global__ void __launch_bounds__(VB) k_rb_p_red(RbMat<V, CI> A, const V *__restrict__ r, V *__restrict__ p,
                                                 V *__restrict__ z, const V *__restrict__ r0, const KState *st,
                                                 double *__restrict__ part, int np) {
  if (idle(st)) return;
  const double beta = st->beta, omega = st->omega;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nr; i += (int64_t)gridDim.x * VB) {
    const V pn = direction(r[i], p[i], p[i], beta, omega);
    p[i] = pn;
    d += (double)r0[i] * (double)pn;
    z[i] = (V)((double)pn - sell_row(i, A.es, A.ec, A.ev, z + A.nr));
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, np, (int)blockIdx.x);
}

// black rows: v = z_b + F z_r; partial of (r0, v)
template <class V, class CI>
__global__ void __launch_bounds__(VB) k_rb_v(RbMat<V, CI> A, const V *__restrict__ z, V *__restrict__ v,
                                             const V *__restrict__ r0, const KState *st, double *__restrict__ part,
                                             int np, int at) {
  if (idle(st)) return;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const V vv = (V)((double)z[k] + sell_row(i, A.fs, A.fc, A.fv, z));
    v[k] = vv;
    d += (double)r0[k] * (double)vv;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, np, at + (int)blockIdx.x);
}

// black rows, alpha: zs = (s - F s_r) / D
template <class V, class CI>
__global__ void __launch_bounds__(VB) k_rb_s_black(RbMat<V, CI> A, const V *__restrict__ r, const V *__restrict__ p,
                                                   const V *__restrict__ v, V *__restrict__ zs,
                                                   const double *__restrict__ part, int np, const KState *in,
                                                   KState *out) {
  Fold<STAGE_ALPHA, 1> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  SellRow<V, false, CI, 2> c;
  V a[3];
  auto load = [&]() {
    c.load(i, A.fs, A.fc, A.fv, r, p, nullptr);
    a[0] = r[A.nr + i];
    a[1] = v[A.nr + i];
    a[2] = A.d[i];
  };
  if (i < A.nb) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double alpha = ks.alpha;
  while (i < A.nb) {
    const double acc = c.sum(i, A.fc, A.fv, r, p, nullptr, [&](V ry, V py, V) { return half_step(ry, py, alpha); });
    zs[A.nr + i] = (V)(((double)half_step(a[0], a[1], alpha) - acc) * (double)a[2]);
    i += (int64_t)gridDim.x * VB;
    if (i < A.nb) load();
  }
}

// red rows: zs = s - E zs_b; partials of (s, t), (t, t), (s, s), all (s, s) on the red rows
template <class V, class CI>
__global__ void __launch_bounds__(VB) k_rb_s_red(RbMat<V, CI> A, const V *__restrict__ r, const V *__restrict__ p,
                                                 V *__restrict__ zs, const KState *st, double *__restrict__ part,
                                                 int np) {
  if (idle(st)) return;
  const double alpha = st->alpha;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nr; i += (int64_t)gridDim.x * VB) {
    const V sv = half_step(r[i], p[i], alpha);
    d += (double)sv * (double)sv;
    zs[i] = (V)((double)sv - sell_row(i, A.es, A.ec, A.ev, zs + A.nr));
  }
  double dd[3] = {d, d, d};
  write_partials_at<3>(dd, part, np, (int)blockIdx.x);
}

// black rows: t = zs_b + F zs_r; partials of (s, t), (t, t), (s, s)
template <class V, class CI>
__global__ void __launch_bounds__(VB) k_rb_t(RbMat<V, CI> A, const V *__restrict__ r, const V *__restrict__ v,
                                             const V *__restrict__ zs, V *__restrict__ t, const KState *st,
                                             double *__restrict__ part, int np, int at) {
  if (idle(st)) return;
  const double alpha = st->alpha;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const V sv = half_step(r[k], v[k], alpha);
    const V tv = (V)((double)zs[k] + sell_row(i, A.fs, A.fc, A.fv, zs));
    t[k] = tv;
    d0 += (double)sv * (double)tv;
    d1 += (double)tv * (double)tv;
    d2 += (double)sv * (double)sv;
  }
  double dd[3] = {d0, d1, d2};
  write_partials_at<3>(dd, part, np, at + (int)blockIdx.x);
}

// all rows, omega: x += alpha z + omega zs, r = s - omega t; partials of (r0, r), (r, r)
template <class V>
__global__ void __launch_bounds__(VB) k_rb_xr(int64_t nr, int64_t n, V *__restrict__ x, const V *__restrict__ z,
                                              const V *__restrict__ zs, const V *__restrict__ p,
                                              const V *__restrict__ v, const V *__restrict__ t, V *__restrict__ r,
                                              const V *__restrict__ r0, const double *__restrict__ part, int np,
                                              const KState *in, KState *out, double *__restrict__ part_rho) {
  Fold<STAGE_SOMEGA, 3> f;
  f.begin(part, np, in);
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  V xi, zi, zsi, ri, vi, ti, r0i;
  auto load = [&]() {
    xi = x[i];
    zi = z[i];
    zsi = zs[i];
    ri = r[i];
    r0i = r0[i];
    vi = i < nr ? p[i] : v[i];
    ti = i < nr ? (V)0 : t[i];
  };
  if (i < n) load();
  const KState &ks = f.finish(part, np, out);
  if (ks.done) return;
  const double alpha = ks.alpha, omega = ks.omega;
  const bool half = ks.half != 0;
  double d0 = 0.0, d1 = 0.0;
  while (i < n) {
    if (half) {
      x[i] = (V)((double)xi + alpha * (double)zi);
    } else {
      x[i] = (V)((double)xi + alpha * (double)zi + omega * (double)zsi);
      const V sv = half_step(ri, vi, alpha);
      const V rv = (V)((double)sv - omega * (double)(i < nr ? sv : ti));
      r[i] = rv;
      d0 += (double)r0i * (double)rv;
      d1 += (double)rv * (double)rv;
    }
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
  double vv[2] = {d0, d1};
  write_partials_at<2>(vv, part_rho, (int)gridDim.x, (int)blockIdx.x);
}
