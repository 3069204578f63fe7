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
// and after: 33^2 rows with point Jacobi 5.73 and 3.36 ms, 3 x 129^2 with block Jacobi 146.8
// and 79.3 ms, 101^2 with ILU(0) 15.8 and 8.6 ms; 129^3 with ILU(0) in FP32, where memory
// counts (ILU and product 128 us, now 79), 64.4 and 43.7 ms.

enum { SLOT_RHO = 0, SLOT_BETA = 1, SLOT_ALPHA = 2, SLOT_REPORT = 3 };

// totals of the previous reduction (NR sums of np partials) and the stage on them; the new
// state in `ks` (shared memory), stored to `out` by block 0.  A finished solve's state is
// passed on unchanged.
template <int STAGE, int NR>
__device__ __forceinline__ void fold_state(const double *__restrict__ part, int np, const KState *__restrict__ in,
                                           KState *__restrict__ out, KState &ks) {
  __shared__ double red[NR][VB / 64];
  double acc[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) acc[k] = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < np; b += VB)
#pragma unroll
    for (int k = 0; k < NR; k++) acc[k] += part[(size_t)k * np + b];
  if (threadIdx.x == 0) ks = *in;
#pragma unroll
  for (int k = 0; k < NR; k++) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc[k] += __shfl_xor(acc[k], o, 64);
    if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot[NR];
#pragma unroll
    for (int k = 0; k < NR; k++) {
      tot[k] = 0.0;
#pragma unroll
      for (int w = 0; w < VB / 64; w++) tot[k] += red[k][w];
    }
    if (!ks.done && !(STAGE == STAGE_OMEGA && ks.half)) run_stage<STAGE>(&ks, tot);
    if (blockIdx.x == 0) *out = ks;
  }
  __syncthreads();
}

template <int NR>
__device__ __forceinline__ void write_partials_at(const double (&v)[NR], double *part, int np, int at) {
  __shared__ double sh[16];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    const double s = block_sum(v[k], sh);
    if (threadIdx.x == 0) part[(size_t)k * np + at] = s;
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

// z = Binv y of node K (block Jacobi)
template <int NS, class V>
__device__ __forceinline__ void node_solve(const double *__restrict__ binv, int64_t K, const V (&y)[NS],
                                           V *__restrict__ z) {
#pragma unroll
  for (int i = 0; i < NS; i++) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < NS; j++) acc += binv[K * NS * NS + i * NS + j] * (double)y[j];
    z[K * NS + i] = (V)acc;
  }
}

// the state after the last queued iteration, for the host (one block)
__global__ void __launch_bounds__(VB) k_bicg_report(const double *__restrict__ part, int np, const KState *in,
                                                    KState *out) {
  __shared__ KState ks;
  fold_state<STAGE_XR, 2>(part, np, in, out, ks);
}

// stage (INIT or XR), then p = r + beta (p - omega v); NS > 0: also ph = Binv p per node of NS
// rows (n counts nodes then)
template <class V, int STAGE, int NS>
__global__ void __launch_bounds__(VB) k_bicg_p(int64_t n, const V *__restrict__ r, V *__restrict__ p,
                                               const V *__restrict__ v, const double *__restrict__ binv,
                                               V *__restrict__ ph, const double *__restrict__ part, int np,
                                               const KState *in, KState *out) {
  __shared__ KState ks;
  fold_state<STAGE, STAGE == STAGE_INIT ? 1 : 2>(part, np, in, out, ks);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    if constexpr (NS == 0) {
      p[i] = direction(r[i], p[i], v[i], beta, omega);
    } else {
      V y[NS];
#pragma unroll
      for (int j = 0; j < NS; j++) {
        y[j] = direction(r[i * NS + j], p[i * NS + j], v[i * NS + j], beta, omega);
        p[i * NS + j] = y[j];
      }
      node_solve<NS, V>(binv, i, y, ph);
    }
  }
}

// alpha, then s = r - alpha v (and sh = Binv s); SS: partials of (s, s)
template <class V, int NS, bool SS>
__global__ void __launch_bounds__(VB) k_bicg_s(int64_t n, const V *__restrict__ r, const V *__restrict__ v,
                                               V *__restrict__ s, const double *__restrict__ binv,
                                               V *__restrict__ sh, const double *__restrict__ part, int np,
                                               const KState *in, KState *out, double *__restrict__ part_ss) {
  __shared__ KState ks;
  fold_state<STAGE_ALPHA, 1>(part, np, in, out, ks);
  if (ks.done) return;
  const double alpha = ks.alpha;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    if constexpr (NS == 0) {
      const V sv = half_step(r[i], v[i], alpha);
      s[i] = sv;
      if (SS) d += (double)sv * (double)sv;
    } else {
      V y[NS];
#pragma unroll
      for (int j = 0; j < NS; j++) {
        y[j] = half_step(r[i * NS + j], v[i * NS + j], alpha);
        s[i * NS + j] = y[j];
      }
      node_solve<NS, V>(binv, i, y, sh);
    }
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
  __shared__ KState ks;
  fold_state<STAGE, STAGE == STAGE_SOMEGA ? 3 : 2>(part, np, in, out, ks);
  if (ks.done) return;
  const double alpha = ks.alpha, omega = ks.omega;
  const bool half = ks.half != 0;
  double d0 = 0.0, d1 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    if (half) {
      x[i] = (VXo)((double)x[i] + alpha * (double)ph[i]);
    } else {
      const V sv = NOS ? half_step(r[i], v[i], alpha) : s[i];
      x[i] = (VXo)((double)x[i] + alpha * (double)ph[i] + omega * (double)(NOS ? sv : sh[i]));
      const V rv = (V)((double)sv - omega * (double)t[i]);
      r[i] = rv;
      d0 += (double)r0[i] * (double)rv;
      d1 += (double)rv * (double)rv;
    }
  }
  double vv[2] = {d0, d1};
  write_partials_at<2>(vv, part_rho, (int)gridDim.x, (int)blockIdx.x);
}

// ---- no preconditioner (point Jacobi on the row-scaled operator) ----

// row r of Ahat y with y(j) formed from the vectors where it is gathered
template <class V, bool NT, class CI, class F>
__device__ __forceinline__ double sell_row(int64_t r, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                           const V *__restrict__ val, F &&y) {
  const int64_t sl = r >> 6;
  const int32_t q1 = sptr[sl + 1];
  double acc = 0.0;
#pragma unroll 4
  for (int32_t q = sptr[sl] + (int32_t)(r & 63); q < q1; q += 64)
    acc += (double)ldm<NT>(val + q) * (double)y(sell_column(ldm<NT>(col + q), r));
  return acc;
}

// stage, p' = r + beta (p - omega v) and v' = Ahat p' in one launch, p' formed again for every
// gathered column; p, v and p', v' are different buffers.  Partials of (r0, v').
template <class V, int STAGE, bool NT, class CI>
__global__ void __launch_bounds__(VB) k_bicg_pv(int64_t n, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                                const V *__restrict__ val, const V *__restrict__ r,
                                                const V *__restrict__ p, const V *__restrict__ v,
                                                V *__restrict__ pn, V *__restrict__ vn, const V *__restrict__ r0,
                                                const double *__restrict__ part, int np, const KState *in,
                                                KState *out, double *__restrict__ part_alpha) {
  __shared__ KState ks;
  fold_state<STAGE, STAGE == STAGE_INIT ? 1 : 2>(part, np, in, out, ks);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const V vv = (V)sell_row<V, NT, CI>(i, sptr, col, val,
                                        [&](int64_t j) { return direction(r[j], p[j], v[j], beta, omega); });
    pn[i] = direction(r[i], p[i], v[i], beta, omega);
    vn[i] = vv;
    d += (double)r0[i] * (double)vv;
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
  __shared__ KState ks;
  fold_state<STAGE_ALPHA, 1>(part, np, in, out, ks);
  if (ks.done) return;
  const double alpha = ks.alpha;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const V tv = (V)sell_row<V, NT, CI>(i, sptr, col, val, [&](int64_t j) { return half_step(r[j], v[j], alpha); });
    const V sv = half_step(r[i], v[i], alpha);
    t[i] = tv;
    d0 += (double)sv * (double)tv;
    d1 += (double)tv * (double)tv;
    d2 += (double)sv * (double)sv;
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
template <class V>
struct RbMat {
  int64_t nr, nb;
  const int32_t *es, *fs;    // slice pointers
  const int16_t *eo, *fo;    // columns as offsets from the row, or
  const int32_t *ec, *fc;    // as they are
  const V *ev, *fv, *d;      // values; 1 / D
};

template <class V, bool OFF, class F>
__device__ __forceinline__ double rb_row(int64_t i, const int32_t *__restrict__ sptr, const int16_t *__restrict__ off,
                                         const int32_t *__restrict__ col, const V *__restrict__ val, F &&y) {
  const int64_t sl = i >> 6;
  const int32_t q1 = sptr[sl + 1];
  double acc = 0.0;
#pragma unroll 4
  for (int32_t q = sptr[sl] + (int32_t)(i & 63); q < q1; q += 64)
    acc += (double)val[q] * (double)y(OFF ? i + off[q] : (int64_t)col[q]);
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

// the red part of v is p, so p' = r + beta (p - omega p)
template <class V>
__device__ __forceinline__ V direction_red(V r, V p, double beta, double omega) {
  return (V)((double)r + beta * ((double)p - omega * (double)p));
}

// black rows, stage: p' = r + beta (p - omega v), z = (p' - F p'_r) / D with p'_r formed from
// the old red p (the red launch writes it)
template <class V, int STAGE, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_p_black(RbMat<V> A, const V *__restrict__ r, V *__restrict__ p,
                                                   const V *__restrict__ v, V *__restrict__ z,
                                                   const double *__restrict__ part, int np, const KState *in,
                                                   KState *out) {
  __shared__ KState ks;
  fold_state<STAGE, STAGE == STAGE_INIT ? 1 : 2>(part, np, in, out, ks);
  if (ks.done) return;
  const double beta = ks.beta, omega = ks.omega;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const double acc = rb_row<V, OFF>(i, A.fs, A.fo, A.fc, A.fv,
                                      [&](int64_t j) { return direction_red(r[j], p[j], beta, omega); });
    const V pn = direction(r[k], p[k], v[k], beta, omega);
    p[k] = pn;
    z[k] = (V)(((double)pn - acc) * (double)A.d[i]);
  }
}

// red rows: p' and z = p' - E z_b; partial of (r0, v) = (r0, p') on the red rows
template <class V, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_p_red(RbMat<V> A, const V *__restrict__ r, V *__restrict__ p,
                                                 V *__restrict__ z, const V *__restrict__ r0, const KState *st,
                                                 double *__restrict__ part, int np) {
  if (idle(st)) return;
  const double beta = st->beta, omega = st->omega;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nr; i += (int64_t)gridDim.x * VB) {
    const double acc = rb_row<V, OFF>(i, A.es, A.eo, A.ec, A.ev, [&](int64_t j) { return z[A.nr + j]; });
    const V pn = direction_red(r[i], p[i], beta, omega);
    p[i] = pn;
    z[i] = (V)((double)pn - acc);
    d += (double)r0[i] * (double)pn;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, np, (int)blockIdx.x);
}

// black rows: v = z_b + F z_r; partial of (r0, v)
template <class V, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_v(RbMat<V> A, const V *__restrict__ z, V *__restrict__ v,
                                             const V *__restrict__ r0, const KState *st, double *__restrict__ part,
                                             int np, int at) {
  if (idle(st)) return;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const V vv = (V)((double)z[k] + rb_row<V, OFF>(i, A.fs, A.fo, A.fc, A.fv, [&](int64_t j) { return z[j]; }));
    v[k] = vv;
    d += (double)r0[k] * (double)vv;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, np, at + (int)blockIdx.x);
}

// black rows, alpha: zs = (s - F s_r) / D
template <class V, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_s_black(RbMat<V> A, const V *__restrict__ r, const V *__restrict__ p,
                                                   const V *__restrict__ v, V *__restrict__ zs,
                                                   const double *__restrict__ part, int np, const KState *in,
                                                   KState *out) {
  __shared__ KState ks;
  fold_state<STAGE_ALPHA, 1>(part, np, in, out, ks);
  if (ks.done) return;
  const double alpha = ks.alpha;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const double acc = rb_row<V, OFF>(i, A.fs, A.fo, A.fc, A.fv, [&](int64_t j) { return half_step(r[j], p[j], alpha); });
    zs[k] = (V)(((double)half_step(r[k], v[k], alpha) - acc) * (double)A.d[i]);
  }
}

// red rows: zs = s - E zs_b; partials of (s, t), (t, t), (s, s), all (s, s) on the red rows
template <class V, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_s_red(RbMat<V> A, const V *__restrict__ r, const V *__restrict__ p,
                                                 V *__restrict__ zs, const KState *st, double *__restrict__ part,
                                                 int np) {
  if (idle(st)) return;
  const double alpha = st->alpha;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nr; i += (int64_t)gridDim.x * VB) {
    const double acc = rb_row<V, OFF>(i, A.es, A.eo, A.ec, A.ev, [&](int64_t j) { return zs[A.nr + j]; });
    const V sv = half_step(r[i], p[i], alpha);
    zs[i] = (V)((double)sv - acc);
    d += (double)sv * (double)sv;
  }
  __shared__ double sh[16];
  const double s = block_sum(d, sh);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < 3; k++) part[(size_t)k * np + blockIdx.x] = s;
}

// black rows: t = zs_b + F zs_r; partials of (s, t), (t, t), (s, s)
template <class V, bool OFF>
__global__ void __launch_bounds__(VB) k_rb_t(RbMat<V> A, const V *__restrict__ r, const V *__restrict__ v,
                                             const V *__restrict__ zs, V *__restrict__ t, const KState *st,
                                             double *__restrict__ part, int np, int at) {
  if (idle(st)) return;
  const double alpha = st->alpha;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < A.nb; i += (int64_t)gridDim.x * VB) {
    const int64_t k = A.nr + i;
    const V tv = (V)((double)zs[k] + rb_row<V, OFF>(i, A.fs, A.fo, A.fc, A.fv, [&](int64_t j) { return zs[j]; }));
    const V sv = half_step(r[k], v[k], alpha);
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
  __shared__ KState ks;
  fold_state<STAGE_SOMEGA, 3>(part, np, in, out, ks);
  if (ks.done) return;
  const double alpha = ks.alpha, omega = ks.omega;
  const bool half = ks.half != 0;
  double d0 = 0.0, d1 = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    if (half) {
      x[i] = (V)((double)x[i] + alpha * (double)z[i]);
    } else {
      x[i] = (V)((double)x[i] + alpha * (double)z[i] + omega * (double)zs[i]);
      const V sv = half_step(r[i], i < nr ? p[i] : v[i], alpha);
      const V rv = (V)((double)sv - omega * (double)(i < nr ? sv : t[i]));
      r[i] = rv;
      d0 += (double)r0[i] * (double)rv;
      d1 += (double)rv * (double)rv;
    }
  }
  double dd[2] = {d0, d1};
  write_partials_at<2>(dd, part_rho, (int)gridDim.x, (int)blockIdx.x);
}
