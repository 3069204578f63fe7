// BiCGStab of a small system in one block (included by vfvm_linalg.hip, inside its namespace).
//
// A system of a few thousand rows leaves the launches of an iteration with nothing to do but
// wait for each other: 12 us (point Jacobi) and 24 us (two-colour ILU(0)) an iteration at any
// size below about 10,000 rows.  One block of 16 waves keeps the whole solve on one compute unit:
// a thread owns up to R rows (r, p, v, t in registers), the gathered vector is in LDS, and the
// barriers are those of a block.  The matrix is copied to LDS where it fits; else it comes from L2
// in every product, and the time grows with the entries.  The arithmetic is that of the kernels in vfvm_bicgstab.h; the sums differ in their order.

constexpr int ONE_T = 1024;  // threads

// sums over the block, the same in every thread; `buf` alternates between two buffers, so that
// one barrier a sum is enough
template <int NR>
__device__ __forceinline__ void one_sum(double (&v)[NR], double (*red)[3][ONE_T / 64], int &buf) {
  double(*rb)[ONE_T / 64] = red[buf];
  buf ^= 1;
#pragma unroll
  for (int k = 0; k < NR; k++) {
    v[k] = wave_sum(v[k]);
    if ((threadIdx.x & 63) == 0) rb[k][threadIdx.x >> 6] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NR; k++) {
    v[k] = lane_value(row_sum(rb[k][threadIdx.x & 15]), 0);
  }
}

// a SELL-64 matrix of m rows, in global memory or copied to LDS
template <class V, class CI>
struct OneMat {
  const int32_t *sptr;
  const CI *col;
  const V *val;
};
constexpr int ONE_LDS = 96 * 1024;  // bytes of the copy
// bytes that a copy takes: values, columns, slice pointers, each rounded up to 8
__host__ __device__ __forceinline__ int64_t one_bytes(int64_t m, int64_t nval, int vsize, int csize) {
  return (nval * vsize + 7) / 8 * 8 + (nval * csize + 7) / 8 * 8 + ((m + 63) / 64 * 4 + 4 + 7) / 8 * 8;
}
template <class V, class CI>
__device__ __forceinline__ OneMat<V, CI> one_copy(char *lds, int m, const OneMat<V, CI> &A) {
  const int nsl = (m + 63) / 64, nval = A.sptr[nsl];
  V *v = reinterpret_cast<V *>(lds);
  CI *c = reinterpret_cast<CI *>(lds + (nval * (int)sizeof(V) + 7) / 8 * 8);
  int32_t *p = reinterpret_cast<int32_t *>(reinterpret_cast<char *>(c) + (nval * (int)sizeof(CI) + 7) / 8 * 8);
#pragma unroll 4
  for (int q = threadIdx.x; q < nval; q += ONE_T) {
    v[q] = A.val[q];
    c[q] = A.col[q];
  }
  for (int q = threadIdx.x; q <= nsl; q += ONE_T) p[q] = A.sptr[q];
  return {p, c, v};
}

// SELL-64 row i times y (LDS), entries in chunks of CH loads
template <class V, class CI>
__device__ __forceinline__ double one_row(int i, const OneMat<V, CI> &A, const V *y) {
  constexpr int CH = 4;
  const int sl = __builtin_amdgcn_readfirstlane(i >> 6);
  const int32_t s0 = A.sptr[sl];
  const int w = (A.sptr[sl + 1] - s0) >> 6;
  const int32_t q = s0 + (i & 63);
  double acc = 0.0;
  for (int j0 = 0; j0 < w; j0 += CH) {
    CI c[CH];
    V a[CH];
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (j0 + j < w) {
        c[j] = A.col[q + 64 * (j0 + j)];
        a[j] = A.val[q + 64 * (j0 + j)];
      }
#pragma unroll
    for (int j = 0; j < CH; j++)
      if (j0 + j < w) acc += (double)a[j] * (double)y[sell_column(c[j], i)];
  }
  return acc;
}

// solver scalars, the same in every thread (KState's fields that run_stage works on)
struct OneState {
  double rho, rho_old, alpha, omega, beta, rr, rr0, ss, tol2, rtol, atol;
  int iters, maxit, done, status, half;
  double best;
  int best_at;
  __device__ __forceinline__ OneState(double rt, double at, int mx) {
    rtol = rt;
    atol = at;
    maxit = mx;
    iters = done = status = half = best_at = 0;
    best = -1.0;
  }
  // looked at every `every` iterations (window 0: never)
  __device__ __forceinline__ bool stagnated(int every, int window) {
    if (window <= 0 || iters % every) return false;
    if (best < 0.0 || rr < 0.81 * best) {
      best = rr;
      best_at = iters;
      return false;
    }
    return iters - best_at >= window;
  }
  __device__ __forceinline__ void report(KState *out) const {
    if (threadIdx.x != 0) return;
    out->rr = rr;
    out->rr0 = rr0;
    out->iters = iters;
    out->done = done;
    out->status = status;
  }
};

// point Jacobi (the row-scaled operator as it is); x starts at 0
template <class V, class VBin, class VXo, class CI, int R, bool COPY>
__global__ void __launch_bounds__(ONE_T) k_bicg_one(int n, OneMat<V, CI> A0, const VBin *__restrict__ b, VXo *__restrict__ x,
                                                    V *__restrict__ r0, double rtol, double atol, int maxit,
                                                    int every, int stag, KState *pinned) {
  __shared__ V y[R * ONE_T];
  __shared__ double red[2][3][ONE_T / 64];
  __shared__ alignas(16) char lds[COPY ? ONE_LDS : 16];
  int buf = 0;
  const int t0 = threadIdx.x;
  const OneMat<V, CI> A = COPY ? one_copy(lds, n, A0) : A0;
  V r[R], p[R], v[R], t[R];
  OneState ks(rtol, atol, maxit);
  {
    double d[1] = {0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      r[k] = p[k] = v[k] = t[k] = (V)0;
      if (i < n) {
        r[k] = (V)b[i];
        r0[i] = r[k];
        x[i] = (VXo)0;
        d[0] += (double)r[k] * (double)r[k];
      }
    }
    one_sum<1>(d, red, buf);
    run_stage<STAGE_INIT>(&ks, d);
  }
  while (!ks.done) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      p[k] = direction(r[k], p[k], v[k], ks.beta, ks.omega);
      if (i < n) y[i] = p[k];
    }
    __syncthreads();
    double d[1] = {0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < n) {
        v[k] = (V)one_row(i, A, y);
        d[0] += (double)r0[i] * (double)v[k];
      }
    }
    one_sum<1>(d, red, buf);
    run_stage<STAGE_ALPHA>(&ks, d);
    if (ks.done) break;
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      r[k] = half_step(r[k], v[k], ks.alpha);  // s
      if (i < n) y[i] = r[k];
    }
    __syncthreads();
    double e[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < n) {
        t[k] = (V)one_row(i, A, y);
        e[0] += (double)r[k] * (double)t[k];
        e[1] += (double)t[k] * (double)t[k];
        e[2] += (double)r[k] * (double)r[k];
      }
    }
    one_sum<3>(e, red, buf);
    run_stage<STAGE_SOMEGA>(&ks, e);
    double f[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < n) {
        if (ks.half) {
          x[i] = (VXo)((double)x[i] + ks.alpha * (double)p[k]);
        } else {
          x[i] = (VXo)((double)x[i] + ks.alpha * (double)p[k] + ks.omega * (double)r[k]);
          r[k] = (V)((double)r[k] - ks.omega * (double)t[k]);
          f[0] += (double)r0[i] * (double)r[k];
          f[1] += (double)r[k] * (double)r[k];
        }
      }
    }
    one_sum<2>(f, red, buf);
    run_stage<STAGE_XR>(&ks, f);
    if (!ks.done && ks.stagnated(every, stag)) break;
  }
  ks.report(pinned);
}

// two-colour ILU(0) (vectors in colour order, RbMat); at most R red and R black rows a thread
template <class V, class VBin, class VXo, class CI, int R, bool COPY>
__global__ void __launch_bounds__(ONE_T) k_rb_one(RbMat<V, CI> A, const int32_t *__restrict__ rowr,
                                                  const int32_t *__restrict__ rowb, const VBin *__restrict__ b,
                                                  VXo *__restrict__ x, V *__restrict__ xc, V *__restrict__ r0,
                                                  double rtol, double atol, int maxit, int every, int stag,
                                                  KState *pinned) {
  __shared__ V yr[R * ONE_T], yb[R * ONE_T];
  __shared__ double red[2][3][ONE_T / 64];
  __shared__ alignas(16) char lds[COPY ? ONE_LDS : 16];
  int buf = 0;
  const int t0 = threadIdx.x, nr = (int)A.nr, nb = (int)A.nb;
  OneMat<V, CI> E{A.es, A.ec, A.ev}, F{A.fs, A.fc, A.fv};
  if constexpr (COPY) {
    const int ne = E.sptr[(nr + 63) / 64];
    E = one_copy(lds, nr, E);
    F = one_copy(lds + one_bytes(nr, ne, sizeof(V), sizeof(CI)), nb, F);
  }
  V rr[R], pr[R], rb[R], pb[R], vb[R], tb[R];
  OneState ks(rtol, atol, maxit);
  {
    double d[1] = {0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      rr[k] = pr[k] = rb[k] = pb[k] = vb[k] = tb[k] = (V)0;
      if (i < nr) {
        rr[k] = (V)b[rowr[i]];
        r0[i] = rr[k];
        xc[i] = (V)0;
        d[0] += (double)rr[k] * (double)rr[k];
      }
      if (i < nb) {
        rb[k] = (V)b[rowb[i]];
        r0[nr + i] = rb[k];
        xc[nr + i] = (V)0;
        d[0] += (double)rb[k] * (double)rb[k];
      }
    }
    one_sum<1>(d, red, buf);
    run_stage<STAGE_INIT>(&ks, d);
  }
  // z = M^-1 (ar, ab) in yr, yb (ar is there already); returns F z_r per black row with `use`
  auto solve = [&](const V(&ar)[R], const V(&ab)[R], auto &&use) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < nb) yb[i] = (V)(((double)ab[k] - one_row(i, F, yr)) * (double)A.d[i]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < nr) yr[i] = (V)((double)ar[k] - one_row(i, E, yb));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < nb) use(k, i, (V)((double)yb[i] + one_row(i, F, yr)));
    }
  };
  while (!ks.done) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      pr[k] = direction(rr[k], pr[k], pr[k], ks.beta, ks.omega);
      pb[k] = direction(rb[k], pb[k], vb[k], ks.beta, ks.omega);
      if (i < nr) yr[i] = pr[k];
    }
    double d[1] = {0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int i = t0 + k * ONE_T;
      if (i < nr) d[0] += (double)r0[i] * (double)pr[k];
    }
    solve(pr, pb, [&](int k, int i, V w) {
      vb[k] = w;
      d[0] += (double)r0[nr + i] * (double)w;
    });
    one_sum<1>(d, red, buf);
    run_stage<STAGE_ALPHA>(&ks, d);
    if (ks.done) break;
    double e[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {  // x += alpha z; s in place of r; its red part for the next solve
      const int i = t0 + k * ONE_T;
      if (i < nr) xc[i] = (V)((double)xc[i] + ks.alpha * (double)yr[i]);
      if (i < nb) xc[nr + i] = (V)((double)xc[nr + i] + ks.alpha * (double)yb[i]);
      rr[k] = half_step(rr[k], pr[k], ks.alpha);
      rb[k] = half_step(rb[k], vb[k], ks.alpha);
      if (i < nr) yr[i] = rr[k];
      const double s2 = (double)rr[k] * (double)rr[k];
      e[0] += s2;
      e[1] += s2;
      e[2] += s2;
    }
    solve(rr, rb, [&](int k, int, V w) {
      tb[k] = w;
      e[0] += (double)rb[k] * (double)w;
      e[1] += (double)w * (double)w;
      e[2] += (double)rb[k] * (double)rb[k];
    });
    one_sum<3>(e, red, buf);
    run_stage<STAGE_SOMEGA>(&ks, e);
    double f[2] = {0.0, 0.0};
    if (!ks.half) {
#pragma unroll
      for (int k = 0; k < R; k++) {
        const int i = t0 + k * ONE_T;
        if (i < nr) {
          xc[i] = (V)((double)xc[i] + ks.omega * (double)yr[i]);
          rr[k] = (V)((double)rr[k] - ks.omega * (double)rr[k]);
          f[0] += (double)r0[i] * (double)rr[k];
          f[1] += (double)rr[k] * (double)rr[k];
        }
        if (i < nb) {
          xc[nr + i] = (V)((double)xc[nr + i] + ks.omega * (double)yb[i]);
          rb[k] = (V)((double)rb[k] - ks.omega * (double)tb[k]);
          f[0] += (double)r0[nr + i] * (double)rb[k];
          f[1] += (double)rb[k] * (double)rb[k];
        }
      }
    }
    one_sum<2>(f, red, buf);
    run_stage<STAGE_XR>(&ks, f);
    if (!ks.done && ks.stagnated(every, stag)) break;
  }
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int i = t0 + k * ONE_T;
    if (i < nr) x[rowr[i]] = (VXo)xc[i];
    if (i < nb) x[rowb[i]] = (VXo)xc[nr + i];
  }
  ks.report(pinned);
}
