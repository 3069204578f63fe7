// Kernels of the restarted GMRES (included by vfvm_linalg.hip, inside its namespace).
//
// An Arnoldi step has four kernels (and the preconditioner's, if it is not a node solve):
//   k_gm_next   finishes the column before: ||w||, Givens rotations (block 0); v = w / ||w||,
//               z = Binv v
//   k_gm_av     w = Ahat z, partials of (V_j, w)
//   k_gm_ortho  w -= sum_j h_j V_j, partials of (V_j, w)            (first Gram-Schmidt pass)
//   k_gm_ortho  w -= sum_j h_j V_j, partials of ||w||^2             (second pass)
// Each sums the partials of the one before it at its entry, as the BiCGStab kernels do; the
// state alternates between two slots, so that no block reads what another one writes.  Small
// systems, for which GMRES is used, are bound by this chain of launches: before, a step had
// twelve (72 us of a solve at 3 x 49^2 rows, 25 now: a Newton sweep 182 and 65 ms).  The dots give each wave its own basis vectors:
// a block-wide sum per basis vector, one after the other, took 12.5 us for up to 30 of them.

// h_j (j < nv) of np partials each in shared memory
__device__ __forceinline__ void gm_fold(const double *__restrict__ part, int np, int nv, double *h) {
  const int lane = threadIdx.x & 63;
#pragma unroll 4
  for (int j = threadIdx.x >> 6; j < nv; j += VB / 64) {
    double a = 0.0;
    for (int b = lane; b < np; b += 64) a += part[(size_t)j * np + b];
    a = wave_sum(a);
    if (lane == 0) h[j] = a;
  }
  __syncthreads();
}

// per-lane sums of (V_j, w) over one tile of VB rows (w of the tile in shared memory, 0 past the
// end); wave k holds j = k, k + 4, ...
template <class V>
struct GmDots {
  static constexpr int MAXQ = 16;  // 64 basis vectors
  double d[MAXQ];
  __device__ __forceinline__ GmDots() {
#pragma unroll
    for (int q = 0; q < MAXQ; q++) d[q] = 0.0;
  }
  // loads in groups of 4 vectors x 4 rows, all issued before the first is used; past the last
  // vector and row they repeat it (those sums are not stored, w is 0 there)
  __device__ __forceinline__ void tile(int64_t row0, int64_t n, int nv, const V *__restrict__ Vb, const V *wt) {
    constexpr int W = VB / 64, GR = 4;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    V wr[W];
    int64_t row[W];
#pragma unroll
    for (int c = 0; c < W; c++) {
      wr[c] = wt[lane + 64 * c];
      row[c] = row0 + lane + 64 * c;
      if (row[c] >= n) row[c] = n - 1;
    }
#pragma unroll
    for (int q0 = 0; q0 < MAXQ; q0 += GR) {
      if (wave + q0 * W >= nv) break;
      V v[GR][W];
#pragma unroll
      for (int q = 0; q < GR; q++) {
        const V *vj = Vb + (int64_t)min(wave + (q0 + q) * W, nv - 1) * n;
#pragma unroll
        for (int c = 0; c < W; c++) v[q][c] = vj[row[c]];
      }
#pragma unroll
      for (int q = 0; q < GR; q++)
#pragma unroll
        for (int c = 0; c < W; c++) d[q0 + q] += (double)v[q][c] * (double)wr[c];
    }
  }
  __device__ __forceinline__ void store(int nv, double *__restrict__ part) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
#pragma unroll
    for (int q = 0; q < MAXQ; q++) {
      const int j = wave + q * (VB / 64);
      if (j < nv) {
        const double s = wave_sum(d[q]);
        if (lane == 0) part[(size_t)j * gridDim.x + blockIdx.x] = s;
      }
    }
  }
};

// sums of np partials for each of gridDim.x values
__global__ void __launch_bounds__(VB) k_gm_sum(int np, const double *__restrict__ part, double *__restrict__ h,
                                               const KState *st) {
  if (idle(st)) return;
  __shared__ double sh[16];
  double a = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < np; b += VB) a += part[(size_t)blockIdx.x * np + b];
  const double s = block_sum(a, sh);
  if (threadIdx.x == 0) h[blockIdx.x] = s;
}

// b in the solve precision, x = 0; partials of (b, b)
template <class V, class VBin, class VXo>
__global__ void __launch_bounds__(VB) k_gm_init(int64_t n, const VBin *__restrict__ b, V *__restrict__ bb,
                                                VXo *__restrict__ x, double *__restrict__ part) {
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const V bv = (V)b[i];
    bb[i] = bv;
    x[i] = (VXo)0;
    d += (double)bv * (double)bv;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, (int)gridDim.x, (int)blockIdx.x);
}

// r = b - Ahat x (restart); partials of (r, r)
template <class V, class VXo, class CI>
__global__ void __launch_bounds__(VB) k_gm_residual(int64_t n, const int32_t *__restrict__ sptr,
                                                    const CI *__restrict__ col, const V *__restrict__ val,
                                                    const VXo *__restrict__ x, const V *__restrict__ b,
                                                    V *__restrict__ r, const KState *st, double *__restrict__ part) {
  if (idle(st)) return;
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const int64_t sl = i >> 6;
    const int32_t p1 = sptr[sl + 1];
    double acc = 0.0;
#pragma unroll 4
    for (int32_t q = sptr[sl] + (int32_t)(i & 63); q < p1; q += 64)
      acc += (double)val[q] * (double)x[sell_column(col[q], i)];
    const V rv = (V)((double)b[i] - acc);
    r[i] = rv;
    d += (double)rv * (double)rv;
  }
  double dd[1] = {d};
  write_partials_at<1>(dd, part, (int)gridDim.x, (int)blockIdx.x);
}

struct GmArrays {
  double *H, *h1, *h2, *cs, *sn, *g;
  int m;
};

// column k of the Hessenberg matrix from the two Gram-Schmidt passes and hn = ||w||: rotations,
// residual estimate, stop flags (one block; ks in shared memory).  Thread t <= k passes entry t of
// the column and of the earlier rotations.
__device__ __forceinline__ void gm_column(const GmArrays &G, int k, double ht, double ct, double st, double hn,
                                          KState &ks) {
  __shared__ double col[66], cs[65], sn[65];
  const int t = threadIdx.x;
  const double gk = t == 0 ? G.g[k] : 0.0;
  if (t <= k) {
    col[t] = ht;
    cs[t] = ct;
    sn[t] = st;
  }
  __syncthreads();
  if (t == 0) {
    double c = col[0];  // the entry that the next rotation changes
#pragma unroll 4
    for (int j = 0; j < k; j++) {
      const double o = col[j + 1];
      col[j] = cs[j] * c + sn[j] * o;
      c = -sn[j] * c + cs[j] * o;
    }
    const double den = sqrt(c * c + hn * hn);
    const double ck = den > 0 ? c / den : 1.0, sk = den > 0 ? hn / den : 0.0;
    col[k] = den;
    G.cs[k] = ck;
    G.sn[k] = sk;
    G.g[k + 1] = -sk * gk;
    G.g[k] = ck * gk;
    ks.iters += 1;
    ks.gm_k = k + 1;
    const double res = fabs(sk * gk);
    ks.rr = res * res;
    if (res * res <= ks.tol2) ks.gm_conv = 1;
    if (ks.iters >= ks.maxit) ks.gm_stop = 1;
    if (hn == 0.0) ks.gm_conv = 1;  // lucky breakdown: exact solution in the subspace
    if (ks.gm_conv || ks.gm_stop) ks.done = 1;
  }
  __syncthreads();
  if (t <= k) G.H[t * G.m + k] = col[t];
}

// start of a cycle: residual norm, stop flags
__device__ __forceinline__ void gm_start(const GmArrays &G, double rr, int first, KState &ks) {
  if (threadIdx.x <= G.m) G.g[threadIdx.x] = threadIdx.x == 0 ? sqrt(rr) : 0.0;
  if (threadIdx.x != 0) return;
  if (first) {
    const double tol = ks.atol + ks.rtol * sqrt(rr);
    ks.tol2 = tol * tol;
    ks.rr0 = rr;
  }
  ks.rr = rr;
  ks.gm_k = 0;
  if (rr <= ks.tol2) ks.gm_conv = 1;
  if (ks.iters >= ks.maxit) ks.gm_stop = 1;
  if (ks.gm_conv || ks.gm_stop) ks.done = 1;
}

// k < 0: start of a cycle (w the residual); k >= 0: column k is finished.  Then v = w / ||w|| and,
// with NS > 0, z = Binv v per node of NS rows (n counts nodes then).  `pinned` (host memory, may
// be null) gets a copy of the state.  Only block 0 knows whether the
// solve has ended; the other blocks' v and z are not used then.
template <class V, int NS>
__global__ void __launch_bounds__(VB) k_gm_next(int64_t n, const V *__restrict__ w, V *__restrict__ v,
                                                const double *__restrict__ binv, V *__restrict__ z, GmArrays G, int k,
                                                int first, const double *__restrict__ part, int np, const KState *in,
                                                KState *out, KState *pinned) {
  constexpr int M = NS == 0 ? 1 : NS;
  __shared__ double red[VB / 64];
  __shared__ KState ks;
  constexpr int WORDS = sizeof(KState) / 4;
  double a = threadIdx.x < np ? part[threadIdx.x] : 0.0;
  if (threadIdx.x < WORDS)
    reinterpret_cast<uint32_t *>(&ks)[threadIdx.x] = reinterpret_cast<const uint32_t *>(in)[threadIdx.x];
  int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x;
  V y[M];
  double B[NS == 0 ? 1 : NS * NS];
  auto load = [&]() {
#pragma unroll
    for (int j = 0; j < M; j++) y[j] = w[i * M + j];
    if constexpr (NS > 0)
#pragma unroll
      for (int j = 0; j < NS * NS; j++) B[j] = binv[i * NS * NS + j];
  };
  if (i < n) load();
  double ht = 0.0, ct = 0.0, st = 0.0;
  if (blockIdx.x == 0 && (int)threadIdx.x <= k) {
    ht = G.h1[threadIdx.x] + G.h2[threadIdx.x];
    if ((int)threadIdx.x < k) {
      ct = G.cs[threadIdx.x];
      st = G.sn[threadIdx.x];
    }
  }
#pragma unroll 4
  for (int b = threadIdx.x + VB; b < np; b += VB) a += part[b];
  a = wave_sum(a);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  const bool done = ks.done != 0;
  double rr = 0.0;
#pragma unroll
  for (int q = 0; q < VB / 64; q++) rr += red[q];
  if (blockIdx.x == 0) {
    __syncthreads();
    if (!done) {
      if (k < 0)
        gm_start(G, rr, first, ks);
      else
        gm_column(G, k, ht, ct, st, sqrt(rr), ks);
    }
    __syncthreads();
    if (threadIdx.x < WORDS) {
      const uint32_t word = reinterpret_cast<const uint32_t *>(&ks)[threadIdx.x];
      reinterpret_cast<uint32_t *>(out)[threadIdx.x] = word;
      if (pinned) reinterpret_cast<uint32_t *>(pinned)[threadIdx.x] = word;
    }
  }
  if (done) return;
  const double inv = rr > 0.0 ? 1.0 / sqrt(rr) : 0.0;
  while (i < n) {
    V u[M];
#pragma unroll
    for (int j = 0; j < M; j++) {
      u[j] = (V)((double)y[j] * inv);
      v[i * M + j] = u[j];
    }
    if constexpr (NS > 0) node_solve<NS, V>(B, u, z + i * NS);
    i += (int64_t)gridDim.x * VB;
    if (i < n) load();
  }
}

// w = Ahat z; partials of (V_j, w), j < nv
template <class V, bool NT, class CI>
__global__ void __launch_bounds__(VB) k_gm_av(int64_t n, const int32_t *__restrict__ sptr, const CI *__restrict__ col,
                                              const V *__restrict__ val, const V *__restrict__ z, V *__restrict__ w,
                                              int nv, const V *__restrict__ Vb, double *__restrict__ part,
                                              const KState *st) {
  if (idle(st)) return;
  __shared__ V wt[VB];
  GmDots<V> D;
  for (int64_t r0 = (int64_t)blockIdx.x * VB; r0 < n; r0 += (int64_t)gridDim.x * VB) {
    const int64_t i = r0 + threadIdx.x;
    V wv = (V)0;
    if (i < n) {
      const int64_t sl = i >> 6;
      const int32_t p1 = sptr[sl + 1];
      double acc = 0.0;
#pragma unroll 4
      for (int32_t q = sptr[sl] + (int32_t)(i & 63); q < p1; q += 64)
        acc += (double)ldm<NT>(val + q) * (double)z[sell_column(ldm<NT>(col + q), i)];
      wv = (V)acc;
      w[i] = wv;
    }
    __syncthreads();
    wt[threadIdx.x] = wv;
    __syncthreads();
    D.tile(r0, n, nv, Vb, wt);
  }
  D.store(nv, part);
}

// w -= sum_j h_j V_j with h summed from np partials each (block 0 stores it); partials of (V_j, w),
// or with LAST of ||w||^2
template <class V, bool LAST>
__global__ void __launch_bounds__(VB) k_gm_ortho(int64_t n, int nv, const V *__restrict__ Vb, V *__restrict__ w,
                                                 const double *__restrict__ part_in, int np, double *__restrict__ hout,
                                                 double *__restrict__ part_out, const KState *st) {
  if (idle(st)) return;
  constexpr int CH = 8;
  __shared__ double h[64 + CH];
  __shared__ V wt[VB];
  if (threadIdx.x >= nv && threadIdx.x < 64 + CH) h[threadIdx.x] = 0.0;
  gm_fold(part_in, np, nv, h);
  if (blockIdx.x == 0 && threadIdx.x < nv) hout[threadIdx.x] = h[threadIdx.x];
  GmDots<V> D;
  double d = 0.0;
  for (int64_t r0 = (int64_t)blockIdx.x * VB; r0 < n; r0 += (int64_t)gridDim.x * VB) {
    const int64_t i = r0 + threadIdx.x;
    V wv = (V)0;
    if (i < n) {
      double acc = (double)w[i];
      for (int j0 = 0; j0 < nv; j0 += CH) {  // CH loads at once; past the last vector times 0
        V v[CH];
#pragma unroll
        for (int j = 0; j < CH; j++) v[j] = Vb[(int64_t)min(j0 + j, nv - 1) * n + i];
#pragma unroll
        for (int j = 0; j < CH; j++) acc -= h[j0 + j] * (double)v[j];
      }
      wv = (V)acc;
      w[i] = wv;
      if (LAST) d += (double)wv * (double)wv;
    }
    if constexpr (!LAST) {
      __syncthreads();
      wt[threadIdx.x] = wv;
      __syncthreads();
      D.tile(r0, n, nv, Vb, wt);
    }
  }
  if constexpr (LAST) {
    double dd[1] = {d};
    write_partials_at<1>(dd, part_out, (int)gridDim.x, (int)blockIdx.x);
  } else {
    D.store(nv, part_out);
  }
}

// end of a cycle of k columns (the state's count): y from the triangular system (every block),
// w = sum_j y_j V_j; ADD: x += Binv w per node (NS > 0) or x += w.  `out` is the state with its
// count of columns at 0: a cycle is added once.
template <class V, class VXo, int NS, bool ADD>
__global__ void __launch_bounds__(VB) k_gm_combine(int64_t n, int64_t ldv, const V *__restrict__ Vb,
                                                   const double *__restrict__ binv, V *__restrict__ w,
                                                   VXo *__restrict__ x, GmArrays G, const KState *in, KState *out) {
  constexpr int M = NS == 0 ? 1 : NS;
  __shared__ double y[64], R[64 * 65];
  const int k = in->gm_k, t = threadIdx.x;
  for (int q = t; q < k * G.m; q += VB)
    if (q % G.m < k) R[q / G.m * 65 + q % G.m] = G.H[q];
  __syncthreads();
  if (t < 64) {  // one wave: lane i holds row i
    double acc = t < k ? G.g[t] : 0.0;
    const double dg = t < k ? R[t * 65 + t] : 1.0;
    for (int j = k - 1; j >= 0; j--) {
      const double hij = t < j ? R[t * 65 + j] : 0.0;
      const double yj = lane_value(acc, j) / lane_value(dg, j);
      if (t == j) y[j] = yj;
      acc -= hij * yj;
    }
  }
  if (blockIdx.x == 0 && t >= 64 && t < 64 + (int)(sizeof(KState) / 4)) {
    const int q = t - 64;
    uint32_t word = reinterpret_cast<const uint32_t *>(in)[q];
    if (q == (int)(offsetof(KState, gm_k) / 4)) word = 0;
    reinterpret_cast<uint32_t *>(out)[q] = word;
  }
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * VB + t; i < n; i += (int64_t)gridDim.x * VB) {
    double acc[M];
#pragma unroll
    for (int c = 0; c < M; c++) acc[c] = 0.0;
#pragma unroll 4
    for (int j = 0; j < k; j++)
#pragma unroll
      for (int c = 0; c < M; c++) acc[c] += y[j] * (double)Vb[(int64_t)j * ldv + i * M + c];
    V wv[M];
#pragma unroll
    for (int c = 0; c < M; c++) wv[c] = (V)acc[c];
    if constexpr (!ADD) {
      w[i] = wv[0];
    } else if constexpr (NS == 0) {
      x[i] = (VXo)((double)x[i] + (double)wv[0]);
    } else {
      double B[NS * NS];
#pragma unroll
      for (int j = 0; j < NS * NS; j++) B[j] = binv[i * NS * NS + j];
      V zv[NS];
      node_solve<NS, V>(B, wv, zv);
#pragma unroll
      for (int c = 0; c < NS; c++) x[i * NS + c] = (VXo)((double)x[i * NS + c] + (double)zv[c]);
    }
  }
}
