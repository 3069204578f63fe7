// Sparse linear algebra for the Newton step on gfx950: CSR SpMV, fused BLAS-1
// with on-device reductions, BiCGStab and GMRES(m) whose scalars never leave
// the device, point/block-Jacobi and multicolour ILU(0) preconditioners, and
// FP32 Krylov inside FP64 iterative refinement.
//
// Replaces _solve_linear! (src/vfvm_linsolve.jl:6-61), i.e. what LinearSolve's
// KrylovJL_BICGSTAB / KrylovJL_GMRES with ILUZero / Jacobi / block
// preconditioners do for the reference.  All kernels are HBM-bandwidth bound.
//
// Conventions: the operator is the row-scaled Jacobian  Ahat = S A  with
// S = diag(1 / A_ii), which turns the 1e30 Dirichlet-penalty rows into unit
// rows before any FP32 cast (1e30^2 would overflow an FP32 dot product).
// Reductions: every reducing kernel writes one partial per block; the next kernel of the
// solver (vfvm_bicgstab.h, vfvm_gmres.h) or a one-block finalize kernel sums the partials
// in fixed order and runs a small "stage" that updates the solver scalars in device memory
// (no cross-block fences, deterministic sums).  Kernels of a finished solve return at
// entry, so the host can enqueue several iterations between status reads.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>
#include <cmath>

#include "vfvm_linalg.h"
#include "vfvm_wave.h"

namespace vfvm {

namespace {

constexpr int VB = 256;  // threads per block of vector kernels

__device__ __forceinline__ double block_sum(double v, double *sh) {
  // wave reduction then across the 4 waves of the block
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) r += sh[k];
  return r;  // valid in thread 0
}

// Every reducing kernel writes one partial per block (no fence, no atomics); a
// one-block finalize kernel launched next on the same stream sums the partials in
// fixed block order and runs the stage.  The kernel boundary orders the two.
template <int NR>
__device__ __forceinline__ void write_partials(const double (&v)[NR], double *partials) {
  __shared__ double sh[16];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    const double s = block_sum(v[k], sh);
    if (threadIdx.x == 0) partials[(size_t)k * gridDim.x + blockIdx.x] = s;
  }
}

__device__ __forceinline__ bool idle(const KState *st) { return st->done != 0; }

// stages that only store a total
enum { STAGE_RR = 100 };

template <int NR, int STAGE>
__global__ void __launch_bounds__(VB) k_finalize(const double *__restrict__ partials, int nparts, KState *st,
                                                 int check_idle) {
  if (check_idle && st->done) return;
  if (STAGE == STAGE_OMEGA && st->half) return;
  __shared__ double sh[16];
  double tot[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) {
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[(size_t)k * nparts + b];
    tot[k] = block_sum(acc, sh);
  }
  if (threadIdx.x != 0) return;
  if constexpr (STAGE == STAGE_RR) {
    st->rr = tot[0];
  } else {
    run_stage<STAGE>(st, tot);
  }
}

// ---------------------------------------------------------------- SpMV -----
// y = rowscale .* (A x)   (rowscale may be null), fused dots (w0, y) and, for
// NDOT = 2, (y, y) taken from the register value (stage runs in the last block).
// G lanes per row.
template <class VA, class VX, int G, int NDOT, int STAGE>
__global__ void __launch_bounds__(VB) k_spmv(int64_t nrows, const int32_t *__restrict__ rowptr,
                                             const int32_t *__restrict__ colind, const VA *__restrict__ val,
                                             const VX *__restrict__ x, VX *__restrict__ y,
                                             const double *__restrict__ rowscale, const VX *__restrict__ w0,
                                             const VX *__restrict__ w1, double *partials, KState *st) {
  if (st && idle(st)) return;
  if (STAGE == STAGE_OMEGA && st->half) return;
  const int lane = threadIdx.x & (G - 1);
  const int64_t rows_per_block = VB / G;
  double d0 = 0.0, d1 = 0.0;
  for (int64_t r = (int64_t)blockIdx.x * rows_per_block + threadIdx.x / G; r < nrows;
       r += (int64_t)gridDim.x * rows_per_block) {
    const int32_t k0 = rowptr[r], k1 = rowptr[r + 1];
    double acc = 0.0;
    for (int32_t k = k0 + lane; k < k1; k += G) acc += (double)val[k] * (double)x[colind[k]];
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
    if (lane == 0) {
      if (rowscale) acc *= rowscale[r];
      const VX yv = (VX)acc;
      y[r] = yv;
      if (NDOT >= 1) d0 += (double)w0[r] * (double)yv;
      if (NDOT >= 2) d1 += (double)yv * (double)yv;
    }
  }
  if constexpr (NDOT > 0) {
    double v[2] = {d0, d1};
    write_partials<2>(v, partials);
  }
}

// SELL-64 SpMV of the row-scaled operator: y = Ahat x, one lane per row.  A wave
// covers one slice of 64 rows, so each load of entry j (values and column indices)
// is one coalesced access; no row pointers, no cross-lane reduction.  Fused dots
// (w0, y), (y, y) and (w0, w0), the first NDOT of them.  Rows past nrows exist only as padding
// of the last slice.
// matrix stream loads; NT: non-temporal (the values and indices are read once per
// application, so they need not displace the gathered vector from the caches)
template <bool NT, class T>
__device__ __forceinline__ T ldm(const T *p) {
  if constexpr (NT)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

template <class VA, class VX, int NDOT, int STAGE, bool NT, class CI>
__global__ void __launch_bounds__(VB) k_sell_spmv(int64_t nrows, const int32_t *__restrict__ sptr,
                                                  const CI *__restrict__ col, const VA *__restrict__ val,
                                                  const VX *__restrict__ x, VX *__restrict__ y,
                                                  const VX *__restrict__ w0, double *partials, KState *st) {
  if (st && idle(st)) return;
  if (STAGE == STAGE_OMEGA && st->half) return;
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int64_t r = (int64_t)blockIdx.x * VB + threadIdx.x; r < nrows; r += (int64_t)gridDim.x * VB) {
    const int64_t sl = r >> 6;
    const int32_t p1 = sptr[sl + 1];
    double acc = 0.0;
#pragma unroll 4
    for (int32_t q = sptr[sl] + (int32_t)(r & 63); q < p1; q += 64)
      acc += (double)ldm<NT>(val + q) * (double)x[sell_column(ldm<NT>(col + q), r)];
    const VX yv = (VX)acc;
    y[r] = yv;
    if (NDOT >= 1) d0 += (double)w0[r] * (double)yv;
    if (NDOT >= 2) d1 += (double)yv * (double)yv;
    if (NDOT >= 3) d2 += (double)w0[r] * (double)w0[r];
  }
  if constexpr (NDOT == 1) {
    double v[1] = {d0};
    write_partials<1>(v, partials);
  } else if constexpr (NDOT == 2) {
    double v[2] = {d0, d1};
    write_partials<2>(v, partials);
  } else if constexpr (NDOT == 3) {
    double v[3] = {d0, d1, d2};
    write_partials<3>(v, partials);
  }
}

// residual of the refinement: y = S (b - A x) in FP64, ||y||^2 -> st->rr
template <int G>
__global__ void __launch_bounds__(VB) k_scaled_residual(int64_t nrows, const int32_t *__restrict__ rowptr,
                                                        const int32_t *__restrict__ colind,
                                                        const double *__restrict__ val, const double *__restrict__ x,
                                                        const double *__restrict__ b, const double *__restrict__ rowscale,
                                                        double *__restrict__ y, double *partials, KState *st) {
  const int lane = threadIdx.x & (G - 1);
  const int64_t rows_per_block = VB / G;
  double d0 = 0.0;
  for (int64_t r = (int64_t)blockIdx.x * rows_per_block + threadIdx.x / G; r < nrows;
       r += (int64_t)gridDim.x * rows_per_block) {
    const int32_t k0 = rowptr[r], k1 = rowptr[r + 1];
    double acc = 0.0;
    for (int32_t k = k0 + lane; k < k1; k += G) acc += val[k] * x[colind[k]];
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
    if (lane == 0) {
      const double v = rowscale[r] * (b[r] - acc);
      y[r] = v;
      d0 += v * v;
    }
  }
  double v[1] = {d0};
  write_partials<1>(v, partials);
}

// ---------------------------------------------------------- BiCGStab -------
// start: r = r0 = b (x = 0), (r, r) -> rho, rr; tolerance from ||b||
template <class V, class VB_>
__global__ void __launch_bounds__(VB) k_bicg_init(int64_t n, const VB_ *__restrict__ b, V *__restrict__ r,
                                                  V *__restrict__ r0, V *__restrict__ p, V *__restrict__ v,
                                                  double *partials, KState *st) {
  double d = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const V bv = (V)b[i];
    r[i] = bv;
    r0[i] = bv;
    p[i] = (V)0;
    v[i] = (V)0;
    d += (double)bv * (double)bv;
  }
  double vv[1] = {d};
  write_partials<1>(vv, partials);
}

template <class T>
__global__ void __launch_bounds__(VB) k_fill(int64_t n, T *__restrict__ x, T v) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) x[i] = v;
}

template <class TO, class TI>
__global__ void __launch_bounds__(VB) k_convert(int64_t n, const TI *__restrict__ a, TO *__restrict__ b) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) b[i] = (TO)a[i];
}

__global__ void __launch_bounds__(VB) k_negate(int64_t n, double *__restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) x[i] = -x[i];
}

// x64 += d32
template <class VD>
__global__ void __launch_bounds__(VB) k_add_correction(int64_t n, double *__restrict__ x, const VD *__restrict__ d,
                                                       double sign) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
    x[i] += sign * (double)d[i];
}

// -------------------------------------------------- scaling / conversion ---
// rowscale = 1 / A_ii (1 where the diagonal vanishes); optional Ahat32 = S A and
// block-Jacobi inverse blocks of Ahat
template <int NS>
__global__ void __launch_bounds__(VB) k_scale_rows(int64_t nnodes, const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ colind, const double *__restrict__ A,
                                                   const int32_t *__restrict__ dofdiag,
                                                   const int32_t *__restrict__ rbase, double *__restrict__ rowscale,
                                                   float *__restrict__ A32, double *__restrict__ A64,
                                                   double *__restrict__ binv) {
  for (int64_t K = (int64_t)blockIdx.x * VB + threadIdx.x; K < nnodes; K += (int64_t)gridDim.x * VB) {
    double sc[NS];
    double B[NS][NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
      const int64_t r = K * NS + i;
      const double d = A[dofdiag[r]];
      sc[i] = (d != 0.0 && d == d) ? 1.0 / d : 1.0;
      rowscale[r] = sc[i];
#pragma unroll
      for (int j = 0; j < NS; j++) B[i][j] = (i == j) ? 1.0 : 0.0;
      const int32_t k0 = rowptr[r], k1 = rowptr[r + 1];
      // scaled copies go to CSR positions, or to SELL-64 positions when rbase is given
      const int64_t q0 = rbase ? (int64_t)rbase[r] : (int64_t)k0;
      const int64_t qs = rbase ? 64 : 1;
      for (int32_t k = k0; k < k1; k++) {
        const double v = A[k] * sc[i];
        const int64_t q = q0 + (int64_t)(k - k0) * qs;
        if (A32) A32[q] = (float)v;
        if (A64) A64[q] = v;
        if (NS > 1 && binv) {
          const int32_t c = colind[k];
          if (c >= K * NS && c < K * NS + NS) B[i][c - K * NS] = v;
        }
      }
    }
    if (NS > 1 && binv) {
      // Gauss-Jordan inverse of the NS x NS block (no pivoting: unit diagonal after scaling)
      double I[NS][NS];
#pragma unroll
      for (int i = 0; i < NS; i++)
#pragma unroll
        for (int j = 0; j < NS; j++) I[i][j] = (i == j) ? 1.0 : 0.0;
#pragma unroll
      for (int c = 0; c < NS; c++) {
        const double piv = 1.0 / B[c][c];
#pragma unroll
        for (int j = 0; j < NS; j++) {
          B[c][j] *= piv;
          I[c][j] *= piv;
        }
#pragma unroll
        for (int i = 0; i < NS; i++) {
          if (i == c) continue;
          const double f = B[i][c];
#pragma unroll
          for (int j = 0; j < NS; j++) {
            B[i][j] -= f * B[c][j];
            I[i][j] -= f * I[c][j];
          }
        }
      }
#pragma unroll
      for (int i = 0; i < NS; i++)
#pragma unroll
        for (int j = 0; j < NS; j++) binv[K * NS * NS + i * NS + j] = I[i][j];
    }
  }
}

// -------------------------------------------------- multicolour ILU(0) ------
// LU values (permuted CSR) gathered from Ahat: lu[k] = S_row * A[src[k]]
template <class VL>
__global__ void __launch_bounds__(VB) k_ilu_gather(int64_t nnz, const int32_t *__restrict__ src,
                                                   const int32_t *__restrict__ srcrow, const double *__restrict__ A,
                                                   const double *__restrict__ rowscale, VL *__restrict__ lu) {
  for (int64_t k = (int64_t)blockIdx.x * VB + threadIdx.x; k < nnz; k += (int64_t)gridDim.x * VB)
    lu[k] = (VL)(A[src[k]] * rowscale[srcrow[k]]);
}

// factor the rows of one colour (rows of earlier colours are final)
template <class VL>
__global__ void __launch_bounds__(VB) k_ilu_factor(int32_t r0, int32_t r1, const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ colind, const int32_t *__restrict__ diag,
                                                   VL *__restrict__ lu) {
  const int32_t i = r0 + (int32_t)(blockIdx.x * VB + threadIdx.x);
  if (i >= r1) return;
  const int32_t k0 = rowptr[i], k1 = rowptr[i + 1], di = diag[i];
  for (int32_t k = k0; k < di; k++) {
    const int32_t c = colind[k];
    const double l = (double)lu[k] / (double)lu[diag[c]];
    lu[k] = (VL)l;
    // a_ij -= l * u_cj for j > c present in both rows (sorted merge)
    int32_t q = diag[c] + 1, qe = rowptr[c + 1], m = k + 1;
    while (q < qe && m < k1) {
      const int32_t cq = colind[q], cm = colind[m];
      if (cq == cm) {
        lu[m] = (VL)((double)lu[m] - l * (double)lu[q]);
        q++;
        m++;
      } else if (cq < cm) {
        q++;
      } else {
        m++;
      }
    }
  }
}

// factor values from CSR order to SELL-64 order (after each factorisation)
template <class VI, class VO>
__global__ void __launch_bounds__(VB) k_to_sell(int64_t nrows, const int32_t *__restrict__ rowptr,
                                                const int32_t *__restrict__ sptr, const VI *__restrict__ a,
                                                VO *__restrict__ as) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < nrows; i += (int64_t)gridDim.x * VB) {
    const int32_t k0 = rowptr[i], k1 = rowptr[i + 1];
    const int64_t q0 = (int64_t)sptr[i >> 6] + (i & 63);
    for (int32_t k = k0; k < k1; k++) as[q0 + (int64_t)(k - k0) * 64] = (VO)a[k];
  }
}

// Triangular solves of one colour on the SELL-64 factor: lanes are permuted rows
// i of the slices that overlap the colour's row range [r0, r1).  Lower part =
// entries before the diagonal position sdpos[i], upper part = entries after it
// (padding entries carry value 0 and the row's own column).
// LAST: the colour is the last one, whose rows have no upper part, so the backward
// solve of these rows (x = y / u_ii) is done here and the backward sweep starts at
// the previous colour
template <class VL, class V, bool LAST>
__global__ void __launch_bounds__(VB) k_ilu_lower_sell(int32_t r0, int32_t r1, const int32_t *__restrict__ sptr,
                                                       const int32_t *__restrict__ col,
                                                       const int32_t *__restrict__ sdpos, const VL *__restrict__ lu,
                                                       const int32_t *__restrict__ perm, const V *__restrict__ r,
                                                       V *__restrict__ y, V *__restrict__ z, const KState *st,
                                                       int skip_if_half) {
  if (st && idle(st)) return;
  if (st && skip_if_half && st->half) return;
  const int32_t i = (r0 & ~63) + (int32_t)(blockIdx.x * VB + threadIdx.x);
  if (i < r0 || i >= r1) return;
  const int32_t pi = perm[i];
  double acc = (double)r[pi];
  const int32_t q0 = sptr[i >> 6] + (i & 63), qd = q0 + 64 * sdpos[i];
  for (int32_t q = q0; q < qd; q += 64) acc -= (double)lu[q] * (double)y[col[q]];
  if constexpr (LAST) {
    const V xv = (V)(acc / (double)lu[qd]);
    y[i] = xv;
    z[pi] = xv;
  } else {
    y[i] = (V)acc;
  }
}

template <class VL, class V>
__global__ void __launch_bounds__(VB) k_ilu_upper_sell(int32_t r0, int32_t r1, const int32_t *__restrict__ sptr,
                                                       const int32_t *__restrict__ col,
                                                       const int32_t *__restrict__ sdpos, const VL *__restrict__ lu,
                                                       const int32_t *__restrict__ perm, V *__restrict__ y,
                                                       V *__restrict__ z, const KState *st, int skip_if_half) {
  if (st && idle(st)) return;
  if (st && skip_if_half && st->half) return;
  const int32_t i = (r0 & ~63) + (int32_t)(blockIdx.x * VB + threadIdx.x);
  if (i < r0 || i >= r1) return;
  const int32_t sl = i >> 6, q0 = sptr[sl] + (i & 63), qd = q0 + 64 * sdpos[i], qe = sptr[sl + 1];
  double acc = (double)y[i];
  for (int32_t q = qd + 64; q < qe; q += 64) acc -= (double)lu[q] * (double)y[col[q]];
  const V xv = (V)(acc / (double)lu[qd]);
  y[i] = xv;  // x overwrites y in place (later colours read x of their upper neighbours)
  z[perm[i]] = xv;
}

// x += z
template <class VXo, class V>
__global__ void __launch_bounds__(VB) k_axpy_out(int64_t n, VXo *__restrict__ x, const V *__restrict__ z) {
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
    x[i] = (VXo)((double)x[i] + (double)z[i]);
}

// Newton update: U -= damp * dU ; ||dU||_inf, ||U||_1 (src/vfvm_solver.jl:116-135)
__global__ void __launch_bounds__(VB) k_newton_update(int64_t n, double *__restrict__ U, const double *__restrict__ dU,
                                                      double damp, double *partials, unsigned *ticket,
                                                      double *out /* [0] = ||dU||_inf, [1] = ||U||_1 */) {
  double m = 0.0, s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
    const double d = dU[i];
    const double u = U[i] - damp * d;
    U[i] = u;
    m = nanmax(m, fabs(d));
    s += fabs(u);
  }
  // block max and sum -> partials [sum | max]; k_newton_finalize combines them
  __shared__ double shm[16];
  const double bs = block_sum(s, shm);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = nanmax(m, __shfl_xor(m, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double bm = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) bm = nanmax(bm, shm[k]);
    partials[blockIdx.x] = bs;
    partials[(size_t)gridDim.x + blockIdx.x] = bm;
  }
}

// out[0] = max of the max partials, out[1] = sum of the sum partials (one block)
__global__ void __launch_bounds__(VB) k_newton_finalize(const double *__restrict__ partials, int nparts,
                                                        double *__restrict__ out_max, double *__restrict__ out_sum) {
  const bool with_max = out_max != nullptr;
  __shared__ double sh[16];
  double acc = 0.0, mx = 0.0;
  for (int b = threadIdx.x; b < nparts; b += blockDim.x) {
    acc += partials[b];
    if (with_max) mx = nanmax(mx, partials[(size_t)nparts + b]);
  }
  acc = block_sum(acc, sh);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = nanmax(mx, __shfl_xor(mx, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m2 = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) m2 = nanmax(m2, sh[k]);
    if (with_max) *out_max = m2;
    *out_sum = acc;
  }
}

// ||U||_1
__global__ void __launch_bounds__(VB) k_norm1(int64_t n, const double *__restrict__ U, double *partials, unsigned *ticket,
                                              double *out) {
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) s += fabs(U[i]);
  __shared__ double sh[16];
  const double bs = block_sum(s, sh);
  if (threadIdx.x == 0) partials[blockIdx.x] = bs;
}

// max |a - b| (the step-size control's update norm); partials [0 | max] for k_newton_finalize
__global__ void __launch_bounds__(VB) k_maxdiff(int64_t n, const double *__restrict__ a, const double *__restrict__ b,
                                                double *partials) {
  double m = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
    m = nanmax(m, fabs(a[i] - b[i]));
  __shared__ double shm[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = nanmax(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) shm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double bm = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) bm = nanmax(bm, shm[k]);
    partials[blockIdx.x] = 0.0;
    partials[(size_t)gridDim.x + blockIdx.x] = bm;
  }
}

#include "vfvm_bicgstab.h"
#include "vfvm_bicgone.h"
#include "vfvm_gmres.h"

// CSC gather: out[k] = J[perm[k]]
__global__ void __launch_bounds__(VB) k_gather(int64_t n, const int32_t *__restrict__ perm, const double *__restrict__ J,
                                               double *__restrict__ out) {
  for (int64_t k = (int64_t)blockIdx.x * VB + threadIdx.x; k < n; k += (int64_t)gridDim.x * VB) out[k] = J[perm[k]];
}

}  // namespace

// ============================================================================ host side

static unsigned grid_for(int64_t n, int per_thread_rows = 1) {
  int64_t b = (n + (int64_t)VB * per_thread_rows - 1) / ((int64_t)VB * per_thread_rows);
  if (b < 1) b = 1;
  if (b > MAX_RED_BLOCKS) b = MAX_RED_BLOCKS;
  return (unsigned)b;
}

// Blocks of the vector updates of BiCGStab.  Each of them sums all partials of the product
// before it, and its own partials are summed by every block of the product after it, so fewer
// blocks than a pure stream wants: on 129^3 rows in FP32 the update of x and r takes 21.9 us
// with 2048 blocks, 16.7 with 1024 and 16.1 with 512, and the product after it 20.5, 19.6 and
// 18.6.  The products keep one row per thread as far as it goes (13.4 us with 1024 blocks and
// 18.1 with 512, against 11.5).
constexpr unsigned FOLD_BLOCKS = 512;
// Blocks up to which every block of GMRES sums the previous kernel's partial dot products itself
// (up to 64 sums; beyond, a launch with one block per sum goes before).  A step took, folded and
// summed, 24.4 and 27.6 us with 66 blocks, 25.8 and 27.6 with 128, 32.8 and 29.3 with 259.
constexpr int GM_FOLD = 128;
static unsigned fold_blocks(int64_t n) { return std::min(grid_for(n), FOLD_BLOCKS); }

void LinearSolver::setup(const LinSetup &ls, hipStream_t s) {
  L = ls;
  stream = s;
  int64_t n = L.ndof;
  st.alloc(4);
  for (int i = 0; i < 2; i++) {
    if (!hst[i]) VFVM_HIP_CHECK(hipHostMalloc((void **)&hst[i], sizeof(KState), hipHostMallocDefault));
    if (!sev[i]) VFVM_HIP_CHECK(hipEventCreateWithFlags(&sev[i], hipEventDisableTiming));
  }
  partials.alloc((size_t)4 * MAX_RED_BLOCKS);
  part_alpha.alloc((size_t)2 * MAX_RED_BLOCKS);
  part_omega.alloc((size_t)6 * MAX_RED_BLOCKS);
  part_rho.alloc((size_t)4 * MAX_RED_BLOCKS);
  rowscale.alloc((size_t)n);
  // the ILU structure may have been rebuilt in another ordering: factor copies are
  // reallocated, so that the SELL padding of the new layout starts at zero
  ilu_ready = false;
  ilu_sell_ready[0] = ilu_sell_ready[1] = false;
  ilu32s.release();
  ilu64s.release();
  hipLaunchKernelGGL((k_fill<unsigned char>), dim3(grid_for((int64_t)(4 * sizeof(KState)))), dim3(VB), 0, s,
                     (int64_t)(4 * sizeof(KState)), reinterpret_cast<unsigned char *>(st.p), (unsigned char)0);
  hipLaunchKernelGGL((k_fill<double>), dim3(grid_for(4 * MAX_RED_BLOCKS)), dim3(VB), 0, s,
                     (int64_t)4 * MAX_RED_BLOCKS, partials.p, 0.0);
  VFVM_HIP_CHECK(hipGetLastError());
}

template <class V>
void LinearSolver::Work<V>::alloc(int64_t n, int nvec) {
  if (n == this->n && nvec <= (int)vecs.size()) return;
  vecs.clear();
  vecs.resize(nvec);
  for (auto &v : vecs) v.alloc((size_t)n);
  this->n = n;
}

void LinearSolver::ensure_work(int precision, int krylov, int m) {
  int64_t n = L.ndof;
  int nv = krylov == VFVM_KRYLOV_GMRES ? 4 : 9;
  // SELL-64 operator values: padding entries must hold 0, so a new buffer is cleared once
  if (precision == VFVM_PREC_FP32_REFINE) {
    w32.alloc(n, nv);
    if (A32.n != (size_t)L.sell_nnz) {
      A32.alloc((size_t)L.sell_nnz);
      hipLaunchKernelGGL((k_fill<float>), dim3(grid_for(L.sell_nnz)), dim3(VB), 0, stream, L.sell_nnz, A32.p, 0.0f);
    }
  } else {
    w64.alloc(n, nv);
    if (A64s.n != (size_t)L.sell_nnz) {
      A64s.alloc((size_t)L.sell_nnz);
      hipLaunchKernelGGL((k_fill<double>), dim3(grid_for(L.sell_nnz)), dim3(VB), 0, stream, L.sell_nnz, A64s.p, 0.0);
    }
  }
  if (krylov == VFVM_KRYLOV_GMRES) {
    if (precision == VFVM_PREC_FP32_REFINE)
      vbasis32.alloc((size_t)n * (m + 1));
    else
      vbasis64.alloc((size_t)n * (m + 1));
    gmH.alloc((size_t)(m + 1) * m);
    gmh1.alloc((size_t)m + 2);
    gmh2.alloc((size_t)m + 2);
    gmcs.alloc((size_t)m);
    gmsn.alloc((size_t)m);
    gmg.alloc((size_t)m + 2);
    gmsum.alloc((size_t)m + 2);
    gmpart.alloc((size_t)(m + 2) * MAX_RED_BLOCKS);
    gmpart2.alloc((size_t)(m + 2) * GM_FOLD);
  }
}

// scaling, FP32 copy and preconditioner set-up for the current Jacobian values
void LinearSolver::prepare(const double *J, const vfvm_control_t &c, bool refactor) {
  if (fp32_off && c.precision == VFVM_PREC_FP32_REFINE) {  // FP32 switched off: the FP64 operator
    vfvm_control_t c64 = c;
    c64.precision = VFVM_PREC_FP64;
    prepare(J, c64, refactor);
    return;
  }
  ensure_work(c.precision, c.krylov, c.gmres_restart);
  const bool fp32 = c.precision == VFVM_PREC_FP32_REFINE;
  const bool blk = c.precon == VFVM_PRECON_BLOCKJACOBI && L.nspec > 1;
  if (blk) binv.alloc((size_t)L.nnodes * L.nspec * L.nspec);
  unsigned g = grid_for(L.nnodes);
  float *a32 = fp32 ? A32.p : nullptr;
  double *a64 = fp32 ? nullptr : A64s.p;
  double *bi = blk ? binv.p : nullptr;
  switch (L.nspec) {
    case 1:
      hipLaunchKernelGGL((k_scale_rows<1>), dim3(g), dim3(VB), 0, stream, L.nnodes, L.rowptr, L.colind, J, L.dofdiag,
                         L.sell_rbase, rowscale.p, a32, a64, bi);
      break;
    case 2:
      hipLaunchKernelGGL((k_scale_rows<2>), dim3(g), dim3(VB), 0, stream, L.nnodes, L.rowptr, L.colind, J, L.dofdiag,
                         L.sell_rbase, rowscale.p, a32, a64, bi);
      break;
    case 3:
      hipLaunchKernelGGL((k_scale_rows<3>), dim3(g), dim3(VB), 0, stream, L.nnodes, L.rowptr, L.colind, J, L.dofdiag,
                         L.sell_rbase, rowscale.p, a32, a64, bi);
      break;
  }
  VFVM_HIP_CHECK(hipGetLastError());
  if (c.precon == VFVM_PRECON_AMG) {
    if (L.nspec != 1) throw Error(VFVM_ERR_ARG, "the AMG preconditioner is provided for scalar systems");
    if (!amg.built()) {
      if (!L.h_rowptr || !L.h_colind) throw Error(VFVM_ERR_ARG, "AMG needs the host pattern");
      AmgMember m;
      m.n = L.ndof;
      m.rowptr = L.h_rowptr;
      m.colind = L.h_colind;
      amg.build({m}, nullptr, stream);
    }
    // the hierarchy of the first Newton step is reused like an ILU(0) factor
    // (src/vfvm_solvercontrol.jl:123-131); the level-0 operator is always the current one
    if (refactor || !amg.ready()) amg.setup(L.rowptr, L.colind, L.dofdiag, J, rowscale.p, stream);
    amg.refresh_fine(L.rowptr, J, rowscale.p, false, stream);  // both precisions: FP32 may fall back
  }
  const bool ilu = c.precon == VFVM_PRECON_ILU0 || c.precon == VFVM_PRECON_ILU0_NATURAL;
  if (ilu && (refactor || !ilu_ready)) {
    if (!L.ilu) throw Error(VFVM_ERR_ARG, "ILU(0) needs its level structure (build_ilu)");
    const IluStruct &I = *L.ilu;
    // the factorisation runs in FP64 for both precisions (pivots of non-M-matrices can
    // shrink); each precision's solve gets a SELL-64 copy of the factor
    ilu64.alloc((size_t)L.nnz);
    hipLaunchKernelGGL((k_ilu_gather<double>), dim3(grid_for(L.nnz)), dim3(VB), 0, stream, L.nnz, I.src, I.srcrow, J,
                       rowscale.p, ilu64.p);
    for (int c0 = 0; c0 < I.ncolors; c0++) {
      int32_t r0 = I.cptr[c0], r1 = I.cptr[c0 + 1];
      if (r1 > r0)
        hipLaunchKernelGGL((k_ilu_factor<double>), dim3((r1 - r0 + VB - 1) / VB), dim3(VB), 0, stream, r0, r1,
                           I.rowptr, I.colind, I.diag, ilu64.p);
    }
    ilu_ready = true;
    ilu_sell_ready[0] = ilu_sell_ready[1] = false;
  }
  if (red_black(c)) prepare_red_black(J, fp32);
  else if (ilu && !ilu_sell_ready[fp32 ? 0 : 1]) {
    const IluStruct &I = *L.ilu;
    if (fp32) {
      if (ilu32s.n != (size_t)I.snnz) {
        ilu32s.alloc((size_t)I.snnz);
        hipLaunchKernelGGL((k_fill<float>), dim3(grid_for(I.snnz)), dim3(VB), 0, stream, I.snnz, ilu32s.p, 0.0f);
      }
      hipLaunchKernelGGL((k_to_sell<double, float>), dim3(grid_for(L.ndof)), dim3(VB), 0, stream, L.ndof, I.rowptr,
                         I.sptr, (const double *)ilu64.p, ilu32s.p);
    } else {
      if (ilu64s.n != (size_t)I.snnz) {
        ilu64s.alloc((size_t)I.snnz);
        hipLaunchKernelGGL((k_fill<double>), dim3(grid_for(I.snnz)), dim3(VB), 0, stream, I.snnz, ilu64s.p, 0.0);
      }
      hipLaunchKernelGGL((k_to_sell<double, double>), dim3(grid_for(L.ndof)), dim3(VB), 0, stream, L.ndof,
                         I.rowptr, I.sptr, (const double *)ilu64.p, ilu64s.p);
    }
    ilu_sell_ready[fp32 ? 0 : 1] = true;
    VFVM_HIP_CHECK(hipGetLastError());
  }
}

template <class V>
const V *LinearSolver::precond(const V *r, V *z, KState *stp, int skip_if_half, const vfvm_control_t &c) {
  if (c.precon == VFVM_PRECON_ILU0 || c.precon == VFVM_PRECON_ILU0_NATURAL) {
    const IluStruct &I = *L.ilu;
    const V *lu = nullptr;
    if constexpr (sizeof(V) == 4) lu = ilu32s.p;
    else lu = ilu64s.p;
    V *y = iluy_ptr<V>();
    auto blocks = [](int32_t r0, int32_t r1) { return (unsigned)((r1 - (r0 & ~63) + VB - 1) / VB); };
    for (int c0 = 0; c0 < I.ncolors; c0++) {
      int32_t r0 = I.cptr[c0], r1 = I.cptr[c0 + 1];
      if (r1 <= r0) continue;
      if (c0 == I.ncolors - 1)
        hipLaunchKernelGGL((k_ilu_lower_sell<V, V, true>), dim3(blocks(r0, r1)), dim3(VB), 0, stream, r0, r1, I.sptr,
                           I.scol, I.sdpos, lu, I.perm, r, y, z, stp, skip_if_half);
      else
        hipLaunchKernelGGL((k_ilu_lower_sell<V, V, false>), dim3(blocks(r0, r1)), dim3(VB), 0, stream, r0, r1, I.sptr,
                           I.scol, I.sdpos, lu, I.perm, r, y, z, stp, skip_if_half);
    }
    for (int c0 = I.ncolors - 2; c0 >= 0; c0--) {
      int32_t r0 = I.cptr[c0], r1 = I.cptr[c0 + 1];
      if (r1 > r0)
        hipLaunchKernelGGL((k_ilu_upper_sell<V, V>), dim3(blocks(r0, r1)), dim3(VB), 0, stream, r0, r1, I.sptr, I.scol,
                           I.sdpos, lu, I.perm, y, z, stp, skip_if_half);
    }
    return z;
  }
  if (c.precon == VFVM_PRECON_AMG) {
    amg.apply<V>(r, z, stp, skip_if_half, stream, L.probe);
    return z;
  }
  // point Jacobi on the row-scaled operator is the identity; node solves are part of the
  // kernels that use them
  return r;
}

template <class V>
V *LinearSolver::iluy_ptr() {
  if constexpr (sizeof(V) == 4) {
    iluy32.alloc((size_t)L.ndof);
    return iluy32.p;
  } else {
    iluy64.alloc((size_t)L.ndof);
    return iluy64.p;
  }
}

// y = Ahat x with optional fused dots (partials to `part`), in the working precision V
template <class V, int NDOT, int STAGE>
void LinearSolver::apply_op(const V *x, V *y, const V *w0, KState *stp, double *part) {
  const unsigned g = grid_for(L.ndof);
  const int kid = sizeof(V) == 4 ? VFVM_KERNEL_SPMV32 : VFVM_KERNEL_SPMV64;
  if (L.probe) L.probe->before(kid, stream);
  auto go = [&](auto ntc, const auto *col) {
    constexpr bool NT = decltype(ntc)::value;
    using CI = std::remove_const_t<std::remove_pointer_t<decltype(col)>>;
    if constexpr (sizeof(V) == 4)
      VFVM_LAUNCH((k_sell_spmv<float, V, NDOT, STAGE, NT, CI>), dim3(g), dim3(VB), 0, stream, L.ndof, L.sell_ptr, col,
                  (const float *)A32.p, x, y, w0, part, stp);
    else
      VFVM_LAUNCH((k_sell_spmv<double, V, NDOT, STAGE, NT, CI>), dim3(g), dim3(VB), 0, stream, L.ndof, L.sell_ptr,
                  col, (const double *)A64s.p, x, y, w0, part, stp);
  };
  const bool nt = sell_nt[sizeof(V) == 4 ? 0 : 1];
  if (L.sell_off16 && sell16) {
    if (nt)
      go(std::true_type(), L.sell_off16);
    else
      go(std::false_type(), L.sell_off16);
  } else {
    if (nt)
      go(std::true_type(), L.sell_col);
    else
      go(std::false_type(), L.sell_col);
  }
  if (L.probe) L.probe->after(kid, stream, L.ndof, L.nnz);
}

void LinearSolver::apply_plain(bool fp32, const double *J, const void *x, void *y) {
  (void)J;
  if (fp32)
    apply_op<float, 0, STAGE_NONE>((const float *)x, (float *)y, (const float *)nullptr, nullptr, nullptr);
  else
    apply_op<double, 0, STAGE_NONE>((const double *)x, (double *)y, (const double *)nullptr, nullptr, nullptr);
  VFVM_HIP_CHECK(hipGetLastError());
}

void LinearSolver::read_state(KState &h) {
  VFVM_HIP_CHECK(hipMemcpyAsync(&h, st.p, sizeof(KState), hipMemcpyDeviceToHost, stream));
  VFVM_HIP_CHECK(hipStreamSynchronize(stream));
}

// values of the two-colour form from J and the row scaling, in the solve precision
void LinearSolver::prepare_red_black(const double *J, bool fp32) {
  const RedBlack &R = L.ilu->rb;
  auto go = [&](auto &e, auto &f, auto &d) {
    using V = std::remove_reference_t<decltype(*e.p)>;
    e.alloc((size_t)R.e.nval);
    f.alloc((size_t)R.f.nval);
    d.alloc((size_t)R.nb);
    hipLaunchKernelGGL((k_rb_values<V, false>), dim3((unsigned)((R.nr + VB - 1) / VB)), dim3(VB), 0, stream, R.nr,
                       R.e.sptr, R.e.src, (const int32_t *)nullptr, R.e.row, L.colind, L.dofdiag, J,
                       (const double *)rowscale.p, e.p, (V *)nullptr);
    hipLaunchKernelGGL((k_rb_values<V, true>), dim3((unsigned)((R.nb + VB - 1) / VB)), dim3(VB), 0, stream, R.nb,
                       R.f.sptr, R.f.src, R.tsrc, R.f.row, L.colind, L.dofdiag, J, (const double *)rowscale.p, f.p,
                       d.p);
  };
  if (fp32)
    go(rb_e32, rb_f32, rb_d32);
  else
    go(rb_e64, rb_f64, rb_d64);
  VFVM_HIP_CHECK(hipGetLastError());
}

// rows up to which the point Jacobi form also forms the search direction inside the product
// (three gathered vectors instead of one, but one launch less).  An iteration took, fused and
// not, 16.2 and 20.0 us at 33^2 rows, 17.9 and 19.6 us at 257^2 (also 33^3: 17.9 and 20.1), and
// the same from 363^2 on (23.9 and 24.2; 51^3: 29.1 and 29.6; 513^2: 31.9 and 31.8).
constexpr int64_t FUSE_P_ROWS = 1 << 17;

// Matrix entries (with two colours: of the black rows) up to which one block solves the whole
// system.  An iteration takes, in one block and in launches: point Jacobi 4.6 and 12 us at 33^2 rows
// (7,700 entries, copied to LDS), 7.6 and 12 at 45^2, 10.1 and 12 at 55^2 (21,500), 12.7 and 12 at
// 64^2 (29,000), 23.6 and 15.9 at 16^3; two-colour ILU(0) 3.9 and 15 us at 33^2 rows, 6.1 and 20 at
// 45^2, 14 and 24 at 55^2, 20.7 and 24 at 71^2 (10,200), 29 and 24 at 80^2 (13,000).
constexpr int64_t ONE_ENTRIES = 22000, ONE_ENTRIES_RB = 11000;

// The launches of BiCGStab in the form that fits the preconditioner.  init() sets the start
// state (slot 0 and the partials of (r, r)), iterate(first) queues one iteration, report() the
// host's copy of the state after it.
template <class V, class VXo>
struct LinearSolver::Bicg {
  LinearSolver &S;
  const vfvm_control_t &c;
  VXo *x;
  hipStream_t st;
  int64_t n;
  unsigned g, gv;  // blocks of the products, of the vector updates
  V *r, *r0, *p, *v, *s, *t, *ph, *sh, *xx;
  KState *k;
  const bool rb, blk, plain;
  int nrho = 0;  // partials of the last (r0, r), (r, r)
  Bicg(LinearSolver &ls, const vfvm_control_t &cc, VXo *xo)
      : S(ls), c(cc), x(xo), st(ls.stream), n(ls.L.ndof), g(grid_for(ls.L.ndof)), gv(fold_blocks(ls.L.ndof)), k(ls.st.p), rb(ls.red_black(cc)),
        blk(cc.precon == VFVM_PRECON_BLOCKJACOBI && ls.L.nspec > 1),
        plain(cc.precon == VFVM_PRECON_JACOBI || (cc.precon == VFVM_PRECON_BLOCKJACOBI && ls.L.nspec == 1)) {
    Work<V> &W = S.work<V>();
    r = W.vecs[0].p, r0 = W.vecs[1].p, p = W.vecs[2].p, v = W.vecs[3].p, s = W.vecs[4].p, t = W.vecs[5].p,
    ph = W.vecs[6].p, sh = W.vecs[7].p, xx = W.vecs[8].p;
  }
  // matrix values, column indices and their load form of the SELL-64 operator
  template <class F>
  void with_operator(F &&f) {
    const V *val;
    if constexpr (sizeof(V) == 4) val = S.A32.p;
    else val = S.A64s.p;
    const bool nt = S.sell_nt[sizeof(V) == 4 ? 0 : 1];
    if (S.L.sell_off16 && S.sell16) {
      if (nt) f(std::true_type(), S.L.sell_off16, val);
      else f(std::false_type(), S.L.sell_off16, val);
    } else {
      if (nt) f(std::true_type(), S.L.sell_col, val);
      else f(std::false_type(), S.L.sell_col, val);
    }
  }
  template <class VBin>
  void init(const VBin *b) {
    if (rb) {
      const RedBlack &R = S.L.ilu->rb;
      hipLaunchKernelGGL((k_rb_init<V, VBin>), dim3(gv), dim3(VB), 0, st, R.nr, n, R.e.row, R.f.row, b, r, r0, p, v, xx,
                         S.part_rho.p);
    } else {
      hipLaunchKernelGGL((k_fill<VXo>), dim3(g), dim3(VB), 0, st, n, x, (VXo)0);
      hipLaunchKernelGGL((k_bicg_init<V, VBin>), dim3(gv), dim3(VB), 0, st, n, b, r, r0, p, v, S.part_rho.p, k);
    }
    nrho = (int)gv;
  }
  void iterate(bool first) {
    if (first)
      iterate_at(std::integral_constant<int, STAGE_INIT>());
    else
      iterate_at(std::integral_constant<int, STAGE_XR>());
  }
  template <class ST>
  void iterate_at(ST) {
    constexpr int STAGE = ST::value;
    KState *k0 = k + SLOT_RHO, *k1 = k + SLOT_BETA, *k2 = k + SLOT_ALPHA;
    const double *rho = S.part_rho.p, *al = S.part_alpha.p, *om = S.part_omega.p;
    const int kid = sizeof(V) == 4 ? VFVM_KERNEL_SPMV32 : VFVM_KERNEL_SPMV64;
    if (rb) {
      const RedBlack &R = S.L.ilu->rb;
      if (R.e.off && R.f.off)
        iterate_rb<STAGE, int16_t>(R.e.off, R.f.off);
      else
        iterate_rb<STAGE, int32_t>(R.e.col, R.f.col);
    } else if (plain) {
      const bool fuse = n <= FUSE_P_ROWS;
      with_operator([&](auto ntc, const auto *col, const V *val) {
        constexpr bool NT = decltype(ntc)::value;
        using CI = std::remove_const_t<std::remove_pointer_t<decltype(col)>>;
        if (fuse) {
          hipLaunchKernelGGL((k_bicg_pv<V, STAGE, NT, CI>), dim3(g), dim3(VB), 0, st, n, S.L.sell_ptr, col, val, r, p,
                             v, ph, s, r0, rho, nrho, k0, k1, S.part_alpha.p);
          std::swap(p, ph);
          std::swap(v, s);
        } else {
          hipLaunchKernelGGL((k_bicg_p<V, STAGE, 0>), dim3(gv), dim3(VB), 0, st, n, r, p, v, (const double *)nullptr,
                             (V *)nullptr, rho, nrho, k0, k1);
          S.apply_op<V, 1, STAGE_NONE>(p, v, r0, k1, S.part_alpha.p);
        }
        if (S.L.probe) S.L.probe->before(kid, st);
        VFVM_LAUNCH((k_bicg_st<V, NT, CI>), dim3(g), dim3(VB), 0, st, n, S.L.sell_ptr, col, val, r, v, t, al, (int)g,
                    k1, k2, S.part_omega.p);
        if (S.L.probe) S.L.probe->after(kid, st, S.L.ndof, S.L.nnz);
      });
      hipLaunchKernelGGL((k_bicg_xr<V, VXo, STAGE_SOMEGA, true>), dim3(gv), dim3(VB), 0, st, n, x, p, (const V *)nullptr,
                         (const V *)nullptr, v, t, r, r0, om, (int)g, k2, k0, S.part_rho.p);
    } else if (blk) {
      auto go = [&](auto ns) {
        constexpr int NS = decltype(ns)::value;
        const unsigned gn = fold_blocks(S.L.nnodes);
        hipLaunchKernelGGL((k_bicg_p<V, STAGE, NS>), dim3(gn), dim3(VB), 0, st, S.L.nnodes, r, p, v,
                           (const double *)S.binv.p, ph, rho, nrho, k0, k1);
        S.apply_op<V, 1, STAGE_NONE>(ph, v, r0, k1, S.part_alpha.p);
        hipLaunchKernelGGL((k_bicg_s<V, NS, false>), dim3(gn), dim3(VB), 0, st, S.L.nnodes, r, v, s,
                           (const double *)S.binv.p, sh, al, (int)g, k1, k2, (double *)nullptr);
      };
      if (S.L.nspec == 2) go(std::integral_constant<int, 2>());
      else go(std::integral_constant<int, 3>());
      S.apply_op<V, 3, STAGE_NONE>(sh, t, s, k2, S.part_omega.p);
      hipLaunchKernelGGL((k_bicg_xr<V, VXo, STAGE_SOMEGA, false>), dim3(gv), dim3(VB), 0, st, n, x, ph, sh, s, v, t, r,
                         r0, om, (int)g, k2, k0, S.part_rho.p);
    } else {
      // a costly preconditioner: its second application and product are skipped when the half
      // step has converged, which takes a launch to decide
      hipLaunchKernelGGL((k_bicg_p<V, STAGE, 0>), dim3(gv), dim3(VB), 0, st, n, r, p, v, (const double *)nullptr,
                         (V *)nullptr, rho, nrho, k0, k1);
      const V *php = S.precond<V>(p, ph, k1, 0, c);
      S.apply_op<V, 1, STAGE_NONE>(php, v, r0, k1, S.part_alpha.p);
      hipLaunchKernelGGL((k_bicg_s<V, 0, true>), dim3(gv), dim3(VB), 0, st, n, r, v, s, (const double *)nullptr,
                         (V *)nullptr, al, (int)g, k1, k2, S.partials.p);
      hipLaunchKernelGGL((k_finalize<1, STAGE_SNORM>), dim3(1), dim3(VB), 0, st, (const double *)S.partials.p, (int)gv,
                         k2, 1);
      const V *shp = S.precond<V>(s, sh, k2, 1, c);
      S.apply_op<V, 2, STAGE_OMEGA>(shp, t, s, k2, S.part_omega.p);
      hipLaunchKernelGGL((k_bicg_xr<V, VXo, STAGE_OMEGA, false>), dim3(gv), dim3(VB), 0, st, n, x, php, shp, s, v, t, r,
                         r0, om, (int)g, k2, k0, S.part_rho.p);
    }
    nrho = (int)gv;
  }
  template <class CI>
  RbMat<V, CI> rb_matrix(const CI *ec, const CI *fc) {
    const RedBlack &R = S.L.ilu->rb;
    RbMat<V, CI> A;
    A.nr = R.nr;
    A.nb = R.nb;
    A.es = R.e.sptr;
    A.fs = R.f.sptr;
    A.ec = ec;
    A.fc = fc;
    if constexpr (sizeof(V) == 4) {
      A.ev = S.rb_e32.p;
      A.fv = S.rb_f32.p;
      A.d = S.rb_d32.p;
    } else {
      A.ev = S.rb_e64.p;
      A.fv = S.rb_f64.p;
      A.d = S.rb_d64.p;
    }
    return A;
  }
  // whole solve in one block: point Jacobi, two-colour ILU(0)
  bool one_block() const {
    if (rb) {
      const RedBlack &R = S.L.ilu->rb;
      return std::max(R.nr, R.nb) <= 3 * ONE_T && R.f.nval <= ONE_ENTRIES_RB;
    }
    return plain && n <= 3 * ONE_T && S.L.sell_nnz <= ONE_ENTRIES;
  }
  template <class VBin>
  void solve_one(const VBin *b, const KState &h, int every, int stag, KState *pinned) {
    auto go = [&](auto rc, auto cc) {
      constexpr int R = decltype(rc)::value;
      constexpr bool COPY = decltype(cc)::value;
      if (rb) {
        const RedBlack &B = S.L.ilu->rb;
        auto launch = [&](const auto *ec, const auto *fc) {
          using CI = std::remove_const_t<std::remove_pointer_t<decltype(ec)>>;
          hipLaunchKernelGGL((k_rb_one<V, VBin, VXo, CI, R, COPY>), dim3(1), dim3(ONE_T), 0, st, rb_matrix<CI>(ec, fc),
                             B.e.row, B.f.row, b, x, xx, r0, h.rtol, h.atol, h.maxit, every, stag, pinned);
        };
        if (B.e.off && B.f.off) launch(B.e.off, B.f.off);
        else launch(B.e.col, B.f.col);
      } else {
        with_operator([&](auto, const auto *col, const V *val) {
          using CI = std::remove_const_t<std::remove_pointer_t<decltype(col)>>;
          const OneMat<V, CI> A{S.L.sell_ptr, col, val};
          hipLaunchKernelGGL((k_bicg_one<V, VBin, VXo, CI, R, COPY>), dim3(1), dim3(ONE_T), 0, st, (int)n, A, b, x, r0,
                             h.rtol, h.atol, h.maxit, every, stag, pinned);
        });
      }
    };
    int64_t m = n, bytes;
    const int vs = sizeof(V);
    if (rb) {
      const RedBlack &R = S.L.ilu->rb;
      const int cs = R.e.off && R.f.off ? 2 : 4;
      m = std::max(R.nr, R.nb);
      bytes = one_bytes(R.nr, R.e.nval, vs, cs) + one_bytes(R.nb, R.f.nval, vs, cs);
    } else {
      bytes = one_bytes(n, S.L.sell_nnz, vs, S.L.sell_off16 && S.sell16 ? 2 : 4);
    }
    auto rows = [&](auto cc) {
      if (m <= ONE_T) go(std::integral_constant<int, 1>(), cc);
      else if (m <= 2 * ONE_T) go(std::integral_constant<int, 2>(), cc);
      else go(std::integral_constant<int, 3>(), cc);
    };
    if (bytes <= ONE_LDS) rows(std::true_type());
    else rows(std::false_type());
  }
  template <int STAGE, class CI>
  void iterate_rb(const CI *ec, const CI *fc) {
    const RedBlack &R = S.L.ilu->rb;
    const RbMat<V, CI> A = rb_matrix<CI>(ec, fc);
    KState *k0 = k + SLOT_RHO, *k1 = k + SLOT_BETA, *k2 = k + SLOT_ALPHA;
    const unsigned gr = grid_for(R.nr), gb = grid_for(R.nb);
    const int np = (int)(gr + gb);
    double *al = S.part_alpha.p, *om = S.part_omega.p;
    hipLaunchKernelGGL((k_rb_p_black<V, STAGE, CI>), dim3(gb), dim3(VB), 0, st, A, r, p, v, ph,
                       (const double *)S.part_rho.p, nrho, k0, k1);
    hipLaunchKernelGGL((k_rb_p_red<V, CI>), dim3(gr), dim3(VB), 0, st, A, r, p, ph, r0, k1, al, np);
    hipLaunchKernelGGL((k_rb_v<V, CI>), dim3(gb), dim3(VB), 0, st, A, ph, v, r0, k1, al, np, (int)gr);
    hipLaunchKernelGGL((k_rb_s_black<V, CI>), dim3(gb), dim3(VB), 0, st, A, r, p, v, sh, (const double *)al, np, k1,
                       k2);
    hipLaunchKernelGGL((k_rb_s_red<V, CI>), dim3(gr), dim3(VB), 0, st, A, r, p, sh, k2, om, np);
    hipLaunchKernelGGL((k_rb_t<V, CI>), dim3(gb), dim3(VB), 0, st, A, r, v, sh, t, k2, om, np, (int)gr);
    hipLaunchKernelGGL((k_rb_xr<V>), dim3(gv), dim3(VB), 0, st, R.nr, n, xx, ph, sh, p, v, t, r, r0, (const double *)om,
                       np, k2, k0, S.part_rho.p);
  }
  void report(KState *pinned) {
    hipLaunchKernelGGL(k_bicg_report, dim3(1), dim3(VB), 0, st, (const double *)S.part_rho.p, nrho, k + SLOT_RHO,
                       pinned);
  }
  void finish() {
    if (!rb) return;
    const RedBlack &R = S.L.ilu->rb;
    hipLaunchKernelGGL((k_rb_out<V, VXo>), dim3(g), dim3(VB), 0, st, R.nr, n, R.e.row, R.f.row, xx, x);
  }
};

// BiCGStab on Ahat x = bhat in precision V; b is given in precision VB_ (already scaled)
template <class V, class VBin, class VXo>
int LinearSolver::bicgstab(const VBin *b, VXo *x, const double *J, const vfvm_control_t &c, double rtol, double atol,
                           int maxit, int &iters, int stag_window) {
  (void)J;
  KState h{};
  h.maxit = maxit;
  h.rtol = rtol;
  h.atol = atol;
  Bicg<V, VXo> K(*this, c, x);
  if (K.one_block()) {
    K.solve_one(b, h, std::max(1, c.check_every), stag_window, hst[0]);
    VFVM_HIP_CHECK(hipGetLastError());
    VFVM_HIP_CHECK(hipEventRecord(sev[0], stream));
    VFVM_HIP_CHECK(hipEventSynchronize(sev[0]));
    h = *hst[0];
    iters = h.iters;
    last_iters = h.iters;
    last_rr = h.rr;
    last_rr0 = h.rr0;
    return h.status == 1 ? 0 : VFVM_ERR_LINEAR;
  }
  VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &h, sizeof(KState), hipMemcpyHostToDevice, stream));
  K.init(b);
  // First chunk: about as many iterations as the previous solve needed (Newton steps of one
  // solve need similar counts), then poll every check_every iterations; an iteration with
  // multigrid costs more than a poll (40 launches even when it has nothing left to do), so
  // there every one: of 123 iterations queued in a Newton solve on 513^2 rows 72 were needed.
  const int every = c.precon == VFVM_PRECON_AMG ? 1 : std::max(1, c.check_every);
  int check = std::max(every, std::min(maxit, last_iters - 1));
  int launched = 0, best_at = 0;
  double best = -1.0;
  // Pipelined: the next block of iterations is queued before the state after the current
  // block is examined (a block queued after convergence runs kernels that return at
  // entry); each block ends with the state's report to its pinned slot.
  auto enqueue = [&](int nit, int slot) {
    for (int q = 0; q < nit; q++) K.iterate(launched + q == 0);
    K.report(hst[slot]);
    VFVM_HIP_CHECK(hipGetLastError());
    launched += nit;
    VFVM_HIP_CHECK(hipEventRecord(sev[slot], stream));
  };
  int slot = 0, last = 0;
  enqueue(check, 0);
  while (true) {
    const bool more = launched < maxit + every;
    if (more) {
      enqueue(every, 1 - slot);
      last = 1 - slot;
    }
    VFVM_HIP_CHECK(hipEventSynchronize(sev[slot]));
    h = *hst[slot];
    if (h.done || !more) break;
    if (stag_window > 0) {
      if (best < 0.0 || h.rr < 0.81 * best) {
        best = h.rr;
        best_at = h.iters;
      } else if (h.iters - best_at >= stag_window) {
        break;  // stagnated: no further blocks are queued
      }
    }
    slot = 1 - slot;
  }
  VFVM_HIP_CHECK(hipEventSynchronize(sev[last]));  // state after the last queued block
  h = *hst[last];
  K.finish();
  VFVM_HIP_CHECK(hipGetLastError());
  iters = h.iters;
  last_iters = h.iters;
  last_rr = h.rr;
  last_rr0 = h.rr0;
  return h.status == 1 ? 0 : VFVM_ERR_LINEAR;
}

// restarted GMRES(m), right preconditioned, CGS2 orthogonalisation
template <class V, class VBin, class VXo>
int LinearSolver::gmres(const VBin *b, VXo *x, const double *J, const vfvm_control_t &c, double rtol, double atol,
                        int maxit, int &iters) {
  int64_t n = L.ndof;
  const int m = std::min(std::max(c.gmres_restart, 1), 64);
  Work<V> &W = work<V>();
  V *r = W.vecs[0].p, *w = W.vecs[1].p, *z = W.vecs[2].p, *bb = W.vecs[3].p;
  V *Vb = nullptr;
  if constexpr (sizeof(V) == 4) Vb = vbasis32.p;
  else Vb = vbasis64.p;
  KState h{};
  h.maxit = maxit;
  h.rtol = rtol;
  h.atol = atol;
  VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &h, sizeof(KState), hipMemcpyHostToDevice, stream));
  const bool blk = c.precon == VFVM_PRECON_BLOCKJACOBI && L.nspec > 1;
  const bool plain = c.precon == VFVM_PRECON_JACOBI || (c.precon == VFVM_PRECON_BLOCKJACOBI && L.nspec == 1);
  const unsigned g = grid_for(n), gv = fold_blocks(n), gn = fold_blocks(L.nnodes);
  const int kid = sizeof(V) == 4 ? VFVM_KERNEL_SPMV32 : VFVM_KERNEL_SPMV64;
  const bool nt = sell_nt[sizeof(V) == 4 ? 0 : 1];
  const V *val;
  if constexpr (sizeof(V) == 4) val = A32.p;
  else val = A64s.p;
  GmArrays G{gmH.p, gmh1.p, gmh2.p, gmcs.p, gmsn.p, gmg.p, m};
  int cur = 0, col = 0;  // slot of the current state; columns of the cycle
  // v_k and z = M^-1 v_k from w after the norm partials in part_rho
  auto next = [&](int k, bool first, int np, const V *from, KState *pinned) {
    V *vk = Vb + (int64_t)(k + 1) * n;
    auto go = [&](auto nsc) {
      constexpr int NS = decltype(nsc)::value;
      hipLaunchKernelGGL((k_gm_next<V, NS>), dim3(NS ? gn : gv), dim3(VB), 0, stream, NS ? L.nnodes : n, from, vk,
                         (const double *)binv.p, z, G, k, first ? 1 : 0, (const double *)part_rho.p, np, st.p + cur,
                         st.p + 1 - cur, pinned);
    };
    if (!blk) go(std::integral_constant<int, 0>());
    else if (L.nspec == 2) go(std::integral_constant<int, 2>());
    else go(std::integral_constant<int, 3>());
    cur = 1 - cur;
  };
  // x += M^-1 (V y) and the state with no columns left
  auto combine = [&]() {
    auto go = [&](auto nsc, auto addc) {
      constexpr int NS = decltype(nsc)::value;
      hipLaunchKernelGGL((k_gm_combine<V, VXo, NS, decltype(addc)::value>), dim3(NS ? gn : gv), dim3(VB), 0, stream,
                         NS ? L.nnodes : n, n, (const V *)Vb, (const double *)binv.p, w, x, G, st.p + cur,
                         st.p + 1 - cur);
    };
    if (plain) {
      go(std::integral_constant<int, 0>(), std::true_type());
    } else if (blk) {
      if (L.nspec == 2) go(std::integral_constant<int, 2>(), std::true_type());
      else go(std::integral_constant<int, 3>(), std::true_type());
    } else {
      go(std::integral_constant<int, 0>(), std::false_type());
      const V *zp = precond<V>(w, z, nullptr, 0, c);
      hipLaunchKernelGGL((k_axpy_out<VXo, V>), dim3(g), dim3(VB), 0, stream, n, x, zp);
    }
    cur = 1 - cur;
  };
  auto with_columns = [&](auto &&f) {
    if (L.sell_off16 && sell16) f(L.sell_off16);
    else f(L.sell_col);
  };
  auto step = [&](KState *pinned) {
    if (col == m) {
      combine();
      with_columns([&](const auto *ci) {
        using CI = std::remove_const_t<std::remove_pointer_t<decltype(ci)>>;
        hipLaunchKernelGGL((k_gm_residual<V, VXo, CI>), dim3(g), dim3(VB), 0, stream, n, L.sell_ptr, ci, val,
                           (const VXo *)x, (const V *)bb, r, (const KState *)(st.p + cur), part_rho.p);
      });
      next(-1, false, (int)g, r, nullptr);
      col = 0;
    }
    const int k = col++, nv = k + 1;
    KState *sk = st.p + cur;
    const V *vk = Vb + (int64_t)k * n;
    const V *zp = plain ? vk : blk ? (const V *)z : precond<V>(vk, z, sk, 0, c);
    if (L.probe) L.probe->before(kid, stream);
    with_columns([&](const auto *ci) {
      using CI = std::remove_const_t<std::remove_pointer_t<decltype(ci)>>;
      if (nt)
        VFVM_LAUNCH((k_gm_av<V, true, CI>), dim3(g), dim3(VB), 0, stream, n, L.sell_ptr, ci, val, zp, w, nv,
                    (const V *)Vb, gmpart.p, (const KState *)sk);
      else
        VFVM_LAUNCH((k_gm_av<V, false, CI>), dim3(g), dim3(VB), 0, stream, n, L.sell_ptr, ci, val, zp, w, nv,
                    (const V *)Vb, gmpart.p, (const KState *)sk);
    });
    if (L.probe) L.probe->after(kid, stream, L.ndof, L.nnz);
    const bool fold = (int)g <= GM_FOLD;
    auto ortho = [&](auto lastc, const double *part, double *hout, double *pout) {
      if (!fold)
        hipLaunchKernelGGL(k_gm_sum, dim3(nv), dim3(VB), 0, stream, (int)g, part, gmsum.p, (const KState *)sk);
      hipLaunchKernelGGL((k_gm_ortho<V, decltype(lastc)::value>), dim3(g), dim3(VB), 0, stream, n, nv, (const V *)Vb, w,
                         fold ? part : (const double *)gmsum.p, fold ? (int)g : 1, hout, pout, (const KState *)sk);
    };
    double *second = fold ? gmpart2.p : gmpart.p;
    ortho(std::false_type(), gmpart.p, gmh1.p, second);
    ortho(std::true_type(), second, gmh2.p, part_rho.p);
    next(k, false, (int)g, w, pinned);
  };
  hipLaunchKernelGGL((k_gm_init<V, VBin, VXo>), dim3(gv), dim3(VB), 0, stream, n, b, bb, x, part_rho.p);
  next(-1, true, (int)gv, bb, nullptr);
  // queued and polled as in bicgstab
  const int every = std::max(1, c.check_every);
  int launched = 0;
  auto enqueue = [&](int nit, int slot) {
    for (int q = 0; q < nit; q++) step(q == nit - 1 ? hst[slot] : nullptr);
    VFVM_HIP_CHECK(hipGetLastError());
    launched += nit;
    VFVM_HIP_CHECK(hipEventRecord(sev[slot], stream));
  };
  int slot = 0, last = 0;
  enqueue(std::max(every, std::min(maxit, last_iters - 1)), 0);
  while (true) {
    const bool more = launched < maxit + every;
    if (more) {
      enqueue(every, 1 - slot);
      last = 1 - slot;
    }
    VFVM_HIP_CHECK(hipEventSynchronize(sev[slot]));
    h = *hst[slot];
    if (h.done || !more) break;
    slot = 1 - slot;
  }
  combine();  // of the cycle that the solve ended in, unless the queue has done it
  VFVM_HIP_CHECK(hipGetLastError());
  VFVM_HIP_CHECK(hipEventSynchronize(sev[last]));
  h = *hst[last];
  iters = h.iters;
  last_iters = h.iters;
  last_rr = h.rr;
  last_rr0 = h.rr0;
  return h.gm_conv ? 0 : VFVM_ERR_LINEAR;
}

// Solve A x = b (b, x FP64 device vectors) with the prepared operator.
int LinearSolver::solve(const double *J, const double *b, double *x, const vfvm_control_t &c, vfvm_linstats_t *stats) {
  int64_t n = L.ndof;
  unsigned g = grid_for(n);
  const int Gs = L.spmv_group;
  // bhat = S b  (as a residual with x = 0)
  bhat.alloc((size_t)n);
  KState h{};
  VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &h, sizeof(KState), hipMemcpyHostToDevice, stream));
  hipLaunchKernelGGL((k_fill<double>), dim3(g), dim3(VB), 0, stream, n, x, 0.0);
  auto scaled_res = [&](const double *xx, double *out) {
    auto go = [&](auto gconst) {
      constexpr int GG = decltype(gconst)::value;
      const unsigned gg = grid_for(n * GG);
      hipLaunchKernelGGL((k_scaled_residual<GG>), dim3(gg), dim3(VB), 0, stream, n, L.rowptr, L.colind, J, xx, b,
                         (const double *)rowscale.p, out, partials.p, st.p);
      hipLaunchKernelGGL((k_finalize<1, STAGE_RR>), dim3(1), dim3(VB), 0, stream, (const double *)partials.p, (int)gg,
                         st.p, 0);
    };
    switch (Gs) {
      case 2: go(std::integral_constant<int, 2>()); break;
      case 4: go(std::integral_constant<int, 4>()); break;
      case 8: go(std::integral_constant<int, 8>()); break;
      case 16: go(std::integral_constant<int, 16>()); break;
      default: go(std::integral_constant<int, 32>()); break;
    }
    VFVM_HIP_CHECK(hipGetLastError());
  };
  scaled_res(x, bhat.p);
  read_state(h);
  const double bnorm = std::sqrt(h.rr);
  const double tol = c.abstol_linear + c.reltol_linear * bnorm;
  int iters = 0, rc = 0, nref = 0;
  bool used_fallback = false;
  double rn = bnorm;
  if (c.precision == VFVM_PREC_FP32_REFINE) {
    // FP64 iterative refinement around FP32 Krylov solves of Ahat d = rhat
    rhs32.alloc((size_t)n);
    d32.alloc((size_t)n);
    rres.alloc((size_t)n);
    float *r32 = d32.p;
    double *rh = rres.p;
    hipLaunchKernelGGL((k_convert<double, double>), dim3(g), dim3(VB), 0, stream, n, (const double *)bhat.p, rh);
    const int maxref = std::max(1, c.max_refinements);
    // after an FP32 failure earlier in this Newton solve or sweep, go to FP64 directly
    const bool fp32_skipped = fp32_off;  // prepare() already built the FP64 operator
    bool fp32_failed = fp32_off;
    // an FP32 inner solve that stops improving is cut short (the FP64 residual then
    // decides between another round and the FP64 finish)
    const int stag = std::max(200, c.maxiters_linear / 20);
    while (!fp32_failed && rn > tol && nref < maxref) {
      hipLaunchKernelGGL((k_convert<float, double>), dim3(g), dim3(VB), 0, stream, n, (const double *)rh, rhs32.p);
      int it = 0;
      const double inner = std::max(c.inner_reltol, 1e-6);
      if (c.krylov == VFVM_KRYLOV_GMRES)
        gmres<float, float, float>(rhs32.p, r32, nullptr, c, inner, 0.0, c.maxiters_linear, it);
      else
        bicgstab<float, float, float>(rhs32.p, r32, nullptr, c, inner, 0.0, c.maxiters_linear, it, stag);
      iters += it;
      xsave.alloc((size_t)n);
      hipLaunchKernelGGL((k_convert<double, double>), dim3(g), dim3(VB), 0, stream, n, (const double *)x, xsave.p);
      hipLaunchKernelGGL((k_add_correction<float>), dim3(g), dim3(VB), 0, stream, n, x, (const float *)r32, 1.0);
      KState z{};
      VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &z, sizeof(KState), hipMemcpyHostToDevice, stream));
      scaled_res(x, rh);
      read_state(h);
      const double rnew = std::sqrt(h.rr);
      nref++;
      if (!(rnew < rn)) {
        // the FP32 solve did not reduce the FP64 residual (stagnation, breakdown or an
        // overflow at this conditioning): restore x and finish in FP64
        hipLaunchKernelGGL((k_convert<double, double>), dim3(g), dim3(VB), 0, stream, n, (const double *)xsave.p, x);
        VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &z, sizeof(KState), hipMemcpyHostToDevice, stream));
        scaled_res(x, rh);
        read_state(h);
        rn = std::sqrt(h.rr);
        fp32_failed = true;
        fp32_off = true;
        break;
      }
      rn = rnew;
      if (it == 0) break;
    }
    if (fp32_failed && rn > tol) {
      // FP64 fallback on the current refinement residual rh = S (b - A x): the FP64
      // operator and preconditioner copies of the same Jacobian (no refactorisation)
      vfvm_control_t c64 = c;
      c64.precision = VFVM_PREC_FP64;
      if (!fp32_skipped) prepare(J, c64, false);
      DevBuf<double> &d64 = fallback64;
      d64.alloc((size_t)n);
      int it = 0;
      const double rtol = tol / std::max(rn, 1e-300);
      if (c.krylov == VFVM_KRYLOV_GMRES)
        gmres<double, double, double>(rh, d64.p, J, c, rtol, 0.0, c.maxiters_linear, it);
      else
        bicgstab<double, double, double>(rh, d64.p, J, c, rtol, 0.0, c.maxiters_linear, it);
      iters += it;
      fallbacks++;
      used_fallback = true;
      hipLaunchKernelGGL((k_add_correction<double>), dim3(g), dim3(VB), 0, stream, n, x, (const double *)d64.p, 1.0);
      KState z{};
      VFVM_HIP_CHECK(hipMemcpyAsync(st.p, &z, sizeof(KState), hipMemcpyHostToDevice, stream));
      scaled_res(x, rh);
      read_state(h);
      rn = std::sqrt(h.rr);
      nref++;
    }
    rc = rn <= tol ? 0 : VFVM_ERR_LINEAR;
  } else {
    if (c.krylov == VFVM_KRYLOV_GMRES)
      rc = gmres<double, double, double>(bhat.p, x, J, c, c.reltol_linear, c.abstol_linear, c.maxiters_linear, iters);
    else
      rc = bicgstab<double, double, double>(bhat.p, x, J, c, c.reltol_linear, c.abstol_linear, c.maxiters_linear,
                                            iters);
    rn = std::sqrt(last_rr);
    nref = 1;
  }
  if (stats) {
    stats->iters = iters;
    stats->refinements = nref;
    stats->converged = rc == 0;
    stats->fp64_fallback = used_fallback ? 1 : 0;
    stats->resnorm0 = bnorm;
    stats->resnorm = rn;
  }
  return rc;
}

// ---- small utilities used by the Newton driver ----
void launch_newton_update(int64_t n, double *U, const double *dU, double damp, double *partials, unsigned *ticket,
                          double *out, hipStream_t s) {
  const unsigned g = grid_for(n);
  hipLaunchKernelGGL(k_newton_update, dim3(g), dim3(VB), 0, s, n, U, dU, damp, partials, ticket, out);
  hipLaunchKernelGGL(k_newton_finalize, dim3(1), dim3(VB), 0, s, (const double *)partials, (int)g, out, out + 1);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_norm1(int64_t n, const double *U, double *partials, unsigned *ticket, double *out, hipStream_t s) {
  const unsigned g = grid_for(n);
  hipLaunchKernelGGL(k_norm1, dim3(g), dim3(VB), 0, s, n, U, partials, ticket, out);
  hipLaunchKernelGGL(k_newton_finalize, dim3(1), dim3(VB), 0, s, (const double *)partials, (int)g, (double *)nullptr,
                     out);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_maxdiff(int64_t n, const double *a, const double *b, double *partials, double *out, hipStream_t s) {
  const unsigned g = grid_for(n);
  hipLaunchKernelGGL(k_maxdiff, dim3(g), dim3(VB), 0, s, n, a, b, partials);
  hipLaunchKernelGGL(k_newton_finalize, dim3(1), dim3(VB), 0, s, (const double *)partials, (int)g, out, out + 1);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_gather(int64_t n, const int32_t *perm, const double *J, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3(grid_for(n)), dim3(VB), 0, s, n, perm, J, out);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_fill_u64(int64_t n, unsigned long long *p, hipStream_t s) {
  hipLaunchKernelGGL((k_fill<unsigned long long>), dim3(grid_for(n)), dim3(VB), 0, s, n, p, 0ull);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_fill_i32(int64_t n, int32_t *p, int32_t v, hipStream_t s) {
  hipLaunchKernelGGL((k_fill<int32_t>), dim3(grid_for(n)), dim3(VB), 0, s, n, p, v);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_negate(int64_t n, double *x, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_negate, dim3(grid_for(n)), dim3(VB), 0, s, n, x);
  VFVM_HIP_CHECK(hipGetLastError());
}
void launch_copy(int64_t n, const double *a, double *b, hipStream_t s) {
  hipLaunchKernelGGL((k_convert<double, double>), dim3(grid_for(n)), dim3(VB), 0, s, n, a, b);
  VFVM_HIP_CHECK(hipGetLastError());
}

void launch_scale_rows(int nspec, int64_t nnodes, const int32_t *rowptr, const int32_t *colind, const double *A,
                       const int32_t *dofdiag, const int32_t *rbase, double *rowscale, float *A32, double *A64,
                       double *binv, hipStream_t s) {
  unsigned g = grid_for(nnodes);
  switch (nspec) {
    case 1:
      hipLaunchKernelGGL((k_scale_rows<1>), dim3(g), dim3(VB), 0, s, nnodes, rowptr, colind, A, dofdiag, rbase,
                         rowscale, A32, A64, binv);
      break;
    case 2:
      hipLaunchKernelGGL((k_scale_rows<2>), dim3(g), dim3(VB), 0, s, nnodes, rowptr, colind, A, dofdiag, rbase,
                         rowscale, A32, A64, binv);
      break;
    default:
      hipLaunchKernelGGL((k_scale_rows<3>), dim3(g), dim3(VB), 0, s, nnodes, rowptr, colind, A, dofdiag, rbase,
                         rowscale, A32, A64, binv);
      break;
  }
  VFVM_HIP_CHECK(hipGetLastError());
}

// timing helper for the autotuner: plain FP64 SpMV y = A x
void time_spmv(const LinSetup &L, int G, const double *A, const double *x, double *y, hipStream_t s) {
  unsigned g = grid_for(L.ndof * G);
  auto go = [&](auto gconst) {
    constexpr int GG = decltype(gconst)::value;
    hipLaunchKernelGGL((k_spmv<double, double, GG, 0, STAGE_NONE>), dim3(g), dim3(VB), 0, s, L.ndof, L.rowptr,
                       L.colind, A, x, y, (const double *)nullptr, (const double *)nullptr, (const double *)nullptr,
                       (double *)nullptr, (KState *)nullptr);
  };
  switch (G) {
    case 2: go(std::integral_constant<int, 2>()); break;
    case 4: go(std::integral_constant<int, 4>()); break;
    case 8: go(std::integral_constant<int, 8>()); break;
    case 16: go(std::integral_constant<int, 16>()); break;
    default: go(std::integral_constant<int, 32>()); break;
  }
  VFVM_HIP_CHECK(hipGetLastError());
}

}  // namespace vfvm
