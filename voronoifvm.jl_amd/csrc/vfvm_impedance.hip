// Small-signal impedance (src/vfvm_impedance.jl): the frequency-domain system
//   (J(U0) + i w M) UZ = F
// around a steady state U0, for a whole sweep of frequencies w at once, and the
// measurement z(w) = dstdy . UZ + i w dtran . UZ, impedance 1 / z.
//
// J(U0) is the Jacobian assembled with tstep = 1e30 and Uold = U0 (as the reference
// does, so the storage entries are in the pattern), M the storage derivative
// (diagonal for the registry: node volume on species with storage), F the excitation
// of one species on one boundary region.  The complex systems are solved together by
// BiCGStab on the row-scaled operator D_w^-1 (J + i w M), D_w its diagonal: every
// frequency is a member of the batch, every kernel covers all members, converged
// members drop out.  Scalar systems of some size are right-preconditioned by a multigrid
// cycle that all frequencies of a group share (sweep_multigrid); the others, and what that
// does not finish, run on the row scaling alone (sweep_jacobi).  Dot products are reduced in
// a fixed order (block partials, one finishing block per member), so a sweep is
// deterministic.
#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>

#include "vfvm_linalg.h"
#include "vfvm_sys.h"

struct vfvm_impedance {
  vfvm_sys *sys = nullptr;
  int64_t n = 0, nnz = 0;
  DevBuf<double> J, M, b;
  // Work of the sweeps, kept between them (a sweep holds the mutex): Krylov vectors and
  // partials, grown to the largest sweep, and the multigrid hierarchy of J + sigma M with its
  // matrix and row scaling (sigma: the shift it was last set up for)
  std::mutex mu;
  DevBuf<double2> ws[10], part;
  DevBuf<double> Ks, ks;
  DevBuf<int32_t> skip;
  vfvm::Amg amg;
  double sigma = -1.0;
};

namespace {

constexpr int ZB = 256;       // threads per block
constexpr int ZMAXBLK = 512;  // row blocks per member

struct ZState {
  double2 rho, alpha, omega, beta;
  double b2, rn2;
  int32_t done, iters, breakdown, pad;
};

__device__ __forceinline__ double2 zadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 zsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// conj(a) * b
__device__ __forceinline__ double2 zcmul(double2 a, double2 b) {
  return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double2 zdiv(double2 a, double2 b) {
  // scaled by the larger component so that penalty-sized diagonals (1e30) do not overflow
  const double s = fmax(fabs(b.x), fabs(b.y));
  const double bx = b.x / s, by = b.y / s, d = bx * bx + by * by;
  return make_double2((a.x * bx + a.y * by) / (s * d), (a.y * bx - a.x * by) / (s * d));
}

// diagonal of member w at row i
__device__ __forceinline__ double2 zdiag(const double *J, const int32_t *dofdiag, const double *M, double om,
                                         int64_t i) {
  return make_double2(J[dofdiag[i]], om * M[i]);
}

template <int ND>
__device__ __forceinline__ void block_partials(double2 (&v)[ND], double2 *out) {
  __shared__ double2 sh[ND][ZB];
#pragma unroll
  for (int k = 0; k < ND; k++) sh[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int h = ZB / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
#pragma unroll
      for (int k = 0; k < ND; k++) sh[k][threadIdx.x] = zadd(sh[k][threadIdx.x], sh[k][threadIdx.x + h]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < ND; k++) out[k] = sh[k][0];
}

// y = D_w^-1 (J + i w M) x for the ZMB members w = blockIdx.y * ZMB + m of a block:
// each thread applies its row to every member of the group in turn, so the row's
// matrix entries come from cache after the first member.  ND = 1: partial (r0, y);
// ND = 2: partials (y, s) and (y, y)
constexpr int ZMB = 8;
constexpr int ZRMAX = 8;  // rows up to this length are kept in registers

template <int ND>
__global__ __launch_bounds__(ZB) void k_zop(int64_t n, int nw, const int32_t *__restrict__ rowptr,
                                            const int32_t *__restrict__ colind, const double *__restrict__ J,
                                            const int32_t *__restrict__ dofdiag, const double *__restrict__ M,
                                            const double *__restrict__ omega, const double2 *__restrict__ X,
                                            double2 *__restrict__ Y, const double2 *__restrict__ R,
                                            double2 *__restrict__ part, const ZState *__restrict__ st) {
  const int w0 = blockIdx.y * ZMB;
  bool live[ZMB];
  bool any = false;
#pragma unroll
  for (int m = 0; m < ZMB; m++) {
    live[m] = w0 + m < nw && !st[w0 + m].done;
    any |= live[m];
  }
  if (!any) return;
  double2 acc[ZMB][ND];
#pragma unroll
  for (int m = 0; m < ZMB; m++)
#pragma unroll
    for (int k = 0; k < ND; k++) acc[m][k] = make_double2(0.0, 0.0);
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const int32_t k0 = rowptr[i], k1 = rowptr[i + 1];
    const double Mi = M[i], Jii = J[dofdiag[i]];
    // a short row is held in registers for all members of the group
    const bool short_row = k1 - k0 <= ZRMAX;
    double jv[ZRMAX];
    int32_t jc[ZRMAX];
#pragma unroll
    for (int q = 0; q < ZRMAX; q++) {
      const bool in = short_row && k0 + q < k1;
      jv[q] = in ? J[k0 + q] : 0.0;
      jc[q] = in ? colind[k0 + q] : (int32_t)i;
    }
#pragma unroll
    for (int m = 0; m < ZMB; m++) {
      if (!live[m]) continue;
      const int w = w0 + m;
      const double om = omega[w];
      const double2 *x = X + (int64_t)w * n;
      double2 sum = make_double2(0.0, 0.0);
      if (short_row) {
#pragma unroll
        for (int q = 0; q < ZRMAX; q++) {
          if (k0 + q < k1) {
            const double2 xv = x[jc[q]];
            sum.x += jv[q] * xv.x;
            sum.y += jv[q] * xv.y;
          }
        }
      } else {
        for (int32_t k = k0; k < k1; k++) {
          const double a = J[k];
          const double2 xv = x[colind[k]];
          sum.x += a * xv.x;
          sum.y += a * xv.y;
        }
      }
      const double2 xi = x[i];
      sum = zadd(sum, make_double2(-om * Mi * xi.y, om * Mi * xi.x));
      const double2 yi = zdiv(sum, make_double2(Jii, om * Mi));
      Y[(int64_t)w * n + i] = yi;
      const double2 ri = R[(int64_t)w * n + i];
      if constexpr (ND == 1) {
        acc[m][0] = zadd(acc[m][0], zcmul(ri, yi));
      } else {
        acc[m][0] = zadd(acc[m][0], zcmul(yi, ri));
        acc[m][1].x += yi.x * yi.x + yi.y * yi.y;
      }
    }
  }
#pragma unroll
  for (int m = 0; m < ZMB; m++)
    if (live[m]) block_partials<ND>(acc[m], part + ((int64_t)(w0 + m) * gridDim.x + blockIdx.x) * ND);
}

// x = 0, r = r0 = p = D_w^-1 b; partials (r0, r) and (r, r)
__global__ __launch_bounds__(ZB) void k_zinit(int64_t n, const double *__restrict__ b, const double *__restrict__ J,
                                              const int32_t *__restrict__ dofdiag, const double *__restrict__ M,
                                              const double *__restrict__ omega, double2 *__restrict__ X,
                                              double2 *__restrict__ R, double2 *__restrict__ R0,
                                              double2 *__restrict__ P, double2 *__restrict__ part) {
  const int w = blockIdx.y;
  const double om = omega[w];
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const int64_t q = (int64_t)w * n + i;
    const double2 ri = zdiv(make_double2(b[i], 0.0), zdiag(J, dofdiag, M, om, i));
    X[q] = make_double2(0.0, 0.0);
    R[q] = ri;
    R0[q] = ri;
    P[q] = ri;
    acc[0] = zadd(acc[0], zcmul(ri, ri));
    acc[1].x += ri.x * ri.x + ri.y * ri.y;
  }
  block_partials<2>(acc, part + ((int64_t)w * gridDim.x + blockIdx.x) * 2);
}

// s = r - alpha v
__global__ __launch_bounds__(ZB) void k_zs(int64_t n, const double2 *__restrict__ R, const double2 *__restrict__ V,
                                           double2 *__restrict__ S, const ZState *__restrict__ st) {
  const int w = blockIdx.y;
  if (st[w].done) return;
  const double2 al = st[w].alpha;
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const int64_t q = (int64_t)w * n + i;
    S[q] = zsub(R[q], zmul(al, V[q]));
  }
}

// x += alpha p + omega s, r = s - omega t; partials (r0, r), (r, r)
__global__ __launch_bounds__(ZB) void k_zx(int64_t n, double2 *__restrict__ X, double2 *__restrict__ R,
                                           const double2 *__restrict__ R0, const double2 *__restrict__ P,
                                           const double2 *__restrict__ S, const double2 *__restrict__ T,
                                           double2 *__restrict__ part, const ZState *__restrict__ st) {
  const int w = blockIdx.y;
  if (st[w].done) return;
  const double2 al = st[w].alpha, om = st[w].omega;
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const int64_t q = (int64_t)w * n + i;
    const double2 si = S[q];
    X[q] = zadd(X[q], zadd(zmul(al, P[q]), zmul(om, si)));
    const double2 ri = zsub(si, zmul(om, T[q]));
    R[q] = ri;
    acc[0] = zadd(acc[0], zcmul(R0[q], ri));
    acc[1].x += ri.x * ri.x + ri.y * ri.y;
  }
  block_partials<2>(acc, part + ((int64_t)w * gridDim.x + blockIdx.x) * 2);
}

// p = r + beta (p - omega v)
__global__ __launch_bounds__(ZB) void k_zp(int64_t n, const double2 *__restrict__ R, double2 *__restrict__ P,
                                           const double2 *__restrict__ V, const ZState *__restrict__ st) {
  const int w = blockIdx.y;
  if (st[w].done) return;
  const double2 be = st[w].beta, om = st[w].omega;
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const int64_t q = (int64_t)w * n + i;
    P[q] = zadd(R[q], zmul(be, zsub(P[q], zmul(om, V[q]))));
  }
}

enum { ZF_INIT = 0, ZF_ALPHA = 1, ZF_OMEGA = 2, ZF_RHO = 3 };

// one block per member: the partials summed in a fixed order, then the scalars
// (block b's partials of member w at (w sw + b sb) ND); skip (nullable): set once done
template <int STAGE, int ND>
__global__ __launch_bounds__(ZB) void k_zfin(int nblk, int64_t sw, int64_t sb, const double2 *__restrict__ part,
                                             ZState *__restrict__ st, double tol2, int iterate,
                                             int32_t *__restrict__ skip) {
  const int w = blockIdx.x;
  ZState &z = st[w];
  if (STAGE != ZF_INIT && z.done) return;
  double2 acc[ND];
#pragma unroll
  for (int k = 0; k < ND; k++) acc[k] = make_double2(0.0, 0.0);
  for (int b = threadIdx.x; b < nblk; b += ZB)
#pragma unroll
    for (int k = 0; k < ND; k++) acc[k] = zadd(acc[k], part[(w * sw + b * sb) * ND + k]);
  __shared__ double2 out[ND];
  block_partials<ND>(acc, out);
  __syncthreads();
  if (threadIdx.x != 0) return;
  struct Mark {  // the member's skip flag follows its state on every way out
    ZState &z;
    int32_t *skip;
    int w;
    __device__ ~Mark() {
      if (skip) skip[w] = z.done;
    }
  } mark{z, skip, w};
  const double2 zero = make_double2(0.0, 0.0);
  if (STAGE == ZF_INIT) {
    z.rho = out[0];
    z.b2 = out[ND - 1].x;
    z.rn2 = z.b2;
    z.alpha = z.omega = make_double2(1.0, 0.0);
    z.beta = zero;
    z.iters = 0;
    z.breakdown = 0;
    z.done = !(z.b2 > 0.0);  // a zero right-hand side: x = 0 is the solution
  } else if (STAGE == ZF_ALPHA) {
    const double2 d = out[0];
    if (!(d.x * d.x + d.y * d.y > 0.0)) {
      z.breakdown = 1;
      z.done = 1;
      return;
    }
    z.alpha = zdiv(z.rho, d);
  } else if (STAGE == ZF_OMEGA) {
    const double tt = out[1].x;
    z.omega = tt > 0.0 ? make_double2(out[0].x / tt, out[0].y / tt) : zero;
  } else {
    z.iters += iterate;
    z.rn2 = out[1].x;
    const double2 rho_new = out[0];
    if (!(z.rn2 == z.rn2)) {
      z.breakdown = 1;
      z.done = 1;
      return;
    }
    if (z.rn2 <= tol2 * z.b2) {
      z.done = 1;
      return;
    }
    const double om2 = z.omega.x * z.omega.x + z.omega.y * z.omega.y;
    const double rh2 = z.rho.x * z.rho.x + z.rho.y * z.rho.y;
    if (!(om2 > 0.0) || !(rh2 > 0.0)) {
      z.breakdown = 1;
      z.done = 1;
      return;
    }
    z.beta = zmul(zdiv(rho_new, z.rho), zdiv(z.alpha, z.omega));
    z.rho = rho_new;
  }
}

// ---- the multigrid-preconditioned form: members interleaved, member w of row i at
// i nw + w, thread (row, member) with 256 / nw rows per block and turn.  A matrix entry is
// read once for all members of a row, and every vector access is contiguous.
struct ZRow {
  int64_t i, step;  // first row (n when the thread has none) and row stride
  int w, r, rpb;
  bool live;
};
__device__ __forceinline__ ZRow zrow(int64_t n, int nw, const ZState *st) {
  ZRow z;
  z.rpb = ZB / nw;
  z.r = (int)threadIdx.x / nw;
  z.w = (int)threadIdx.x - z.r * nw;
  z.i = (int64_t)blockIdx.x * z.rpb + z.r;
  z.step = (int64_t)gridDim.x * z.rpb;
  z.live = z.r < z.rpb && !(st && st[z.w].done);
  if (!z.live) z.i = n;
  return z;
}

// per member sums over the block's rows, in a fixed order, to part[(block nw + w) ND ..]
template <int ND>
__device__ __forceinline__ void zrow_partials(const ZRow &z, int nw, double2 (&v)[ND], double2 *part) {
  __shared__ double2 sh[ND][ZB];
#pragma unroll
  for (int k = 0; k < ND; k++) sh[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int s = z.rpb; s > 1;) {
    const int h = (s + 1) / 2;
    if (z.r < s - h)
#pragma unroll
      for (int k = 0; k < ND; k++) sh[k][threadIdx.x] = zadd(sh[k][threadIdx.x], sh[k][threadIdx.x + h * nw]);
    __syncthreads();
    s = h;
  }
  if (z.r == 0 && z.live)
#pragma unroll
    for (int k = 0; k < ND; k++) part[((int64_t)blockIdx.x * nw + z.w) * ND + k] = sh[k][threadIdx.x];
}

// g = S D_w at row i: what turns the row-scaled system D_w^-1 (J + i w M) into one with the
// scaling of the hierarchy's matrix diag(K)^-1 K, K = J + sigma M
__device__ __forceinline__ double2 zscale(double Jii, double om, double Mi, double ksi) {
  return make_double2(ksi * Jii, ksi * om * Mi);
}

// x = 0, r = r0 = D_w^-1 b, p = v = 0; partials (r0, r), (r, r)
__global__ __launch_bounds__(ZB) void k_ziinit(int64_t n, int nw, const double *__restrict__ b,
                                               const double *__restrict__ J, const int32_t *__restrict__ dofdiag,
                                               const double *__restrict__ M, const double *__restrict__ omega,
                                               double2 *__restrict__ X, double2 *__restrict__ R,
                                               double2 *__restrict__ R0, double2 *__restrict__ P,
                                               double2 *__restrict__ V, double2 *__restrict__ part) {
  const ZRow z = zrow(n, nw, nullptr);
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  const double2 zero = make_double2(0.0, 0.0);
  const double om = z.live ? omega[z.w] : 0.0;
  for (int64_t i = z.i; i < n; i += z.step) {
    const int64_t q = i * nw + z.w;
    const double2 ri = zdiv(make_double2(b[i], 0.0), zdiag(J, dofdiag, M, om, i));
    X[q] = zero;
    R[q] = ri;
    R0[q] = ri;
    P[q] = zero;
    V[q] = zero;
    acc[0] = zadd(acc[0], zcmul(ri, ri));
    acc[1].x += ri.x * ri.x + ri.y * ri.y;
  }
  zrow_partials<2>(z, nw, acc, part);
}

// FIRST: p = r + beta (p - omega v), Q = g p (p = r in the first iteration, where beta = 0);
// else: s = r - alpha v, Q = g s
template <bool FIRST>
__global__ __launch_bounds__(ZB) void k_zivec(int64_t n, int nw, const double *__restrict__ J,
                                              const int32_t *__restrict__ dofdiag, const double *__restrict__ M,
                                              const double *__restrict__ ks, const double *__restrict__ omega,
                                              const double2 *__restrict__ R, const double2 *__restrict__ V,
                                              double2 *__restrict__ PS, double2 *__restrict__ Q,
                                              const ZState *__restrict__ st) {
  const ZRow z = zrow(n, nw, st);
  if (z.i >= n) return;
  const double om = omega[z.w];
  const double2 al = st[z.w].alpha, be = st[z.w].beta, w = st[z.w].omega;
  for (int64_t i = z.i; i < n; i += z.step) {
    const int64_t q = i * nw + z.w;
    const double2 v = V[q];
    const double2 y = FIRST ? zadd(R[q], zmul(be, zsub(PS[q], zmul(w, v)))) : zsub(R[q], zmul(al, v));
    PS[q] = y;
    Q[q] = zmul(zscale(J[dofdiag[i]], om, M[i], ks[i]), y);
  }
}

// Y = D_w^-1 (J + i w M) X; ND = 1: partial (W, Y); ND = 2: partials (Y, W) and (Y, Y)
template <int ND>
__global__ __launch_bounds__(ZB) void k_ziop(int64_t n, int nw, const int32_t *__restrict__ rowptr,
                                             const int32_t *__restrict__ colind, const double *__restrict__ J,
                                             const int32_t *__restrict__ dofdiag, const double *__restrict__ M,
                                             const double *__restrict__ omega, const double2 *__restrict__ X,
                                             double2 *__restrict__ Y, const double2 *__restrict__ W,
                                             double2 *__restrict__ part, const ZState *__restrict__ st) {
  const ZRow z = zrow(n, nw, st);
  double2 acc[ND];
#pragma unroll
  for (int k = 0; k < ND; k++) acc[k] = make_double2(0.0, 0.0);
  const double om = z.live ? omega[z.w] : 0.0;
  for (int64_t i = z.i; i < n; i += z.step) {
    const int32_t k0 = rowptr[i], k1 = rowptr[i + 1];
    double2 sum = make_double2(0.0, 0.0);
#pragma unroll 4
    for (int32_t k = k0; k < k1; k++) {
      const double a = J[k];
      const double2 xv = X[(int64_t)colind[k] * nw + z.w];
      sum.x += a * xv.x;
      sum.y += a * xv.y;
    }
    const int64_t q = i * nw + z.w;
    const double2 xi = X[q];
    const double m = om * M[i];
    const double2 yi = zdiv(make_double2(sum.x - m * xi.y, sum.y + m * xi.x), make_double2(J[dofdiag[i]], m));
    Y[q] = yi;
    const double2 wi = W[q];
    if constexpr (ND == 1) {
      acc[0] = zadd(acc[0], zcmul(wi, yi));
    } else {
      acc[0] = zadd(acc[0], zcmul(yi, wi));
      acc[1].x += yi.x * yi.x + yi.y * yi.y;
    }
  }
  zrow_partials<ND>(z, nw, acc, part);
}

// x += alpha ph + omega sh, r = s - omega t; partials (r0, r), (r, r)
__global__ __launch_bounds__(ZB) void k_zix(int64_t n, int nw, double2 *__restrict__ X, double2 *__restrict__ R,
                                            const double2 *__restrict__ R0, const double2 *__restrict__ PH,
                                            const double2 *__restrict__ SH, const double2 *__restrict__ S,
                                            const double2 *__restrict__ T, double2 *__restrict__ part,
                                            const ZState *__restrict__ st) {
  const ZRow z = zrow(n, nw, st);
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  const double2 zero = make_double2(0.0, 0.0);
  const double2 al = z.live ? st[z.w].alpha : zero, om = z.live ? st[z.w].omega : zero;
  for (int64_t i = z.i; i < n; i += z.step) {
    const int64_t q = i * nw + z.w;
    X[q] = zadd(X[q], zadd(zmul(al, PH[q]), zmul(om, SH[q])));
    const double2 ri = zsub(S[q], zmul(om, T[q]));
    R[q] = ri;
    acc[0] = zadd(acc[0], zcmul(R0[q], ri));
    acc[1].x += ri.x * ri.x + ri.y * ri.y;
  }
  zrow_partials<2>(z, nw, acc, part);
}

// partials of dstdy . x and dtran . x per member
__global__ __launch_bounds__(ZB) void k_zimeas(int64_t n, int nw, const double *__restrict__ ds,
                                               const double *__restrict__ dt, const double2 *__restrict__ X,
                                               double2 *__restrict__ part) {
  const ZRow z = zrow(n, nw, nullptr);
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int64_t i = z.i; i < n; i += z.step) {
    const double2 xi = X[i * nw + z.w];
    acc[0].x += ds[i] * xi.x;
    acc[0].y += ds[i] * xi.y;
    acc[1].x += dt[i] * xi.x;
    acc[1].y += dt[i] * xi.y;
  }
  zrow_partials<2>(z, nw, acc, part);
}

// Y[w n + i] = X[i nw + w]
__global__ __launch_bounds__(ZB) void k_zitrans(int64_t n, int nw, const double2 *__restrict__ X,
                                                double2 *__restrict__ Y) {
  const int64_t q = (int64_t)blockIdx.x * ZB + threadIdx.x;
  if (q >= n * nw) return;
  const int64_t w = q / n, i = q - w * n;
  Y[q] = X[i * nw + w];
}

// K = J + sigma M on the pattern of J, ks = 1 / diag(K) (1 where that vanishes)
__global__ __launch_bounds__(ZB) void k_zishift(int64_t n, const int32_t *__restrict__ rowptr,
                                                const int32_t *__restrict__ dofdiag, const double *__restrict__ J,
                                                const double *__restrict__ M, double sigma, double *__restrict__ K,
                                                double *__restrict__ ks) {
  const int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x;
  if (i >= n) return;
  const int32_t d = dofdiag[i];
  for (int32_t k = rowptr[i]; k < rowptr[i + 1]; k++) {
    const double v = J[k] + (k == d ? sigma * M[i] : 0.0);
    K[k] = v;
    if (k == d) ks[i] = (v != 0.0 && v == v) ? 1.0 / v : 1.0;
  }
}

// partials of dstdy . x and dtran . x per member
__global__ __launch_bounds__(ZB) void k_zmeas(int64_t n, const double *__restrict__ ds, const double *__restrict__ dt,
                                              const double2 *__restrict__ X, double2 *__restrict__ part) {
  const int w = blockIdx.y;
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int64_t i = (int64_t)blockIdx.x * ZB + threadIdx.x; i < n; i += (int64_t)gridDim.x * ZB) {
    const double2 xi = X[(int64_t)w * n + i];
    acc[0].x += ds[i] * xi.x;
    acc[0].y += ds[i] * xi.y;
    acc[1].x += dt[i] * xi.x;
    acc[1].y += dt[i] * xi.y;
  }
  block_partials<2>(acc, part + ((int64_t)w * gridDim.x + blockIdx.x) * 2);
}

// Z_w = 1 / (a + i w b)
__global__ __launch_bounds__(ZB) void k_zmeas_fin(int nblk, int64_t sw, int64_t sb, const double2 *__restrict__ part,
                                                  const double *__restrict__ omega, double2 *__restrict__ Z) {
  const int w = blockIdx.x;
  double2 acc[2] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
  for (int b = threadIdx.x; b < nblk; b += ZB) {
    acc[0] = zadd(acc[0], part[(w * sw + b * sb) * 2]);
    acc[1] = zadd(acc[1], part[(w * sw + b * sb) * 2 + 1]);
  }
  __shared__ double2 out[2];
  block_partials<2>(acc, out);
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double om = omega[w];
  const double2 z = zadd(out[0], zmul(make_double2(0.0, om), out[1]));
  Z[w] = zdiv(make_double2(1.0, 0.0), z);
}

// y_j = -sum over the stored entries (i, j) of J_ij w_i, w_i = T_K on the rows of
// species `spec` (i = K * ns + spec); column-wise in CSC order, so deterministic
__global__ __launch_bounds__(ZB) void k_meas_stdy(int64_t n, int ns, int spec, const int32_t *__restrict__ colptr,
                                                  const int32_t *__restrict__ rowval,
                                                  const int32_t *__restrict__ perm, const double *__restrict__ J,
                                                  const double *__restrict__ T, double *__restrict__ y) {
  const int64_t j = (int64_t)blockIdx.x * ZB + threadIdx.x;
  if (j >= n) return;
  double acc = 0.0;
  for (int32_t p = colptr[j]; p < colptr[j + 1]; p++) {
    const int32_t i = rowval[p];
    if (i % ns == spec) acc += J[perm[p]] * T[i / ns];
  }
  y[j] = -acc;
}

// per-species sums of T_K F[K * ns + i]: one block, fixed order
__global__ __launch_bounds__(ZB) void k_tdot(int64_t nnodes, int ns, const double *__restrict__ T,
                                             const double *__restrict__ F, double *__restrict__ out) {
  __shared__ double sh[ZB];
  for (int i = 0; i < ns; i++) {
    double acc = 0.0;
    for (int64_t K = threadIdx.x; K < nnodes; K += ZB) acc += T[K] * F[K * ns + i];
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int h = ZB / 2; h > 0; h >>= 1) {
      if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[i] = sh[0];
    __syncthreads();
  }
}

// the residual of flux, reaction and source terms alone (every boundary condition
// switched off) at U, tstep = Inf, into F
void residual_without_bc(vfvm_sys &s, const double *dU, const double *dUold, double tstep, double lambda,
                         double *dF) {
  std::vector<vfvm_bc_t> saved = s.bc;
  for (auto &c : s.bc) c.kind = VFVM_BC_NONE;
  try {
    upload_inst(s);
    AsmArgs a = asm_args(s, dU, dUold, dF, nullptr, tstep, lambda);
    run_assembly(s, a, s.res_group, s.ctx->stream);
  } catch (...) {
    s.bc = saved;
    upload_inst(s);
    throw;
  }
  s.bc = saved;
  upload_inst(s);
}

void check_dofs(const vfvm_sys &s, int spec) {
  if (spec < 1 || spec > s.nspec) throw Error(VFVM_ERR_ARG, "species number out of range");
}

}  // namespace

extern "C" {

int vfvm_impedance_destroy(vfvm_impedance *z);

namespace {
int impedance_create_at(vfvm_sys *s, const double *U0, int excited_spec, int excited_bc, double lambda,
                        vfvm_impedance **out);
}

int vfvm_impedance_create(vfvm_sys *s, const double *U0, int excited_spec, int excited_bc, vfvm_impedance **out) {
  return impedance_create_at(s, U0, excited_spec, excited_bc, 0.0, out);
}

namespace {
// the impedance system of J(U0) at the system parameter lambda
int impedance_create_at(vfvm_sys *s, const double *U0, int excited_spec, int excited_bc, double lambda,
                        vfvm_impedance **out) {
  if (!s || !U0 || !out) return VFVM_ERR_ARG;
  try {
    check_dofs(*s, excited_spec);
    if (excited_bc < 1 || excited_bc > MAXBREG + 1) throw Error(VFVM_ERR_ARG, "boundary region out of range");
    VFVM_HIP_CHECK(hipSetDevice(s->ctx->device));
    std::unique_ptr<vfvm_impedance> z(new vfvm_impedance());
    z->sys = s;
    z->n = s->ndof;
    z->nnz = s->nnz;
    hipStream_t st = s->ctx->stream;
    // J(U0) with tstep = 1e30 and Uold = U0 (src/vfvm_impedance.jl:60-71)
    s->d_U.upload(U0, (size_t)s->ndof, st);
    z->J.alloc((size_t)s->nnz);
    launch_fill_i32(1, s->d_flags.p, 0, st);
    AsmArgs a = asm_args(*s, s->d_U.p, s->d_U.p, s->d_F.p, z->J.p, 1.0e30, lambda);
    run_assembly(*s, a, s->asm_group, st);
    int32_t fl = 0;
    VFVM_HIP_CHECK(hipMemcpyAsync(&fl, s->d_flags.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    if (fl & 1) throw Error(VFVM_ERR_ASSEMBLY, "trying to assemble NaN");
    // storage derivative (diagonal for the registry) and the excitation: the legacy
    // Dirichlet factor 1e30 per boundary item of the excited region and species, a
    // Robin factor times the item's face measure (src/vfvm_impedance.jl:159-186)
    sync_host_geometry(*s);
    const int ns = s->nspec;
    std::vector<double> M((size_t)s->ndof, 0.0), b((size_t)s->ndof, 0.0);
    const double ds = s->phys.storage == VFVM_STOR_IDENTITY ? 1.0 : 0.0;
    for (int64_t K = 0; K < s->nnodes; K++)
      for (int i = 0; i < ns; i++) M[(size_t)(K * ns + i)] = ds * s->hs.nodevol[(size_t)K];
    const int ispec = excited_spec - 1;
    if (excited_bc <= s->nbreg) {
      const vfvm_bc_t &bc = s->bc[(size_t)(excited_bc - 1) * ns + ispec];
      for (int64_t K = 0; K < s->nnodes; K++)
        for (int32_t q = s->hs.bn_ptr[(size_t)K]; q < s->hs.bn_ptr[(size_t)K + 1]; q++) {
          if (s->hs.bn_reg[(size_t)q] != excited_bc) continue;
          if (bc.kind == VFVM_BC_DIRICHLET_LEGACY)
            b[(size_t)(K * ns + ispec)] += DIRICHLET_PENALTY;
          else if (bc.kind == VFVM_BC_ROBIN)
            b[(size_t)(K * ns + ispec)] += bc.factor * s->hs.bn_fac[(size_t)q];
        }
    }
    z->M.upload(M, st);
    z->b.upload(b, st);
    *out = z.release();
    return VFVM_OK;
  } catch (const Error &e) {
    s->ctx->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    s->ctx->err = e.what();
    return VFVM_ERR_HIP;
  }
}
}  // namespace

int vfvm_impedance_create_param(vfvm_sys *s, const double *U0, double lambda0, vfvm_impedance **out) {
  if (!s || !U0 || !out) return VFVM_ERR_ARG;
  // as the boundary-excited form with no boundary excitation, then F = -dF/dlambda
  // (src/vfvm_impedance.jl:49-112: params = [lambda0], F .-= dudp[1])
  int rc = impedance_create_at(s, U0, 1, MAXBREG + 1, lambda0, out);
  if (rc) return rc;
  try {
    vfvm_impedance *z = *out;
    hipStream_t st = s->ctx->stream;
    s->d_U.upload(U0, (size_t)s->ndof, st);
    AsmArgs a = asm_args(*s, s->d_U.p, s->d_U.p, s->d_F.p, nullptr, INFINITY, lambda0);
    launch_dudp(s->nnodes, s->nspec, s->d_bn_ptr.p, s->d_bn_reg.p, s->d_bn_fac.p, s->d_nodevol.p,
                s->has_src ? s->d_src.p : nullptr, s->d_inst.p, z->b.p, st);
    if (s->has_dp) launch_dudp_coef(a, s->dpar, z->b.p, st);
    launch_negate(s->ndof, z->b.p, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    return VFVM_OK;
  } catch (const Error &e) {
    vfvm_impedance_destroy(*out);
    *out = nullptr;
    s->ctx->err = e.what();
    return e.code;
  }
}

int vfvm_impedance_destroy(vfvm_impedance *z) {
  if (!z) return VFVM_OK;
  (void)hipSetDevice(z->sys->ctx->device);
  (void)hipStreamSynchronize(z->sys->ctx->stream);
  delete z;
  return VFVM_OK;
}

int vfvm_measurement_derivatives(vfvm_sys *s, const double *U0, const double *T, int spec, double *dstdy,
                                 double *dtran) {
  return vfvm_measurement_derivatives_at(s, U0, T, spec, 0.0, dstdy, dtran);
}

int vfvm_measurement_derivatives_at(vfvm_sys *s, const double *U0, const double *T, int spec, double lambda,
                                    double *dstdy, double *dtran) {
  if (!s || !U0 || !T || !dstdy || !dtran) return VFVM_ERR_ARG;
  std::vector<vfvm_bc_t> saved;
  try {
    check_dofs(*s, spec);
    VFVM_HIP_CHECK(hipSetDevice(s->ctx->device));
    hipStream_t st = s->ctx->stream;
    const int ns = s->nspec, ispec = spec - 1;
    // d/dU of -integrate_stdy(T, U)[spec]: the Jacobian of flux, reaction and source
    // terms alone (no boundary conditions), tstep = Inf (src/vfvm_testfunctions.jl:398-410)
    saved = s->bc;
    for (auto &c : s->bc) c.kind = VFVM_BC_NONE;
    upload_inst(*s);
    s->d_U.upload(U0, (size_t)s->ndof, st);
    launch_fill_i32(1, s->d_flags.p, 0, st);
    AsmArgs a = asm_args(*s, s->d_U.p, s->d_U.p, s->d_F.p, s->d_J.p, INFINITY, lambda);
    run_assembly(*s, a, s->asm_group, st);
    s->bc = saved;
    saved.clear();
    upload_inst(*s);
    std::vector<int32_t> cp((size_t)s->ndof + 1);
    for (size_t j = 0; j < cp.size(); j++) cp[j] = (int32_t)s->csc_colptr[j];
    DevBuf<int32_t> dcp, drv;
    DevBuf<double> dT, dy;
    dcp.upload(cp, st);
    drv.upload(s->csc_rowval.empty() ? std::vector<int32_t>{0} : s->csc_rowval, st);
    dT.upload(T, (size_t)s->nnodes, st);
    dy.alloc((size_t)s->ndof);
    hipLaunchKernelGGL(k_meas_stdy, dim3((unsigned)((s->ndof + ZB - 1) / ZB)), dim3(ZB), 0, st, s->ndof, ns, ispec,
                       dcp.p, drv.p, s->d_csc_perm.p, s->d_J.p, dT.p, dy.p);
    VFVM_HIP_CHECK(hipGetLastError());
    dy.download(dstdy, (size_t)s->ndof, st);
    int32_t fl = 0;
    VFVM_HIP_CHECK(hipMemcpyAsync(&fl, s->d_flags.p, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    if (fl & 1) throw Error(VFVM_ERR_ASSEMBLY, "trying to assemble NaN");
    // d/dU of -integrate_tran(T, U)[spec]: storage derivative times node volume times T
    // (src/vfvm_testfunctions.jl:418-420)
    sync_host_geometry(*s);
    const double ds = s->phys.storage == VFVM_STOR_IDENTITY ? 1.0 : 0.0;
    for (int64_t j = 0; j < s->ndof; j++) dtran[j] = 0.0;
    for (int64_t K = 0; K < s->nnodes; K++) dtran[K * ns + ispec] = -ds * s->hs.nodevol[(size_t)K] * T[K];
    return VFVM_OK;
  } catch (const Error &e) {
    if (!saved.empty()) {
      s->bc = saved;
      try {
        upload_inst(*s);
      } catch (...) {
      }
    }
    s->ctx->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    s->ctx->err = e.what();
    return VFVM_ERR_HIP;
  }
}

int vfvm_integrate_testfunction(vfvm_sys *s, const double *U, const double *Uold, double tstep, const double *T,
                                double *result) {
  // integrate(system, T, U[, Uold, tstep]) evaluates at time 0 with embedding parameter 1
  // (src/vfvm_testfunctions.jl:232, Node(system, 0.0, 1.0))
  return vfvm_integrate_testfunction_at(s, U, Uold, tstep, T, 1.0, result);
}

int vfvm_integrate_testfunction_at(vfvm_sys *s, const double *U, const double *Uold, double tstep, const double *T,
                                   double lambda, double *result) {
  if (!s || !U || !T || !result || !(tstep > 0.0)) return VFVM_ERR_ARG;
  try {
    VFVM_HIP_CHECK(hipSetDevice(s->ctx->device));
    hipStream_t st = s->ctx->stream;
    s->d_U.upload(U, (size_t)s->ndof, st);
    s->d_Uold.upload(Uold ? Uold : U, (size_t)s->ndof, st);
    residual_without_bc(*s, s->d_U.p, s->d_Uold.p, tstep, lambda, s->d_tmp.p);
    DevBuf<double> dT, dr;
    dT.upload(T, (size_t)s->nnodes, st);
    dr.alloc((size_t)s->nspec);
    hipLaunchKernelGGL(k_tdot, dim3(1), dim3(ZB), 0, st, s->nnodes, s->nspec, dT.p, s->d_tmp.p, dr.p);
    VFVM_HIP_CHECK(hipGetLastError());
    dr.download(result, (size_t)s->nspec, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    return VFVM_OK;
  } catch (const Error &e) {
    s->ctx->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    s->ctx->err = e.what();
    return VFVM_ERR_HIP;
  }
}

namespace {

// one sweep's arguments and what it returns per frequency
struct Sweep {
  const double *omega, *dstdy, *dtran;
  double tol2;
  int maxiters;
  double2 *UZ, *Z;           // nullable
  std::vector<ZState> state;  // per frequency
};

double2 *grown(DevBuf<double2> &b, size_t n) {
  if (b.n < n) b.alloc(n);
  return b.p;
}

// The frequencies `list` by BiCGStab on the row-scaled operator alone (point Jacobi), all of
// them in one batch, each member's vectors contiguous.
void sweep_jacobi(vfvm_impedance *z, Sweep &sw, const std::vector<int> &list) {
  vfvm_sys *s = z->sys;
  hipStream_t st = s->ctx->stream;
  const int64_t n = z->n, nw = (int64_t)list.size();
  const int nblk = (int)std::min<int64_t>(ZMAXBLK, std::max<int64_t>(1, (n + ZB - 1) / ZB));
  std::vector<double> om((size_t)nw);
  for (int64_t w = 0; w < nw; w++) om[w] = sw.omega[list[w]];
  DevBuf<double> dom;
  dom.upload(om, st);
  const size_t nv = (size_t)(nw * n);
  double2 *X = grown(z->ws[0], nv), *R = grown(z->ws[1], nv), *R0 = grown(z->ws[2], nv), *P = grown(z->ws[3], nv),
          *V = grown(z->ws[4], nv), *S = grown(z->ws[5], nv), *T = grown(z->ws[6], nv);
  double2 *part = grown(z->part, (size_t)nw * nblk * 2);
  DevBuf<ZState> zst;
  zst.alloc((size_t)nw);
  const dim3 g2((unsigned)nblk, (unsigned)nw), gm((unsigned)nw);
  const dim3 gop((unsigned)nblk, (unsigned)((nw + ZMB - 1) / ZMB));
  int32_t *none = nullptr;
  hipLaunchKernelGGL(k_zinit, g2, dim3(ZB), 0, st, n, z->b.p, z->J.p, s->d_dofdiag.p, z->M.p, dom.p, X, R, R0, P,
                     part);
  hipLaunchKernelGGL((k_zfin<ZF_INIT, 2>), gm, dim3(ZB), 0, st, nblk, (int64_t)nblk, (int64_t)1, part, zst.p, sw.tol2,
                     0, none);
  std::vector<ZState> hz((size_t)nw);
  constexpr int CHECK = 10;
  int it = 0;
  bool all = false;
  while (it < sw.maxiters && !all) {
    const int nb = std::min(CHECK, sw.maxiters - it);
    for (int k = 0; k < nb; k++) {
      hipLaunchKernelGGL((k_zop<1>), gop, dim3(ZB), 0, st, n, (int)nw, s->d_rowptr.p, s->d_colind.p, z->J.p,
                         s->d_dofdiag.p, z->M.p, dom.p, P, V, R0, part, zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_ALPHA, 1>), gm, dim3(ZB), 0, st, nblk, (int64_t)nblk, (int64_t)1, part, zst.p,
                         sw.tol2, 0, none);
      hipLaunchKernelGGL(k_zs, g2, dim3(ZB), 0, st, n, R, V, S, zst.p);
      hipLaunchKernelGGL((k_zop<2>), gop, dim3(ZB), 0, st, n, (int)nw, s->d_rowptr.p, s->d_colind.p, z->J.p,
                         s->d_dofdiag.p, z->M.p, dom.p, S, T, S, part, zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_OMEGA, 2>), gm, dim3(ZB), 0, st, nblk, (int64_t)nblk, (int64_t)1, part, zst.p,
                         sw.tol2, 0, none);
      hipLaunchKernelGGL(k_zx, g2, dim3(ZB), 0, st, n, X, R, R0, P, S, T, part, zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_RHO, 2>), gm, dim3(ZB), 0, st, nblk, (int64_t)nblk, (int64_t)1, part, zst.p,
                         sw.tol2, 1, none);
      hipLaunchKernelGGL(k_zp, g2, dim3(ZB), 0, st, n, R, P, V, zst.p);
    }
    VFVM_HIP_CHECK(hipGetLastError());
    it += nb;
    zst.download(hz.data(), (size_t)nw, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    all = std::all_of(hz.begin(), hz.end(), [](const ZState &q) { return q.done != 0; });
  }
  for (int64_t w = 0; w < nw; w++) sw.state[list[w]] = hz[w];
  if (sw.UZ) {
    for (int64_t w = 0; w < nw; w++)
      VFVM_HIP_CHECK(hipMemcpyAsync(sw.UZ + (int64_t)list[w] * n, X + w * n, sizeof(double2) * n,
                                    hipMemcpyDeviceToHost, st));
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
  }
  if (sw.Z) {
    DevBuf<double> dds, ddt;
    DevBuf<double2> dZ;
    dds.upload(sw.dstdy, (size_t)n, st);
    ddt.upload(sw.dtran, (size_t)n, st);
    dZ.alloc((size_t)nw);
    hipLaunchKernelGGL(k_zmeas, g2, dim3(ZB), 0, st, n, dds.p, ddt.p, X, part);
    hipLaunchKernelGGL(k_zmeas_fin, gm, dim3(ZB), 0, st, nblk, (int64_t)nblk, (int64_t)1, part, dom.p, dZ.p);
    VFVM_HIP_CHECK(hipGetLastError());
    std::vector<double2> hZ((size_t)nw);
    dZ.download(hZ.data(), (size_t)nw, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    for (int64_t w = 0; w < nw; w++) sw.Z[list[w]] = hZ[w];
  }
}

// Frequencies of one group share a hierarchy, that of the real matrix K = J + sigma M: with
// omega within a factor ZG_SPAN of sigma, (lambda + i omega) / (lambda + sigma) stays bounded
// for every eigenvalue lambda of M^-1 J, whatever the grid, so the iteration count does not
// grow with either.  A wider span costs iterations, a narrower one launches and setups:
// 113 frequencies over 4.7 decades on 257 x 257 nodes took 34, 35, 32 and 27 ms with spans of
// 4, 8, 16 and 64 (12 to 19 iterations each; the Jacobi form takes 265 ms and 368 to 650).
// ZG_MAX members of that grid make vectors of 68 MB, a few of which fit the last-level cache.
constexpr double ZG_SPAN = 32.0;
constexpr int ZG_MAX = 64;
constexpr int ZG_ITERS = 100;   // iterations before a group's rest goes to the Jacobi form
// Rows from which the multigrid form is used.  Below, the hierarchy's symbolic setup (host,
// once per handle) and its launches per cycle cost more than the Jacobi form's iterations:
// 113 frequencies on 33 x 33 nodes 4.8 against 3.7 ms, 40 on 49 x 49 nodes 1.8 against 5.4 (3.4
// against 5.4 on the first sweep of a handle).
constexpr int64_t ZG_ROWS = 2048;

// One group by BiCGStab right-preconditioned with the multigrid V-cycle of K.  Frequencies it
// does not finish (breakdown, slow convergence, maxiters) keep done = 0 or breakdown = 1.
void sweep_multigrid(vfvm_impedance *z, Sweep &sw, const std::vector<int> &list, double sigma) {
  vfvm_sys *s = z->sys;
  hipStream_t st = s->ctx->stream;
  const int64_t n = z->n;
  const int nw = (int)list.size();
  const int32_t *rp = s->d_rowptr.p, *ci = s->d_colind.p, *dd = s->d_dofdiag.p;
  if (!z->amg.built()) {
    AmgMember m;
    m.n = n;
    m.rowptr = s->rowptr.data();
    m.colind = s->colind.data();
    z->amg.build({m}, nullptr, st, true);
    z->Ks.alloc((size_t)z->nnz);
    z->ks.alloc((size_t)n);
    z->sigma = -1.0;
  }
  if (z->sigma != sigma) {
    hipLaunchKernelGGL(k_zishift, dim3((unsigned)((n + ZB - 1) / ZB)), dim3(ZB), 0, st, n, rp, dd, z->J.p, z->M.p,
                       sigma, z->Ks.p, z->ks.p);
    z->sigma = -1.0;
    z->amg.setup(rp, ci, dd, z->Ks.p, z->ks.p, st);
    z->sigma = sigma;
  }
  std::vector<double> om((size_t)nw);
  for (int w = 0; w < nw; w++) om[w] = sw.omega[list[w]];
  DevBuf<double> dom;
  dom.upload(om, st);
  const size_t nv = (size_t)nw * n;
  double2 *X = grown(z->ws[0], nv), *R = grown(z->ws[1], nv), *R0 = grown(z->ws[2], nv), *P = grown(z->ws[3], nv),
          *V = grown(z->ws[4], nv), *S = grown(z->ws[5], nv), *T = grown(z->ws[6], nv), *Q = grown(z->ws[7], nv),
          *PH = grown(z->ws[8], nv), *SH = grown(z->ws[9], nv);
  const int rpb = ZB / nw;
  const int nblk = (int)std::min<int64_t>(2048, (n + rpb - 1) / rpb);
  double2 *part = grown(z->part, (size_t)nw * nblk * 2);
  if (z->skip.n < (size_t)ZG_MAX) z->skip.alloc(ZG_MAX);
  int32_t *skip = z->skip.p;
  DevBuf<ZState> zst;
  zst.alloc((size_t)nw);
  const dim3 g((unsigned)nblk), gm((unsigned)nw);
  const int64_t pw = 1, pb = nw;  // partials: block b, member w at b nw + w
  hipLaunchKernelGGL(k_ziinit, g, dim3(ZB), 0, st, n, nw, z->b.p, z->J.p, dd, z->M.p, dom.p, X, R, R0, P, V, part);
  hipLaunchKernelGGL((k_zfin<ZF_INIT, 2>), gm, dim3(ZB), 0, st, nblk, pw, pb, part, zst.p, sw.tol2, 0, skip);
  std::vector<ZState> hz((size_t)nw);
  const int cap = std::min(sw.maxiters, ZG_ITERS);
  for (int it = 0; it < cap;) {
    const int nb = std::min(it == 0 ? 4 : 2, cap - it);
    for (int k = 0; k < nb; k++) {
      hipLaunchKernelGGL((k_zivec<true>), g, dim3(ZB), 0, st, n, nw, z->J.p, dd, z->M.p, z->ks.p, dom.p, R, V, P, Q,
                         zst.p);
      z->amg.apply_columns(Q, PH, nw, rp, ci, skip, st);
      hipLaunchKernelGGL((k_ziop<1>), g, dim3(ZB), 0, st, n, nw, rp, ci, z->J.p, dd, z->M.p, dom.p, PH, V, R0, part,
                         zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_ALPHA, 1>), gm, dim3(ZB), 0, st, nblk, pw, pb, part, zst.p, sw.tol2, 0, skip);
      hipLaunchKernelGGL((k_zivec<false>), g, dim3(ZB), 0, st, n, nw, z->J.p, dd, z->M.p, z->ks.p, dom.p, R, V, S, Q,
                         zst.p);
      z->amg.apply_columns(Q, SH, nw, rp, ci, skip, st);
      hipLaunchKernelGGL((k_ziop<2>), g, dim3(ZB), 0, st, n, nw, rp, ci, z->J.p, dd, z->M.p, dom.p, SH, T, S, part,
                         zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_OMEGA, 2>), gm, dim3(ZB), 0, st, nblk, pw, pb, part, zst.p, sw.tol2, 0, skip);
      hipLaunchKernelGGL(k_zix, g, dim3(ZB), 0, st, n, nw, X, R, R0, PH, SH, S, T, part, zst.p);
      hipLaunchKernelGGL((k_zfin<ZF_RHO, 2>), gm, dim3(ZB), 0, st, nblk, pw, pb, part, zst.p, sw.tol2, 1, skip);
    }
    VFVM_HIP_CHECK(hipGetLastError());
    it += nb;
    zst.download(hz.data(), (size_t)nw, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    bool all = true, hope = it < 16;
    for (const ZState &q : hz) {
      all &= q.done != 0;
      hope |= !q.done && q.rn2 < 1e-2 * q.b2;
    }
    if (all || !hope) break;  // hope: a residual below a tenth after 16 iterations
  }
  for (int w = 0; w < nw; w++) sw.state[list[w]] = hz[w];
  if (sw.UZ) {
    double2 *Y = grown(z->ws[7], nv);
    hipLaunchKernelGGL(k_zitrans, dim3((unsigned)((nv + ZB - 1) / ZB)), dim3(ZB), 0, st, n, nw, X, Y);
    VFVM_HIP_CHECK(hipGetLastError());
    for (int w = 0; w < nw; w++)
      VFVM_HIP_CHECK(hipMemcpyAsync(sw.UZ + (int64_t)list[w] * n, Y + w * n, sizeof(double2) * n,
                                    hipMemcpyDeviceToHost, st));
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
  }
  if (sw.Z) {
    DevBuf<double> dds, ddt;
    DevBuf<double2> dZ;
    dds.upload(sw.dstdy, (size_t)n, st);
    ddt.upload(sw.dtran, (size_t)n, st);
    dZ.alloc((size_t)nw);
    hipLaunchKernelGGL(k_zimeas, g, dim3(ZB), 0, st, n, nw, dds.p, ddt.p, X, part);
    hipLaunchKernelGGL(k_zmeas_fin, gm, dim3(ZB), 0, st, nblk, pw, pb, part, dom.p, dZ.p);
    VFVM_HIP_CHECK(hipGetLastError());
    std::vector<double2> hZ((size_t)nw);
    dZ.download(hZ.data(), (size_t)nw, st);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    for (int w = 0; w < nw; w++) sw.Z[list[w]] = hZ[w];
  }
}

}  // namespace

int vfvm_impedance_sweep(vfvm_impedance *z, int64_t nw, const double *omega, const double *dstdy,
                         const double *dtran, double reltol, int32_t maxiters, double *UZ, double *Zout,
                         int32_t *iters) {
  if (!z || nw < 1 || !omega || maxiters < 1 || !(reltol > 0.0)) return VFVM_ERR_ARG;
  vfvm_sys *s = z->sys;
  try {
    VFVM_HIP_CHECK(hipSetDevice(s->ctx->device));
    if ((dstdy == nullptr) != (dtran == nullptr)) throw Error(VFVM_ERR_ARG, "give both measurement rows or none");
    if (nw > 65535) throw Error(VFVM_ERR_ARG, "at most 65535 frequencies per sweep");
    std::lock_guard<std::mutex> lock(z->mu);
    Sweep sw;
    sw.omega = omega;
    sw.dstdy = dstdy;
    sw.dtran = dtran;
    sw.tol2 = reltol * reltol;
    sw.maxiters = maxiters;
    sw.UZ = reinterpret_cast<double2 *>(UZ);
    sw.Z = dstdy ? reinterpret_cast<double2 *>(Zout) : nullptr;
    sw.state.resize((size_t)nw);
    std::vector<int> rest;
    // scalar systems with positive finite frequencies: the multigrid form, in groups of
    // ascending frequency; the others, and what it leaves unfinished, the Jacobi form
    for (int64_t w = 0; w < nw; w++) rest.push_back((int)w);
    if (s->nspec == 1 && z->n >= ZG_ROWS) {
      std::vector<int> order;
      order.swap(rest);
      std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return std::fabs(omega[a]) < std::fabs(omega[b]); });
      for (size_t k = 0; k < order.size();) {
        const double lo = std::fabs(omega[order[k]]);
        std::vector<int> group;
        if (!std::isfinite(lo)) {
          rest.push_back(order[k++]);
          continue;
        }
        while (k < order.size() && (int)group.size() < ZG_MAX &&
               std::fabs(omega[order[k]]) <= lo * ZG_SPAN * ZG_SPAN)
          group.push_back(order[k++]);
        sweep_multigrid(z, sw, group, std::sqrt(lo * std::fabs(omega[group.back()])));
        for (int w : group)
          if (!sw.state[w].done || sw.state[w].breakdown) rest.push_back(w);
      }
      std::sort(rest.begin(), rest.end());
    }
    if (!rest.empty()) {
      std::vector<int> spent((size_t)nw, 0);
      for (int w : rest) spent[w] = sw.state[w].iters;
      sweep_jacobi(z, sw, rest);
      for (int w : rest) sw.state[w].iters += spent[w];
    }
    if (iters)
      for (int64_t w = 0; w < nw; w++) iters[w] = sw.state[(size_t)w].iters;
    if (Zout && !dstdy) throw Error(VFVM_ERR_ARG, "the impedance needs the measurement rows");
    for (int64_t w = 0; w < nw; w++) {
      const ZState &q = sw.state[(size_t)w];
      if (!q.done || q.breakdown) {
        s->ctx->err = "impedance: frequency " + std::to_string(omega[w]) +
                      (q.breakdown ? ": BiCGStab breakdown" : ": no convergence within maxiters");
        return VFVM_ERR_LINEAR;
      }
    }
    return VFVM_OK;
  } catch (const Error &e) {
    s->ctx->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    s->ctx->err = e.what();
    return VFVM_ERR_HIP;
  }
}

}  // extern "C"
