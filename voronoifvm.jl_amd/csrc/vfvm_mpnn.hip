// Learned Newton initial guess: a message-passing network on the Voronoi edge
// graph of a system, with hand-written forward and backward kernels.  Dense
// layers run on the matrix cores (v_mfma_f32_16x16x16_bf16: bfloat16 operands,
// float32 accumulation); aggregation, activations, loss and Adam are plain
// kernels.  The network (row r = sample s, node i of the system's grid):
//
//   x_r   : 8 input features; channels 8..15 are multi-scale context: the features
//           a = x_1 (asinh(f/2)) and x_0 (f/5) smoothed by K = 16, 64, 160, 324 steps
//           of y <- (y + W y) / 2 on the graph (Gaussian-like, width sqrt(K)/2 edges)
//   h0    = relu(bf(x) We + be)                                   64 wide
//   l = 0..L-1:
//     a_l = sum_j w_ij h_l[j] - h_l[i]     w_ij = sigma_ij/h_ij normalised per row
//     c_l = [bf(h_l), bf(a_l)]                                    128 wide, bfloat16
//     r_l = relu(c_l W_l + b_l),  h_{l+1} = h_l + r_l
//   u     = h_L wd + bd
//
// Parameters live in one float32 vector (layout: We 16x64, be, [W_l 128x64, b_l]*L,
// wd 64, bd) with bfloat16 copies (W_l and its transpose) refreshed after every
// optimiser step.  Training minimises the mean squared error to converged Newton
// solutions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <random>
#include <vector>

#include "vfvm_sys.h"

using namespace vfvm;

namespace {

constexpr int NFEAT = 8;   // host-side input features
constexpr int KPAD = 16;   // padded input width (one MFMA k-step)
constexpr int WID = 64;    // hidden width
constexpr int CW = 2 * WID;  // concatenated width
constexpr int TB = 256;    // threads per block (4 waves)

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16_t;

__device__ __forceinline__ bf16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40u);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);                                          // round to nearest even
  return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// Workgroups are dealt to the 8 XCDs round-robin (workgroup b runs on XCD b % 8).  For a
// grid of G = 8k workgroups, logical block (b % 8) * k + b / 8 gives each XCD one
// contiguous range, so the graph neighbours a block gathers (nearby rows) are mostly
// in the same XCD's L2.
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t G) { return (b & 7) * (G >> 3) + (b >> 3); }

// ---------------------------------------------------------------- GEMM -----
// C[M x ND] = A[M x KD] * B[KD x ND], A and B bfloat16 row-major, float32
// accumulation on the matrix cores.  Block = 4 waves = 64 rows; wave w owns
// rows 16w..16w+15 and all ND columns (ND/16 accumulator tiles).  Both
// operands are staged in LDS (A rows padded by 8 to spread banks).
// Operand layout of v_mfma_f32_16x16x16_bf16 for lane l (g = l / 16, c = l % 16):
//   A: A[c][4g + j], B: B[4g + j][c], D: D[4g + j][c], j = 0..3.
enum { EPI_ENC = 0, EPI_RES = 1, EPI_DCAT = 2 };

struct GemmEpi {
  const float *bias;  // ND (ENC, RES)
  float *hf;          // rows x 64 hidden state (ENC: written, RES: updated in place)
  uint8_t *gate;      // rows x 64: relu(z) > 0, kept for the backward pass (RES)
  bf16_t *cat;        // rows x 128: ENC/RES write bf(h) into cols 0..63 of the next layer input
  float *dh;          // DCAT: dh += dC[:, 0:64]
  float *da;          // DCAT: da  = dC[:, 64:128]
};

template <int KD, int ND, int EPI>
__global__ void __launch_bounds__(TB) k_gemm(int64_t M, const bf16_t *__restrict__ A, const bf16_t *__restrict__ B,
                                             GemmEpi e) {
  constexpr int ASTR = KD + 8;
  __shared__ alignas(16) bf16_t As[64 * ASTR];
  __shared__ alignas(16) bf16_t Bs[KD * ND];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, g = l >> 4, c = l & 15;
  const int64_t row0 = (int64_t)blockIdx.x * 64;
  // B in operand order, one 8-byte fragment per k-step, column tile and lane: a thread transposes
  // a 4 x 4 patch
  for (int q = tid; q < KD * ND / 16; q += TB) {
    const int kq = q / (ND / 4), cq = q % (ND / 4);
    uint64_t v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = reinterpret_cast<const uint64_t *>(B + (4 * kq + i) * ND)[cq];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint64_t o = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) o |= ((v[i] >> (16 * j)) & 0xffffull) << (16 * i);
      const int col = 4 * cq + j;
      reinterpret_cast<uint64_t *>(Bs)[((kq >> 2) * (ND / 16) + (col >> 4)) * 64 + (kq & 3) * 16 + (col & 15)] = o;
    }
  }
  for (int q = tid; q < 64 * KD / 4; q += TB) {  // A tile rows, zero beyond M
    const int r = q / (KD / 4), kq = q % (KD / 4);
    uint64_t v = 0;
    if (row0 + r < M) v = reinterpret_cast<const uint64_t *>(A + (row0 + r) * KD)[kq];
    *reinterpret_cast<uint64_t *>(&As[r * ASTR + kq * 4]) = v;
  }
  __syncthreads();
  f32x4 acc[ND / 16];
#pragma unroll
  for (int t = 0; t < ND / 16; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k0 = 0; k0 < KD; k0 += 16) {
    const bf16x4 a = *reinterpret_cast<const bf16x4 *>(&As[(w * 16 + c) * ASTR + k0 + 4 * g]);
#pragma unroll
    for (int t = 0; t < ND / 16; t++) {
      const bf16x4 b = reinterpret_cast<const bf16x4 *>(Bs)[((k0 >> 4) * (ND / 16) + t) * 64 + l];
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < ND / 16; t++) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int64_t row = row0 + w * 16 + 4 * g + j;
      const int col = t * 16 + c;
      if (row >= M) continue;
      const float v = acc[t][j];
      if constexpr (EPI == EPI_ENC) {
        const float h = fmaxf(v + e.bias[col], 0.f);
        e.hf[row * WID + col] = h;
        if (e.cat) e.cat[row * CW + col] = f2bf(h);
      } else if constexpr (EPI == EPI_RES) {
        const float r = fmaxf(v + e.bias[col], 0.f);
        e.gate[row * WID + col] = r > 0.f;
        const float hn = e.hf[row * WID + col] + r;
        e.hf[row * WID + col] = hn;
        if (e.cat) e.cat[row * CW + col] = f2bf(hn);
      } else {
        if (col < WID)
          e.dh[row * WID + col] += v;
        else
          e.da[row * WID + col - WID] = v;
      }
    }
  }
}

// Weight gradient: P_b[KD x 64] = sum over the block's rows of A[rows x KD]^T Z[rows x 64],
// A and Z bfloat16.  Reduction over rows on the matrix cores (16 rows per step):
// A-operand A'[k][m] = A[m][k] (m = row), B-operand Z[m][n].  Output tiles
// (KD/16) x 4 are split over the 4 waves.  Both operands want four consecutive rows of one
// column per lane, so tiles are staged transposed: a thread loads a 4 x 4 patch (8 bytes of each
// of 4 rows) and stores its columns, and an operand is one 8-byte LDS read (as 4 separate
// 2-byte reads of untransposed tiles the kernel was bound by LDS).
template <int KD>
__device__ __forceinline__ void stage_transposed(int64_t r0, int64_t r_end, const bf16_t *__restrict__ A,
                                                 bf16_t *__restrict__ T, int tstr) {
  for (int q = threadIdx.x; q < 16 * (KD / 4); q += TB) {
    const int rq = q / (KD / 4), kq = q % (KD / 4);
    uint64_t v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int64_t row = r0 + 4 * rq + i;
      v[i] = row < r_end ? reinterpret_cast<const uint64_t *>(A + row * KD)[kq] : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint64_t o = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) o |= ((v[i] >> (16 * j)) & 0xffffull) << (16 * i);
      *reinterpret_cast<uint64_t *>(&T[(4 * kq + j) * tstr + 4 * rq]) = o;
    }
  }
}

template <int KD>
__global__ void __launch_bounds__(TB) k_wgrad(int64_t M, int64_t rows_per_block, const bf16_t *__restrict__ A,
                                              const bf16_t *__restrict__ Z, float *__restrict__ partials) {
  constexpr int NT = (KD / 16) * (WID / 16);
  constexpr int PER = (NT + 3) / 4;
  constexpr int STR = 64 + 4;  // rows of a tile, padded to spread the banks
  __shared__ alignas(16) bf16_t As[KD * STR];
  __shared__ alignas(16) bf16_t Zs[WID * STR];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, g = l >> 4, c = l & 15;
  f32x4 acc[PER];
#pragma unroll
  for (int p = 0; p < PER; p++) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int64_t r_begin = (int64_t)blockIdx.x * rows_per_block;
  const int64_t r_end = std::min<int64_t>(M, r_begin + rows_per_block);
  for (int64_t r0 = r_begin; r0 < r_end; r0 += 64) {
    __syncthreads();
    stage_transposed<KD>(r0, r_end, A, As, STR);
    stage_transposed<WID>(r0, r_end, Z, Zs, STR);
    __syncthreads();
#pragma unroll
    for (int m0 = 0; m0 < 64; m0 += 16) {
#pragma unroll
      for (int p = 0; p < PER; p++) {
        const int tile = w * PER + p;
        if (tile >= NT) break;
        const int kt = tile / (WID / 16), nt = tile % (WID / 16);
        const bf16x4 a = *reinterpret_cast<const bf16x4 *>(&As[(kt * 16 + c) * STR + m0 + 4 * g]);
        const bf16x4 b = *reinterpret_cast<const bf16x4 *>(&Zs[(nt * 16 + c) * STR + m0 + 4 * g]);
        acc[p] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[p], 0, 0, 0);
      }
    }
  }
  float *out = partials + (size_t)blockIdx.x * KD * WID;
#pragma unroll
  for (int p = 0; p < PER; p++) {
    const int tile = w * PER + p;
    if (tile >= NT) break;
    const int kt = tile / (WID / 16), nt = tile % (WID / 16);
#pragma unroll
    for (int j = 0; j < 4; j++) out[(kt * 16 + 4 * g + j) * WID + nt * 16 + c] = acc[p][j];
  }
}

// grad[k] = sum over blocks of partials[b][k]; 64 columns per block, 16 threads each (one thread
// per column waited for one load after the other: 130 us for 65 partials)
constexpr int SP_LANES = 16;
__global__ void __launch_bounds__(64 * SP_LANES) k_sum_partials(int nblocks, int len,
                                                                const float *__restrict__ partials,
                                                                float *__restrict__ grad) {
  __shared__ float sh[SP_LANES][64];
  const int c = threadIdx.x & 63, r = threadIdx.x >> 6, k = blockIdx.x * 64 + c;
  float acc = 0.f;
  if (k < len)
#pragma unroll 8
    for (int b = r; b < nblocks; b += SP_LANES) acc += partials[(size_t)b * len + k];
  sh[r][c] = acc;
  __syncthreads();
  if (r != 0 || k >= len) return;
  float t = 0.f;
#pragma unroll
  for (int q = 0; q < SP_LANES; q++) t += sh[q][c];
  grad[k] = t;
}

// ------------------------------------------------------------ graph ops ----
// Neighbour sums of a row's 4 features per lane (16 lanes and float4 a row, 4 rows a wave): the
// sums are in the order of the row's entries, with the loads of 4 entries issued together.  `at`
// is the sample's first row.
__device__ __forceinline__ f32x4 neighbour_sum(int32_t k0, int32_t k1, const int32_t *__restrict__ gcol,
                                               const float *__restrict__ gw, const float *__restrict__ h, uint32_t at,
                                               int f) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int32_t k = k0; k < k1; k += 4) {
    float w[4];
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {  // past the row's end: its last entry, not added
      const int32_t q = std::min(k + j, k1 - 1);
      w[j] = gw[q];
      v[j] = *reinterpret_cast<const f32x4 *>(h + (size_t)(at + (uint32_t)gcol[q]) * WID + f);
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (k + j < k1)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] += w[j] * v[j][e];
  }
  return acc;
}

// a_i = sum_j w_ij h_j - h_i for row r = s*n + i (rows < 2^32: the hidden state alone has 64
// floats a row).  The wave-per-row form with its 64-bit division took 97 us for 266,256 rows of
// a 2D grid, this one 25 us (with 68 MB read and 34 MB written: 20 us).
__global__ void __launch_bounds__(TB) k_aggregate(uint32_t rows, uint32_t n, const int32_t *__restrict__ gptr,
                                                  const int32_t *__restrict__ gcol, const float *__restrict__ gw,
                                                  const float *__restrict__ hf, bf16_t *__restrict__ cat) {
  const uint32_t row = blockIdx.x * (TB / 16) + (threadIdx.x >> 4);
  const int f = 4 * (threadIdx.x & 15);
  if (row >= rows) return;
  const uint32_t i = row % n;
  const f32x4 self = *reinterpret_cast<const f32x4 *>(hf + (size_t)row * WID + f);
  const f32x4 acc = neighbour_sum(gptr[i], gptr[i + 1], gcol, gw, hf, row - i, f) - self;
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = (short)f2bf(acc[e]);
  *reinterpret_cast<bf16x4 *>(cat + (size_t)row * CW + WID + f) = o;
}

// dh_k += sum_{i in N(k)} w_ik da_i - da_k  (transpose weights gwt on k's entries)
__global__ void __launch_bounds__(TB) k_aggregate_t(uint32_t rows, uint32_t n, const int32_t *__restrict__ gptr,
                                                    const int32_t *__restrict__ gcol, const float *__restrict__ gwt,
                                                    const float *__restrict__ da, float *__restrict__ dh) {
  const uint32_t row = blockIdx.x * (TB / 16) + (threadIdx.x >> 4);
  const int f = 4 * (threadIdx.x & 15);
  if (row >= rows) return;
  const uint32_t k = row % n;
  const f32x4 self = *reinterpret_cast<const f32x4 *>(da + (size_t)row * WID + f);
  f32x4 *d = reinterpret_cast<f32x4 *>(dh + (size_t)row * WID + f);
  const f32x4 old = *d;
  *d = old + (neighbour_sum(gptr[k], gptr[k + 1], gcol, gwt, da, row - k, f) - self);
}

// One hidden layer for inference, aggregation fused into the GEMM: for a tile of 64
// consecutive rows, c = [bf(h_l), bf(sum_j w_ij h_l[j] - h_l[i])] is built in LDS
// (same arithmetic as k_aggregate), multiplied on the matrix cores by W_l, and
// h_{l+1} = h_l + relu(c W_l + b_l) is written to `hout` (a buffer other than `hin`:
// neighbouring tiles still read h_l).  With `wd` set (last layer) the tile writes
// u = h_{l+1} . wd + bd instead.  Blocks loop over tiles; W_l sits in LDS in operand
// order (one 8-byte fragment per lane, k-step and column tile).  Each thread stages
// four (row, 4-column chunk) items and loads the first NB0 neighbours of two items
// before summing them, so 8 neighbour rows are in flight per thread.
constexpr int NB0 = 4;
__global__ void __launch_bounds__(TB, 4) k_layer_infer(int64_t rows, int64_t n, const int32_t *__restrict__ gptr,
                                                    const int32_t *__restrict__ gcol, const float *__restrict__ gw,
                                                    const float *__restrict__ hin, const bf16_t *__restrict__ W,
                                                    const float *__restrict__ bias, float *__restrict__ hout,
                                                    const float *__restrict__ wd, const float *__restrict__ bd,
                                                    float *__restrict__ u) {
  constexpr int ASTR = CW + 8;  // bf16 per LDS row of the layer input
  constexpr int KS = CW / 16, NTL = WID / 16;
  __shared__ alignas(16) bf16_t As[64 * ASTR];
  __shared__ uint64_t Bf[KS * NTL * 64];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, g = l >> 4, c = l & 15;
  for (int q = tid; q < KS * NTL * 64; q += TB) {
    const int k = q / (NTL * 64), t = (q / 64) % NTL, ln = q % 64, gg = ln >> 4, cc = ln & 15;
    uint64_t v = 0;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) v |= (uint64_t)W[(k * 16 + 4 * gg + jj) * WID + t * 16 + cc] << (16 * jj);
    Bf[q] = v;
  }
  float bcol[NTL], wdc[NTL];
#pragma unroll
  for (int t = 0; t < NTL; t++) {
    bcol[t] = bias[t * 16 + c];
    wdc[t] = wd ? wd[t * 16 + c] : 0.f;
  }
  // XCD x takes the contiguous tile range [x T, (x + 1) T), T = ceil(ntiles / 8), in
  // steps of the grid's blocks per XCD
  const int64_t ntiles = (rows + 63) / 64, per = (ntiles + 7) / 8, G8 = gridDim.x / 8;
  const int64_t t_end = std::min<int64_t>(ntiles, (int64_t)(blockIdx.x & 7) * per + per);
  for (int64_t tile = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3); tile < t_end; tile += G8) {
    const int64_t row0 = tile * 64;
    __syncthreads();  // Bf is written; the previous tile's As reads are done
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 hv[4], av[4];
    int64_t base[4];
    int32_t kb[4], ke[4];
#pragma unroll
    for (int it = 0; it < 4; it++) {
      const int q = tid + it * TB, r = q >> 4, ch = q & 15;
      const int64_t row = row0 + r;
      hv[it] = z4;
      av[it] = z4;
      base[it] = ch * 4;
      kb[it] = 0;
      ke[it] = 0;
      if (row < rows) {
        const int64_t smp = row / n, i = row - smp * n;
        base[it] = smp * n * WID + ch * 4;
        hv[it] = *reinterpret_cast<const float4 *>(hin + row * WID + ch * 4);
        kb[it] = gptr[i];
        ke[it] = gptr[i + 1];
      }
    }
#pragma unroll
    for (int p2 = 0; p2 < 4; p2 += 2) {
      // first NB0 neighbours of two items: indices clamped to entry 0 where absent
      // (a valid node of the same sample), skipped in the sum
      float4 v[2][NB0];
      float wk[2][NB0];
#pragma unroll
      for (int it = 0; it < 2; it++)
#pragma unroll
        for (int jj = 0; jj < NB0; jj++) {
          const int32_t kk = kb[p2 + it] + jj;
          const int32_t kc = kk < ke[p2 + it] ? kk : 0;
          wk[it][jj] = gw[kc];
          v[it][jj] = *reinterpret_cast<const float4 *>(hin + base[p2 + it] + (int64_t)gcol[kc] * WID);
        }
#pragma unroll
      for (int it = 0; it < 2; it++)
#pragma unroll
        for (int jj = 0; jj < NB0; jj++)
          if (kb[p2 + it] + jj < ke[p2 + it]) {
            av[p2 + it].x += wk[it][jj] * v[it][jj].x;
            av[p2 + it].y += wk[it][jj] * v[it][jj].y;
            av[p2 + it].z += wk[it][jj] * v[it][jj].z;
            av[p2 + it].w += wk[it][jj] * v[it][jj].w;
          }
    }
#pragma unroll
    for (int it = 0; it < 4; it++) {
      for (int32_t k = kb[it] + NB0; k < ke[it]; k++) {
        const float wv = gw[k];
        const float4 v = *reinterpret_cast<const float4 *>(hin + base[it] + (int64_t)gcol[k] * WID);
        av[it].x += wv * v.x;
        av[it].y += wv * v.y;
        av[it].z += wv * v.z;
        av[it].w += wv * v.w;
      }
      const int q = tid + it * TB, r = q >> 4, ch = q & 15;
      bf16_t *ar = &As[r * ASTR + ch * 4];
      ar[0] = f2bf(hv[it].x);
      ar[1] = f2bf(hv[it].y);
      ar[2] = f2bf(hv[it].z);
      ar[3] = f2bf(hv[it].w);
      ar[WID + 0] = f2bf(av[it].x - hv[it].x);
      ar[WID + 1] = f2bf(av[it].y - hv[it].y);
      ar[WID + 2] = f2bf(av[it].z - hv[it].z);
      ar[WID + 3] = f2bf(av[it].w - hv[it].w);
    }
    __syncthreads();
    f32x4 acc[NTL];
#pragma unroll
    for (int t = 0; t < NTL; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; k++) {
      bf16x4 a;
      const bf16_t *ap = &As[(w * 16 + c) * ASTR + k * 16 + 4 * g];
#pragma unroll
      for (int jj = 0; jj < 4; jj++) a[jj] = (short)ap[jj];
#pragma unroll
      for (int t = 0; t < NTL; t++) {
        const uint64_t bv = Bf[(k * NTL + t) * 64 + l];
        bf16x4 b;
#pragma unroll
        for (int jj = 0; jj < 4; jj++) b[jj] = (short)(uint16_t)(bv >> (16 * jj));
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
      }
    }
    // epilogue: lane holds rows w*16 + 4g + jj, columns t*16 + c; h_l re-read from
    // memory (the tile was just staged, so from cache)
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
      const int64_t row = row0 + w * 16 + 4 * g + jj;
      const bool ok = row < rows;
      float ud = 0.f;
#pragma unroll
      for (int t = 0; t < NTL; t++) {
        const int col = t * 16 + c;
        const float h = ok ? hin[row * WID + col] : 0.f;
        const float hn = h + fmaxf(acc[t][jj] + bcol[t], 0.f);
        if (!wd) {
          if (ok) hout[row * WID + col] = hn;
        } else {
          ud += hn * wdc[t];
        }
      }
      if (wd) {
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) ud += __shfl_xor(ud, o, 16);
        if (c == 0 && ok) u[row] = ud + bd[0];
      }
    }
  }
}

// The 8 input features of a 2D family with one source field and a Dirichlet value
// per side of the bounding box, computed on the device (row r = sample r / n, node
// r % n): f / 5, asinh(f / 2), side value k * exp(-distance to side k / delta)
// (k = south, east, north, west), x, y.  The host-side definition is identical.
__global__ void k_features_sides(int64_t rows, int64_t n, const double *__restrict__ f,
                                 const double *__restrict__ sides, const float *__restrict__ xy,
                                 const float *__restrict__ dist, double inv_delta, float *__restrict__ x) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const int64_t smp = r / n, i = r - smp * n;
  const double fv = f[r];
  float *o = x + r * NFEAT;
  o[0] = (float)(fv / 5.0);
  o[1] = (float)asinh(fv / 2.0);
#pragma unroll
  for (int k = 0; k < 4; k++) o[2 + k] = (float)sides[smp * 4 + k] * (float)exp(-(double)dist[i * 4 + k] * inv_delta);
  o[6] = xy[2 * i];
  o[7] = xy[2 * i + 1];
}

// network input (rows x 16 float) -> bfloat16
__global__ void k_pad_features(int64_t rows, const float *__restrict__ x16, bf16_t *__restrict__ xb) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= rows * KPAD) return;
  xb[q] = f2bf(x16[q]);
}

// ---------------------------------------------------------- context -------
// Channels 8..15 of the network input: two features smoothed on the graph by
// K = 16, 64, 160, 324 steps of y <- (y + W y) / 2.  All samples share the graph, so
// the fields of a launch are kept node-major, Y[i][col] with col = c * ns + s (feature
// c, sample s): a wave takes one node and 64 columns, the node's graph entries are
// wave-uniform and every field load is a coalesced row segment.  One launch per step.
constexpr int SMOOTH_STEPS_H[4] = {16, 64, 160, 324};
constexpr int SMOOTH_SRC[2] = {1, 0};  // asinh(f/2), f/5

// x16[r, 0..7] = x[r, 0..7]
__global__ void k_expand_copy(int64_t rows, const float *__restrict__ x, float *__restrict__ x16) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= rows * KPAD) return;
  const int64_t r = q / KPAD;
  const int k = (int)(q % KPAD);
  if (k < NFEAT) x16[q] = x[r * NFEAT + k];
}

// Y[i][c ns + s] = x16[s n + i][src_c]  (to node-major; row stride Cs >= 2 ns, a multiple
// of 4, padding columns zero), or back: x16[..][slot_c] = Y
template <bool TO_NODE_MAJOR>
__global__ void k_smooth_io(int64_t n, int64_t ns, int64_t Cs, float *__restrict__ x16, float *__restrict__ Y,
                            int snap) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n * Cs) return;
  const int64_t i = q / Cs, col = q - i * Cs;
  if (col >= 2 * ns) {
    if (TO_NODE_MAJOR) Y[q] = 0.f;
    return;
  }
  const int c = (int)(col / ns);
  const int64_t s = col - (int64_t)c * ns;
  float *xr = x16 + (s * n + i) * KPAD;
  if (TO_NODE_MAJOR)
    Y[q] = xr[c == 0 ? SMOOTH_SRC[0] : SMOOTH_SRC[1]];
  else
    xr[NFEAT + 4 * c + snap] = Y[q];
}

// one step: Yo[i][:] = (Yi[i][:] + sum_j w_ij Yi[j][:]) / 2.  A wave takes one node (its
// graph entries are wave-uniform) and walks the row in float4 columns; the neighbour
// rows are loaded four at a time and summed in entry order.
__global__ void __launch_bounds__(256) k_smooth_step(int64_t n, int64_t C4, const int32_t *__restrict__ gptr,
                                                     const int32_t *__restrict__ gcol,
                                                     const float *__restrict__ gw, const float4 *__restrict__ Yi,
                                                     float4 *__restrict__ Yo) {
  const int64_t i = __builtin_amdgcn_readfirstlane(
      (int)(xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6)));
  if (i >= n) return;
  const int32_t k0 = gptr[i], k1 = gptr[i + 1];
  for (int64_t c4 = (int64_t)blockIdx.y * 64 + (threadIdx.x & 63); c4 < C4; c4 += (int64_t)gridDim.y * 64) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    int32_t k = k0;
    for (; k + 4 <= k1; k += 4) {
      float wk[4];
      float4 v[4];
#pragma unroll
      for (int jj = 0; jj < 4; jj++) {
        wk[jj] = gw[k + jj];
        v[jj] = Yi[(int64_t)gcol[k + jj] * C4 + c4];
      }
#pragma unroll
      for (int jj = 0; jj < 4; jj++) {
        acc.x += wk[jj] * v[jj].x;
        acc.y += wk[jj] * v[jj].y;
        acc.z += wk[jj] * v[jj].z;
        acc.w += wk[jj] * v[jj].w;
      }
    }
    for (; k < k1; k++) {
      const float wv = gw[k];
      const float4 v = Yi[(int64_t)gcol[k] * C4 + c4];
      acc.x += wv * v.x;
      acc.y += wv * v.y;
      acc.z += wv * v.z;
      acc.w += wv * v.w;
    }
    const float4 y = Yi[i * C4 + c4];
    Yo[i * C4 + c4] = make_float4(0.5f * (y.x + acc.x), 0.5f * (y.y + acc.y), 0.5f * (y.z + acc.z),
                                  0.5f * (y.w + acc.w));
  }
}

// All smoothing steps of a field in one launch, the field resident in LDS: a block takes one
// sample (FPB = 2 features, interleaved) or one feature of a sample (FPB = 1).  The nodes
// whose graph row is the grid's most frequent one (four entries with the same neighbour
// offsets and weights: the inside of a 2D tensor grid) form groups of 64, up to NG per wave,
// so a wave's offsets and weights are scalars; the other nodes (sides and corners) form at
// most one further group per wave, whose lanes carry their own entries in registers.  A
// node's own value stays in a register.  Sums run in entry order as in k_smooth_step, so both
// give the same bits.
// Bound: LDS (four reads and a write per node and step, about 64 bytes a cycle with 4-byte
// and 85 with 8-byte accesses, so two features together cost 1.5 times one).  Pairs of
// consecutive nodes per lane, with three two-word reads instead of eight one-word ones, took
// the same time.  Measured on 129 x 129 nodes, with the copies to and from the node-major
// fields of the launch-per-step form: 0.70 ms instead of 1.85 for one sample, 2.2 ms instead
// of 9.4 for 512.
constexpr int CTX_T = 1024;            // threads per block
constexpr int CTX_W = CTX_T / 64;      // waves per block
constexpr int64_t CTX_LDS = 160 * 1024;
constexpr int CTX_D = 4;               // graph entries of a node
struct CtxGraph {
  int nmain, nmix;      // groups of main nodes; groups of other nodes (at most CTX_W)
  int off[CTX_D];       // the main row's neighbour offsets (in nodes) and weights
  float w[CTX_D];
  const int32_t *node;  // (nmain + nmix) x 64 nodes; a short group repeats its last node
                        // (same value, same place)
  const int32_t *mdeg;  // nmix x 64: entries of the node, then their columns and weights
  const int32_t *mcol;  // nmix x 64 x CTX_D
  const float *mw;
};

template <int FPB>
struct CtxVal;
template <>
struct CtxVal<1> {
  using T = float;
  static __device__ __forceinline__ T fma(float w, T y, T a) { return a + w * y; }
  static __device__ __forceinline__ T half(T y, T a) { return 0.5f * (y + a); }
  static __device__ __forceinline__ T zero() { return 0.f; }
};
template <>
struct CtxVal<2> {
  using T = float2;
  static __device__ __forceinline__ T fma(float w, T y, T a) {
    a.x += w * y.x;
    a.y += w * y.y;
    return a;
  }
  static __device__ __forceinline__ T half(T y, T a) { return make_float2(0.5f * (y.x + a.x), 0.5f * (y.y + a.y)); }
  static __device__ __forceinline__ T zero() { return make_float2(0.f, 0.f); }
};

// x: rows x 8 features; P: 8 planes of `rows` values, plane 4 c + k = feature c after
// SMOOTH_STEPS_H[k] steps
template <int FPB, int NG>
__global__ void __launch_bounds__(CTX_T) k_context(int64_t n, int64_t rows, CtxGraph G, const float *__restrict__ x,
                                                   float *__restrict__ P) {
  using CV = CtxVal<FPB>;
  using T = typename CV::T;
  extern __shared__ __attribute__((aligned(16))) unsigned char ctx_lds[];
  T *Y = reinterpret_cast<T *>(ctx_lds);
  const int64_t smp = FPB == 2 ? blockIdx.x : blockIdx.x >> 1;
  const int c0 = FPB == 2 ? 0 : blockIdx.x & 1;
  const float *xs = x + smp * n * NFEAT;
  for (int i = threadIdx.x; i < (int)n; i += CTX_T) {
    if constexpr (FPB == 2)
      Y[i] = make_float2(xs[(int64_t)i * NFEAT + SMOOTH_SRC[0]], xs[(int64_t)i * NFEAT + SMOOTH_SRC[1]]);
    else
      Y[i] = xs[(int64_t)i * NFEAT + (c0 == 0 ? SMOOTH_SRC[0] : SMOOTH_SRC[1])];
  }
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // main groups w, w + CTX_W, ...: every wave has as many, or one more
  int cnt = __builtin_amdgcn_readfirstlane(w < G.nmain ? (G.nmain - w + CTX_W - 1) / CTX_W : 0);
  uint32_t nd[(NG + 1) / 2];  // the lane's nodes in them, as pairs of 16 bits
#pragma unroll
  for (int q = 0; q < NG; q++) {
    const uint32_t v = q < cnt ? (uint32_t)G.node[(w + q * CTX_W) * 64 + lane] : 0;
    nd[q / 2] = q % 2 ? nd[q / 2] | (v << 16) : v;
  }
  auto node = [&](int q) -> int { return q % 2 ? (int)(nd[q / 2] >> 16) : (int)(nd[q / 2] & 0xffffu); };
  // the wave's group of other nodes
  const bool mix = w < G.nmix;
  int mnode = 0, mdeg = 0, mcol[CTX_D] = {0, 0, 0, 0};
  float mw[CTX_D] = {0.f, 0.f, 0.f, 0.f};
  if (mix) {
    const int k = w * 64 + lane;
    mnode = G.node[(int64_t)G.nmain * 64 + k];
    mdeg = G.mdeg[k];
#pragma unroll
    for (int e = 0; e < CTX_D; e++) {
      mcol[e] = G.mcol[k * CTX_D + e];
      mw[e] = G.mw[k * CTX_D + e];
    }
  }
  const int o0 = G.off[0], o1 = G.off[1], o2 = G.off[2], o3 = G.off[3];
  const float w0 = G.w[0], w1 = G.w[1], w2 = G.w[2], w3 = G.w[3];
  __syncthreads();
  T nv[NG], mv = CV::zero();
#pragma unroll
  for (int q = 0; q < NG; q++) nv[q] = q < cnt ? Y[node(q)] : CV::zero();
  if (mix) mv = Y[mnode];
  int snap = 0;
  for (int step = 1; step <= SMOOTH_STEPS_H[3]; step++) {
    // hides that cnt is loop-invariant (the compiler would keep a mask per group in scalar
    // registers), and the node numbers where the addresses of every group would not fit the
    // vector registers: they are then formed again in each step.  The branch on cnt also
    // keeps the compiler from issuing the loads of all groups at once, which spills (without
    // it, 512 samples of 129 x 129 nodes took 12 ms instead of 2.2).
    asm volatile("" : "+s"(cnt));
    if constexpr (NG * FPB > 16) {
#pragma unroll
      for (int q = 0; q < (NG + 1) / 2; q++) asm volatile("" : "+v"(nd[q]));
    }
#pragma unroll
    for (int q = 0; q < NG; q++)
      if (q < cnt) {  // wave-uniform
        const int i = node(q);
        const T y0 = Y[i + o0], y1 = Y[i + o1], y2 = Y[i + o2], y3 = Y[i + o3];
        T acc = CV::fma(w0, y0, CV::zero());
        acc = CV::fma(w1, y1, acc);
        acc = CV::fma(w2, y2, acc);
        acc = CV::fma(w3, y3, acc);
        nv[q] = CV::half(nv[q], acc);
      }
    if (mix) {
      T acc = CV::zero();
#pragma unroll
      for (int e = 0; e < CTX_D; e++) {
        const T t = CV::fma(mw[e], Y[mcol[e]], acc);
        if (e < mdeg) acc = t;
      }
      mv = CV::half(mv, acc);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NG; q++)
      if (q < cnt) Y[node(q)] = nv[q];
    if (mix) Y[mnode] = mv;
    if (step == SMOOTH_STEPS_H[snap]) {
      float *o = P + (int64_t)(4 * c0 + snap) * rows + smp * n;
      auto put = [&](int i, T v) {
        if constexpr (FPB == 2) {
          o[i] = v.x;
          o[4 * rows + i] = v.y;
        } else {
          o[i] = v;
        }
      };
#pragma unroll
      for (int q = 0; q < NG; q++)
        if (q < cnt) put(node(q), nv[q]);
      if (mix) put(mnode, mv);
      snap++;
    }
    __syncthreads();
  }
}

// x16 = [x, P]: the network input from the features and the context planes
__global__ void k_pack16(int64_t rows, const float *__restrict__ x, const float *__restrict__ P,
                         float *__restrict__ x16) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= rows * KPAD) return;
  const int64_t r = q / KPAD;
  const int k = (int)(q % KPAD);
  x16[q] = k < NFEAT ? x[r * NFEAT + k] : P[(int64_t)(k - NFEAT) * rows + r];
}

// u_r = h_L[r] . wd + bd (one wave per row), du = 2 (u - t) / count, dh = du wd; per-block
// partials (float64) of sum du h (64), sum (u-t)^2 and sum du over DEC_ROWS rows
constexpr int DEC_ROWS = 256;
__global__ void __launch_bounds__(TB) k_decode(int64_t rows, const float *__restrict__ hf, const float *__restrict__ wd,
                                               const float *__restrict__ bd, float *__restrict__ u,
                                               const float *__restrict__ target, float inv_count,
                                               float *__restrict__ dh, double *__restrict__ part) {
  __shared__ double sh_s[4][2];
  __shared__ double sh_g[4][WID];
  const int w = threadIdx.x >> 6, f = threadIdx.x & 63;
  const int64_t r0 = (int64_t)blockIdx.x * DEC_ROWS;
  const int64_t r1 = std::min<int64_t>(rows, r0 + DEC_ROWS);
  const float wf = wd[f], b0 = bd[0];
  double g = 0.0, sd = 0.0, lo = 0.0;
#pragma unroll 4
  for (int64_t row = r0 + w; row < r1; row += 4) {
    const float hv = hf[row * WID + f], t = target[row];
    float v = hv * wf;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const float uu = v + b0;
    if (f == 0) u[row] = uu;
    const float d = uu - t, du = 2.f * d * inv_count;
    dh[row * WID + f] = du * wf;
    g += (double)(du * hv);
    lo += (double)(d * d);
    sd += (double)du;
  }
  sh_g[w][f] = g;
  if (f == 0) {
    sh_s[w][0] = lo;
    sh_s[w][1] = sd;
  }
  __syncthreads();
  double *pb = part + (size_t)blockIdx.x * (WID + 2);
  if (w == 0) pb[f] = (sh_g[0][f] + sh_g[1][f]) + (sh_g[2][f] + sh_g[3][f]);
  if (w == 1 && f < 2) pb[WID + f] = (sh_s[0][f] + sh_s[1][f]) + (sh_s[2][f] + sh_s[3][f]);
}

// decoder gradient (wd, then bd) and the loss sum from the partials; one block per value
__global__ void __launch_bounds__(TB) k_decode_sum(int nblocks, const double *__restrict__ part,
                                                   float *__restrict__ grad, double *__restrict__ loss) {
  __shared__ double sh[TB / 64];
  double a = 0.0;
#pragma unroll 4
  for (int b = threadIdx.x; b < nblocks; b += TB) a += part[(size_t)b * (WID + 2) + blockIdx.x];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double t = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  const int q = blockIdx.x;
  if (q < WID) grad[q] = (float)t;
  if (q == WID) loss[0] = t;
  if (q == WID + 1) grad[WID] = (float)t;
}

// dz = dh where the gate is open -> bfloat16; per-block column sums of dz (bias gradient).  The
// gate is the layer's byte per value or, for the encoder, bf(h0) > 0 in the first half of cat_0.
// 16 lanes and 4 columns each per row.
template <bool GATE_BF>
__global__ void __launch_bounds__(TB) k_gate(int64_t rows, const float *__restrict__ dh,
                                             const uint8_t *__restrict__ gate, const bf16_t *__restrict__ gate_bf,
                                             bf16_t *__restrict__ dzb, float *__restrict__ part, int rows_per_block) {
  constexpr int RL = TB / 16;
  __shared__ f32x4 sh[RL][16];
  const int w = threadIdx.x >> 4, q = threadIdx.x & 15, f = 4 * q;
  const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
  const int64_t r1 = std::min<int64_t>(rows, r0 + rows_per_block);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int64_t row = r0 + w; row < r1; row += RL) {
    const f32x4 d = *reinterpret_cast<const f32x4 *>(dh + row * WID + f);
    bf16x4 o;
    uint32_t gb = 0;
    bf16x4 gh = {0, 0, 0, 0};
    if constexpr (GATE_BF)
      gh = *reinterpret_cast<const bf16x4 *>(gate_bf + row * CW + f);
    else
      gb = *reinterpret_cast<const uint32_t *>(gate + row * WID + f);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const bool on = GATE_BF ? bf2f((bf16_t)gh[e]) > 0.f : ((gb >> (8 * e)) & 0xffu) != 0;
      const float dz = on ? d[e] : 0.f;
      o[e] = (short)f2bf(dz);
      acc[e] += dz;
    }
    *reinterpret_cast<bf16x4 *>(dzb + row * WID + f) = o;
  }
  sh[w][q] = acc;
  __syncthreads();
  if (w != 0) return;
  f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < RL; k++) t += sh[k][q];
  *reinterpret_cast<f32x4 *>(part + (size_t)blockIdx.x * WID + f) = t;
}

// Adam on the float32 parameters (t = step count, bias-corrected)
__global__ void k_adam(int64_t n, float *__restrict__ theta, const float *__restrict__ grad, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const float g = grad[k];
  const float mk = b1 * m[k] + (1.f - b1) * g;
  const float vk = b2 * v[k] + (1.f - b2) * g * g;
  m[k] = mk;
  v[k] = vk;
  theta[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

// bfloat16 copies: W (K x N) as is and transposed
__global__ void k_cast(int K, int N, const float *__restrict__ W, bf16_t *__restrict__ Wb, bf16_t *__restrict__ WTb) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= K * N) return;
  const int k = q / N, j = q % N;
  const bf16_t b = f2bf(W[q]);
  Wb[q] = b;
  if (WTb) WTb[j * K + k] = b;
}

__global__ void k_fill_f(int64_t n, float *p, float v) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

// u (float, rows) -> out (double)
__global__ void k_to_double(int64_t rows, const float *__restrict__ u, double *__restrict__ out) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < rows) out[r] = (double)u[r];
}

}  // namespace

struct vfvm_mpnn {
  vfvm_ctx *ctx = nullptr;
  int nlayers = 4;
  int64_t n = 0;  // nodes per sample
  int64_t np = 0;
  // graph
  DevBuf<int32_t> gptr, gcol;
  DevBuf<float> gw, gwt;
  // the graph as k_context takes it (nmain 0: it does not)
  CtxGraph ctxg{};
  DevBuf<int32_t> ctx_node, ctx_mdeg, ctx_mcol;
  DevBuf<float> ctx_mw, planes;
  // parameters
  DevBuf<float> theta, grad, adam_m, adam_v;
  int64_t adam_t = 0;
  DevBuf<bf16_t> Web, Wb, WTb;  // encoder; layers (L x 128 x 64) and transposes (L x 64 x 128)
  // activations for a batch of `cap` rows
  int64_t cap = 0;
  DevBuf<float> x, x16, hf, dh, da, u, target, part, sm0, sm1;
  DevBuf<uint8_t> gate;
  DevBuf<double> dpart, dloss;
  DevBuf<bf16_t> xb, cat, dzb;
  // device features of the Dirichlet-sides family (2D): per node x, y and the distances
  // to the bounding-box sides (south, east, north, west); per-sample inputs
  DevBuf<float> xy, dist;
  DevBuf<double> fin, sides;
  size_t off_We = 0, off_be = 0, off_wd = 0, off_bd = 0;
  std::vector<size_t> off_W, off_b;
};

namespace {

template <class F>
int mguard(vfvm_ctx *ctx, F &&f) {
  try {
    return f();
  } catch (const Error &e) {
    if (ctx) ctx->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    if (ctx) ctx->err = e.what();
    return VFVM_ERR_HIP;
  }
}

inline unsigned nb(int64_t n, int64_t t) { return (unsigned)((n + t - 1) / t); }

void refresh_bf16(vfvm_mpnn &m) {
  hipStream_t st = m.ctx->stream;
  hipLaunchKernelGGL(k_cast, dim3(nb(KPAD * WID, 256)), dim3(256), 0, st, KPAD, WID, (const float *)m.theta.p + m.off_We,
                     m.Web.p, (bf16_t *)nullptr);
  for (int l = 0; l < m.nlayers; l++)
    hipLaunchKernelGGL(k_cast, dim3(nb(CW * WID, 256)), dim3(256), 0, st, CW, WID,
                       (const float *)m.theta.p + m.off_W[l], m.Wb.p + (size_t)l * CW * WID,
                       m.WTb.p + (size_t)l * CW * WID);
  VFVM_HIP_CHECK(hipGetLastError());
}

// samples per inference launch sequence: at most MAX_INFER_ROWS rows, the samples split
// into chunks of equal size (a short last chunk would pay every launch of the smoothing
// and the layers for a few samples)
constexpr int64_t MAX_INFER_ROWS = int64_t(1) << 24;
inline int64_t sample_chunk(int64_t nsamples, int64_t n) {
  const int64_t most = std::max<int64_t>(1, MAX_INFER_ROWS / n);
  const int64_t nchunk = (nsamples + most - 1) / most;
  return std::max<int64_t>(1, (nsamples + nchunk - 1) / nchunk);
}

// Blocks of the weight-gradient kernels: two per compute unit (with 4096 rows a block, 266,256 rows
// gave 65 blocks and 418 us; now 37 us, of which 21 for 102 MB), but at least 256 rows, as each block writes a whole
// gradient (32 KB) of partial sums.
constexpr int64_t WG_BLOCKS = 512, WG_MIN_ROWS = 256;
inline int64_t wgrad_rows(int64_t rows) {
  return std::max<int64_t>(WG_MIN_ROWS, ((rows + WG_BLOCKS - 1) / WG_BLOCKS + 63) / 64 * 64);
}
constexpr int GATE_ROWS = 256;     // rows per block of the gate kernel

void ensure_cap(vfvm_mpnn &m, int64_t rows) {
  if (rows <= m.cap) return;
  const int L = m.nlayers;
  m.x.alloc((size_t)rows * NFEAT);
  m.x16.alloc((size_t)rows * KPAD);
  m.xb.alloc((size_t)rows * KPAD);
  m.hf.alloc((size_t)rows * WID);
  m.gate.alloc((size_t)rows * WID * L);
  m.dh.alloc((size_t)rows * WID);
  m.da.alloc((size_t)rows * WID);
  m.u.alloc((size_t)rows);
  m.target.alloc((size_t)rows);
  m.cat.alloc((size_t)rows * CW * (L + 1));
  m.dzb.alloc((size_t)rows * WID);
  const int64_t p1 = std::min<int64_t>(WG_BLOCKS, nb(rows, WG_MIN_ROWS)) * CW * WID;
  const int64_t p2 = (int64_t)nb(rows, GATE_ROWS) * WID;
  m.part.alloc((size_t)std::max(p1, p2));
  m.dpart.alloc((size_t)nb(rows, DEC_ROWS) * (WID + 2));
  m.dloss.alloc(1);
  m.cap = rows;
}

// host values into a workspace buffer of at least `count` entries (ensure_cap): the buffer
// keeps its capacity, which later calls with more rows rely on.  Synchronous, as
// DevBuf::upload.
template <class T>
void copy_in(DevBuf<T> &buf, const T *h, size_t count, hipStream_t st) {
  VFVM_HIP_CHECK(hipMemcpyAsync(buf.p, h, count * sizeof(T), hipMemcpyHostToDevice, st));
  VFVM_HIP_CHECK(hipStreamSynchronize(st));
}

// The node groups of k_context: taken where the most frequent graph row has CTX_D entries, no
// row has more, and the nodes with other rows fit one group per wave.  That holds for the 2D
// tensor grids that fit the LDS (up to 202 x 202 nodes); unstructured and 3D grids keep one
// launch per step.
void build_context_groups(vfvm_mpnn &m, const std::vector<int32_t> &ptr, const std::vector<int32_t> &col,
                          const std::vector<float> &w) {
  m.ctxg.nmain = 0;
  if (m.n < 1 || m.n * (int64_t)sizeof(float) > CTX_LDS) return;
  using Row = std::vector<std::pair<int32_t, uint32_t>>;  // offset and weight bits per entry
  std::map<Row, int64_t> count;
  auto row_of = [&](int64_t i) {
    Row row;
    for (int32_t k = ptr[i]; k < ptr[i + 1]; k++) {
      uint32_t bits;
      std::memcpy(&bits, &w[k], sizeof(bits));
      row.emplace_back((int32_t)(col[k] - i), bits);
    }
    return row;
  };
  for (int64_t i = 0; i < m.n; i++) {
    if (ptr[i + 1] - ptr[i] > CTX_D) return;
    count[row_of(i)]++;
    if ((int64_t)count.size() > (int64_t)CTX_T + 1) return;
  }
  auto main = count.begin();
  for (auto it = count.begin(); it != count.end(); ++it)
    if (it->second > main->second) main = it;
  const Row &mr = main->first;
  if ((int)mr.size() != CTX_D || m.n - main->second > (int64_t)CTX_T) return;
  std::vector<int32_t> node, rest;
  for (int64_t i = 0; i < m.n; i++) (row_of(i) == mr ? node : rest).push_back((int32_t)i);
  while (node.size() % 64) node.push_back(node.back());
  const int nmain = (int)(node.size() / 64);
  while (rest.size() % 64) rest.push_back(rest.back());
  const int nmix = (int)(rest.size() / 64);
  std::vector<int32_t> mdeg(rest.size()), mcol(rest.size() * CTX_D);
  std::vector<float> mw(rest.size() * CTX_D, 0.f);
  for (size_t k = 0; k < rest.size(); k++) {
    const int32_t i = rest[k];
    mdeg[k] = ptr[i + 1] - ptr[i];
    for (int e = 0; e < CTX_D; e++) mcol[k * CTX_D + e] = i;  // absent entries read the node itself
    for (int32_t q = ptr[i]; q < ptr[i + 1]; q++) {
      mcol[k * CTX_D + (q - ptr[i])] = col[q];
      mw[k * CTX_D + (q - ptr[i])] = w[q];
    }
  }
  node.insert(node.end(), rest.begin(), rest.end());
  hipStream_t st = m.ctx->stream;
  m.ctx_node.upload(node, st);
  if (nmix) {
    m.ctx_mdeg.upload(mdeg, st);
    m.ctx_mcol.upload(mcol, st);
    m.ctx_mw.upload(mw, st);
  }
  CtxGraph &g = m.ctxg;
  for (int e = 0; e < CTX_D; e++) {
    g.off[e] = mr[e].first;
    std::memcpy(&g.w[e], &mr[e].second, sizeof(float));
  }
  g.node = m.ctx_node.p;
  g.mdeg = m.ctx_mdeg.p;
  g.mcol = m.ctx_mcol.p;
  g.mw = m.ctx_mw.p;
  g.nmix = nmix;
  g.nmain = nmain;
}

// The context planes of `ns` samples into m.planes, or false where k_context does not take
// the graph.  Both features of a sample in one block once that gives every CU a block (256
// CUs), while both fit the LDS.
bool context_planes(vfvm_mpnn &m, const float *x, int64_t ns) {
  if (m.ctxg.nmain == 0) return false;
  hipStream_t st = m.ctx->stream;
  const int64_t rows = ns * m.n;
  const bool two = 2 * ns > 256 && m.n * (int64_t)sizeof(float2) <= CTX_LDS;
  if (m.planes.n < (size_t)(rows * 8)) m.planes.alloc((size_t)(rows * 8));
  auto launch = [&](auto fpb, auto ng) {
    constexpr int FPB = decltype(fpb)::value, NG = decltype(ng)::value;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_context<FPB, NG>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)CTX_LDS);
    VFVM_HIP_CHECK(attr);
    hipLaunchKernelGGL((k_context<FPB, NG>), dim3((unsigned)(FPB == 2 ? ns : 2 * ns)), dim3(CTX_T),
                       (size_t)m.n * sizeof(float) * FPB, st, m.n, rows, m.ctxg, x, m.planes.p);
  };
  // registers grow with NG: the smallest that holds the groups of a wave
  const int need = (m.ctxg.nmain + CTX_W - 1) / CTX_W;
  auto go = [&](auto ng) {
    if constexpr (decltype(ng)::value <= 20) {  // both features: at most 20480 nodes
      if (two) {
        launch(std::integral_constant<int, 2>(), ng);
        return;
      }
    }
    launch(std::integral_constant<int, 1>(), ng);
  };
  if (need <= 5)
    go(std::integral_constant<int, 5>());
  else if (need <= 10)
    go(std::integral_constant<int, 10>());
  else if (need <= 16)
    go(std::integral_constant<int, 16>());
  else if (need <= 20)
    go(std::integral_constant<int, 20>());
  else if (need <= 30)
    go(std::integral_constant<int, 30>());
  else
    go(std::integral_constant<int, 40>());
  VFVM_HIP_CHECK(hipGetLastError());
  return true;
}

// network input of `ns` samples: x16 = [x (8 features), smoothed context (8 channels)]
void expand(vfvm_mpnn &m, const float *x, float *x16, int64_t ns) {
  hipStream_t st = m.ctx->stream;
  if (context_planes(m, x, ns)) {
    hipLaunchKernelGGL(k_pack16, dim3(nb(ns * m.n * KPAD, 256)), dim3(256), 0, st, ns * m.n, x,
                       (const float *)m.planes.p, x16);
    VFVM_HIP_CHECK(hipGetLastError());
    return;
  }
  const int64_t rows = ns * m.n, Cs = (2 * ns + 3) / 4 * 4, C4 = Cs / 4;
  hipLaunchKernelGGL(k_expand_copy, dim3(nb(rows * KPAD, 256)), dim3(256), 0, st, rows, x, x16);
  m.sm0.alloc((size_t)std::max<int64_t>(m.n * Cs, (int64_t)m.sm0.n));
  m.sm1.alloc((size_t)std::max<int64_t>(m.n * Cs, (int64_t)m.sm1.n));
  hipLaunchKernelGGL((k_smooth_io<true>), dim3(nb(m.n * Cs, 256)), dim3(256), 0, st, m.n, ns, Cs, x16, m.sm0.p, 0);
  float *a = m.sm0.p, *b = m.sm1.p;
  const unsigned gy = (unsigned)std::max<int64_t>(1, std::min<int64_t>(C4 / 256, 64));
  int snap = 0;
  for (int step = 1; step <= SMOOTH_STEPS_H[3]; step++) {
    hipLaunchKernelGGL(k_smooth_step, dim3((nb(m.n, 4) + 7) / 8 * 8, gy), dim3(256), 0, st, m.n, C4, (const int32_t *)m.gptr.p,
                       (const int32_t *)m.gcol.p, (const float *)m.gw.p, (const float4 *)a, (float4 *)b);
    std::swap(a, b);
    if (step == SMOOTH_STEPS_H[snap]) {
      hipLaunchKernelGGL((k_smooth_io<false>), dim3(nb(m.n * Cs, 256)), dim3(256), 0, st, m.n, ns, Cs, x16, a,
                         snap);
      snap++;
    }
  }
  VFVM_HIP_CHECK(hipGetLastError());
}

// forward pass on `rows` rows whose network input is in m.x16; keeps what the backward pass needs
void forward(vfvm_mpnn &m, int64_t rows) {
  hipStream_t st = m.ctx->stream;
  const int L = m.nlayers;
  hipLaunchKernelGGL(k_pad_features, dim3(nb(rows * KPAD, 256)), dim3(256), 0, st, rows, (const float *)m.x16.p,
                     m.xb.p);
  GemmEpi e{};
  e.bias = m.theta.p + m.off_be;
  e.hf = m.hf.p;
  e.cat = m.cat.p;  // cat_0 first half = bf(h0)
  hipLaunchKernelGGL((k_gemm<KPAD, WID, EPI_ENC>), dim3(nb(rows, 64)), dim3(TB), 0, st, rows, (const bf16_t *)m.xb.p,
                     (const bf16_t *)m.Web.p, e);
  for (int l = 0; l < L; l++) {
    bf16_t *cl = m.cat.p + (size_t)l * rows * CW;
    hipLaunchKernelGGL(k_aggregate, dim3(nb(rows, TB / 16)), dim3(TB), 0, st, (uint32_t)rows, (uint32_t)m.n, (const int32_t *)m.gptr.p,
                       (const int32_t *)m.gcol.p, (const float *)m.gw.p, (const float *)m.hf.p, cl);
    GemmEpi r{};
    r.bias = m.theta.p + m.off_b[l];
    r.hf = m.hf.p;
    r.gate = m.gate.p + (size_t)l * rows * WID;
    r.cat = m.cat.p + (size_t)(l + 1) * rows * CW;  // next layer's h half (cat_L unused by the decoder)
    hipLaunchKernelGGL((k_gemm<CW, WID, EPI_RES>), dim3(nb(rows, 64)), dim3(TB), 0, st, rows, (const bf16_t *)cl,
                       (const bf16_t *)(m.Wb.p + (size_t)l * CW * WID), r);
  }
  VFVM_HIP_CHECK(hipGetLastError());
}

// inference: encoder, then the fused layers ping-ponging hf / dh; u = network output
void forward_infer(vfvm_mpnn &m, int64_t rows) {
  hipStream_t st = m.ctx->stream;
  const int L = m.nlayers;
  hipLaunchKernelGGL(k_pad_features, dim3(nb(rows * KPAD, 256)), dim3(256), 0, st, rows, (const float *)m.x16.p,
                     m.xb.p);
  GemmEpi e{};
  e.bias = m.theta.p + m.off_be;
  e.hf = m.hf.p;
  hipLaunchKernelGGL((k_gemm<KPAD, WID, EPI_ENC>), dim3(nb(rows, 64)), dim3(TB), 0, st, rows, (const bf16_t *)m.xb.p,
                     (const bf16_t *)m.Web.p, e);
  const unsigned grid = (unsigned)std::min<int64_t>((nb(rows, 64) + 7) / 8 * 8, 2048);  // a multiple of 8
  float *hin = m.hf.p, *hout = m.dh.p;
  for (int l = 0; l < L; l++) {
    const bool last = l == L - 1;
    hipLaunchKernelGGL(k_layer_infer, dim3(grid), dim3(TB), 0, st, rows, m.n, (const int32_t *)m.gptr.p,
                       (const int32_t *)m.gcol.p, (const float *)m.gw.p, (const float *)hin,
                       (const bf16_t *)(m.Wb.p + (size_t)l * CW * WID), (const float *)m.theta.p + m.off_b[l],
                       last ? (float *)nullptr : hout, last ? (const float *)m.theta.p + m.off_wd : nullptr,
                       last ? (const float *)m.theta.p + m.off_bd : nullptr, last ? m.u.p : (float *)nullptr);
    std::swap(hin, hout);
  }
  VFVM_HIP_CHECK(hipGetLastError());
}

// loss and full gradient (into m.grad) for `rows` rows with targets in m.target
float backward(vfvm_mpnn &m, int64_t rows) {
  hipStream_t st = m.ctx->stream;
  const int L = m.nlayers;
  const unsigned dblk = nb(rows, DEC_ROWS);
  hipLaunchKernelGGL(k_decode, dim3(dblk), dim3(TB), 0, st, rows, (const float *)m.hf.p,
                     (const float *)m.theta.p + m.off_wd, (const float *)m.theta.p + m.off_bd, m.u.p,
                     (const float *)m.target.p, 1.0f / (float)rows, m.dh.p, m.dpart.p);
  hipLaunchKernelGGL(k_decode_sum, dim3(WID + 2), dim3(TB), 0, st, (int)dblk, (const double *)m.dpart.p,
                     m.grad.p + m.off_wd, m.dloss.p);
  const int64_t wg_rows = wgrad_rows(rows);
  const unsigned wg_blocks = nb(rows, wg_rows);
  const unsigned gate_blocks = nb(rows, GATE_ROWS);
  for (int l = L - 1; l >= 0; l--) {
    const bf16_t *cl = m.cat.p + (size_t)l * rows * CW;
    hipLaunchKernelGGL((k_gate<false>), dim3(gate_blocks), dim3(TB), 0, st, rows, (const float *)m.dh.p,
                       (const uint8_t *)m.gate.p + (size_t)l * rows * WID, (const bf16_t *)nullptr, m.dzb.p, m.part.p,
                       GATE_ROWS);
    hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(64 * SP_LANES), 0, st, (int)gate_blocks, WID, (const float *)m.part.p,
                       m.grad.p + m.off_b[l]);
    hipLaunchKernelGGL((k_wgrad<CW>), dim3(wg_blocks), dim3(TB), 0, st, rows, wg_rows, cl, (const bf16_t *)m.dzb.p,
                       m.part.p);
    hipLaunchKernelGGL(k_sum_partials, dim3(CW * WID / 64), dim3(64 * SP_LANES), 0, st, (int)wg_blocks, CW * WID,
                       (const float *)m.part.p, m.grad.p + m.off_W[l]);
    GemmEpi e{};
    e.dh = m.dh.p;
    e.da = m.da.p;
    hipLaunchKernelGGL((k_gemm<WID, CW, EPI_DCAT>), dim3(nb(rows, 64)), dim3(TB), 0, st, rows, (const bf16_t *)m.dzb.p,
                       (const bf16_t *)(m.WTb.p + (size_t)l * CW * WID), e);
    hipLaunchKernelGGL(k_aggregate_t, dim3(nb(rows, TB / 16)), dim3(TB), 0, st, (uint32_t)rows, (uint32_t)m.n, (const int32_t *)m.gptr.p,
                       (const int32_t *)m.gcol.p, (const float *)m.gwt.p, (const float *)m.da.p, m.dh.p);
  }
  // encoder: gate from bf(h0) in cat_0
  hipLaunchKernelGGL((k_gate<true>), dim3(gate_blocks), dim3(TB), 0, st, rows, (const float *)m.dh.p,
                     (const uint8_t *)nullptr, (const bf16_t *)m.cat.p, m.dzb.p, m.part.p, GATE_ROWS);
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(64 * SP_LANES), 0, st, (int)gate_blocks, WID, (const float *)m.part.p,
                     m.grad.p + m.off_be);
  hipLaunchKernelGGL((k_wgrad<KPAD>), dim3(wg_blocks), dim3(TB), 0, st, rows, wg_rows, (const bf16_t *)m.xb.p,
                     (const bf16_t *)m.dzb.p, m.part.p);
  hipLaunchKernelGGL(k_sum_partials, dim3(KPAD * WID / 64), dim3(64 * SP_LANES), 0, st, (int)wg_blocks, KPAD * WID,
                     (const float *)m.part.p, m.grad.p + m.off_We);
  VFVM_HIP_CHECK(hipGetLastError());
  double loss = 0.0;
  VFVM_HIP_CHECK(hipMemcpyAsync(&loss, m.dloss.p, sizeof(double), hipMemcpyDeviceToHost, st));
  VFVM_HIP_CHECK(hipStreamSynchronize(st));
  return (float)(loss / (double)rows);
}

// inference with the Dirichlet-sides features computed on the device from the sources f
// (nsamples x n) and the side values (nsamples x 4); host or device arrays
int infer_sides_impl(vfvm_mpnn *m, int64_t nsamples, const double *f, const double *sides, double eps, double *out,
                     bool on_device) {
  return mguard(m->ctx, [&]() {
    if (!m->xy.p) throw Error(VFVM_ERR_ARG, "side features need a 2D system");
    hipStream_t st = m->ctx->stream;
    const int64_t chunk = sample_chunk(nsamples, m->n);
    const double inv_delta = 1.0 / std::sqrt(eps / 2.0);
    std::vector<float> u;
    for (int64_t s0 = 0; s0 < nsamples; s0 += chunk) {
      const int64_t ns = std::min(chunk, nsamples - s0), rows = ns * m->n;
      ensure_cap(*m, rows);
      const double *fp = f + s0 * m->n, *sp = sides + s0 * 4;
      if (!on_device) {
        m->fin.upload(fp, (size_t)rows, st);
        m->sides.upload(sp, (size_t)ns * 4, st);
        fp = m->fin.p;
        sp = m->sides.p;
      }
      hipLaunchKernelGGL(k_features_sides, dim3(nb(rows, 256)), dim3(256), 0, st, rows, m->n, fp, sp,
                         (const float *)m->xy.p, (const float *)m->dist.p, inv_delta, m->x.p);
      expand(*m, m->x.p, m->x16.p, ns);
      forward_infer(*m, rows);
      if (on_device) {
        hipLaunchKernelGGL(k_to_double, dim3(nb(rows, 256)), dim3(256), 0, st, rows, (const float *)m->u.p,
                           out + s0 * m->n);
        VFVM_HIP_CHECK(hipGetLastError());
      } else {
        u.resize((size_t)rows);
        m->u.download(u.data(), (size_t)rows, st);
        VFVM_HIP_CHECK(hipStreamSynchronize(st));
        for (int64_t k = 0; k < rows; k++) out[s0 * m->n + k] = (double)u[k];
      }
    }
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    return VFVM_OK;
  });
}

}  // namespace

extern "C" {

int vfvm_mpnn_create(vfvm_sys *sys, int nlayers, int width, uint64_t seed, vfvm_mpnn **out) {
  if (!sys || !out) return VFVM_ERR_ARG;
  return mguard(sys->ctx, [&]() {
    if (width != WID) throw Error(VFVM_ERR_ARG, "the network width is fixed at 64");
    if (nlayers < 1 || nlayers > 16) throw Error(VFVM_ERR_ARG, "nlayers must be 1..16");
    std::unique_ptr<vfvm_mpnn> m(new vfvm_mpnn());
    m->ctx = sys->ctx;
    m->nlayers = nlayers;
    m->n = sys->nnodes;
    // normalised graph weights from the system's node graph (sigma/h factors)
    sync_host_geometry(*sys);
    const HostSetup &h = sys->hs;
    std::vector<int32_t> ptr((size_t)m->n + 1, 0), col;
    std::vector<float> w, wt;
    std::vector<double> rowsum((size_t)m->n, 0.0);
    for (int64_t i = 0; i < m->n; i++)
      for (int32_t k = h.adj_ptr[i]; k < h.adj_ptr[i + 1]; k++)
        if (h.adj_col[k] != i) rowsum[i] += h.adj_fac[k];
    for (int64_t i = 0; i < m->n; i++) {
      for (int32_t k = h.adj_ptr[i]; k < h.adj_ptr[i + 1]; k++) {
        const int32_t j = h.adj_col[k];
        if (j == i) continue;
        col.push_back(j);
        w.push_back(rowsum[i] > 0 ? (float)(h.adj_fac[k] / rowsum[i]) : 0.f);
        wt.push_back(rowsum[j] > 0 ? (float)(h.adj_fac[k] / rowsum[j]) : 0.f);  // w_ji on i's entry
      }
      ptr[i + 1] = (int32_t)col.size();
    }
    hipStream_t st = m->ctx->stream;
    if (sys->dim == 2) {
      const double *X = sys->coord.data();
      double lo[2] = {X[0], X[1]}, hi[2] = {X[0], X[1]};
      for (int64_t i = 0; i < m->n; i++)
        for (int d = 0; d < 2; d++) {
          lo[d] = std::min(lo[d], X[2 * i + d]);
          hi[d] = std::max(hi[d], X[2 * i + d]);
        }
      std::vector<float> xy((size_t)m->n * 2), dist((size_t)m->n * 4);
      for (int64_t i = 0; i < m->n; i++) {
        const double x = X[2 * i], y = X[2 * i + 1];
        xy[2 * i] = (float)x;
        xy[2 * i + 1] = (float)y;
        dist[4 * i + 0] = (float)(y - lo[1]);
        dist[4 * i + 1] = (float)(hi[0] - x);
        dist[4 * i + 2] = (float)(hi[1] - y);
        dist[4 * i + 3] = (float)(x - lo[0]);
      }
      m->xy.upload(xy, st);
      m->dist.upload(dist, st);
    }
    m->gptr.upload(ptr, st);
    m->gcol.upload(col.empty() ? std::vector<int32_t>{0} : col, st);
    m->gw.upload(w.empty() ? std::vector<float>{0.f} : w, st);
    m->gwt.upload(wt.empty() ? std::vector<float>{0.f} : wt, st);
    build_context_groups(*m, ptr, col, w);
    // parameter layout and He-uniform initialisation
    size_t p = 0;
    m->off_We = p;
    p += KPAD * WID;
    m->off_be = p;
    p += WID;
    for (int l = 0; l < nlayers; l++) {
      m->off_W.push_back(p);
      p += CW * WID;
      m->off_b.push_back(p);
      p += WID;
    }
    m->off_wd = p;
    p += WID;
    m->off_bd = p;
    p += 1;
    m->np = (int64_t)p;
    std::vector<float> th(p, 0.f);
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    for (int k = 0; k < KPAD * WID; k++)
      th[m->off_We + k] = U(rng) * std::sqrt(6.f / KPAD);
    for (int l = 0; l < nlayers; l++)
      for (int k = 0; k < CW * WID; k++) th[m->off_W[l] + k] = U(rng) * std::sqrt(6.f / CW) * 0.5f;
    for (int k = 0; k < WID; k++) th[m->off_wd + k] = U(rng) * std::sqrt(3.f / WID);
    m->theta.upload(th, st);
    m->grad.alloc(p);
    m->adam_m.alloc(p);
    m->adam_v.alloc(p);
    hipLaunchKernelGGL(k_fill_f, dim3(nb(p, 256)), dim3(256), 0, st, (int64_t)p, m->adam_m.p, 0.f);
    hipLaunchKernelGGL(k_fill_f, dim3(nb(p, 256)), dim3(256), 0, st, (int64_t)p, m->adam_v.p, 0.f);
    hipLaunchKernelGGL(k_fill_f, dim3(nb(p, 256)), dim3(256), 0, st, (int64_t)p, m->grad.p, 0.f);
    m->Web.alloc(KPAD * WID);
    m->Wb.alloc((size_t)nlayers * CW * WID);
    m->WTb.alloc((size_t)nlayers * CW * WID);
    refresh_bf16(*m);
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    *out = m.release();
    return VFVM_OK;
  });
}

int vfvm_mpnn_destroy(vfvm_mpnn *m) {
  if (!m) return VFVM_OK;
  (void)hipStreamSynchronize(m->ctx->stream);
  delete m;
  return VFVM_OK;
}

int vfvm_mpnn_params(vfvm_mpnn *m, int64_t *nparams, float *params) {
  if (!m) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    if (nparams) *nparams = m->np;
    if (params) {
      m->theta.download(params, (size_t)m->np, m->ctx->stream);
      VFVM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
    }
    return VFVM_OK;
  });
}

int vfvm_mpnn_set_params(vfvm_mpnn *m, const float *params) {
  if (!m || !params) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    m->theta.upload(params, (size_t)m->np, m->ctx->stream);
    refresh_bf16(*m);
    VFVM_HIP_CHECK(hipStreamSynchronize(m->ctx->stream));
    return VFVM_OK;
  });
}

int vfvm_mpnn_infer(vfvm_mpnn *m, int64_t nsamples, const float *features, double *out) {
  if (!m || !features || !out || nsamples < 1) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    hipStream_t st = m->ctx->stream;
    const int64_t chunk = sample_chunk(nsamples, m->n);
    std::vector<float> u;
    for (int64_t s0 = 0; s0 < nsamples; s0 += chunk) {
      const int64_t ns = std::min(chunk, nsamples - s0), rows = ns * m->n;
      ensure_cap(*m, rows);
      copy_in(m->x, features + s0 * m->n * NFEAT, (size_t)rows * NFEAT, st);
      expand(*m, m->x.p, m->x16.p, ns);
      forward_infer(*m, rows);
      u.resize((size_t)rows);
      m->u.download(u.data(), (size_t)rows, st);
      VFVM_HIP_CHECK(hipStreamSynchronize(st));
      for (int64_t k = 0; k < rows; k++) out[s0 * m->n + k] = (double)u[k];
    }
    return VFVM_OK;
  });
}

int vfvm_mpnn_infer_sides(vfvm_mpnn *m, int64_t nsamples, const double *f, const double *sides, double eps,
                          double *out) {
  if (!m || !f || !sides || !out || nsamples < 1 || !(eps > 0)) return VFVM_ERR_ARG;
  return infer_sides_impl(m, nsamples, f, sides, eps, out, false);
}

int vfvm_mpnn_infer_sides_device(vfvm_mpnn *m, int64_t nsamples, const double *f_dev, const double *sides_dev,
                                 double eps, double *out_dev) {
  if (!m || !f_dev || !sides_dev || !out_dev || nsamples < 1 || !(eps > 0)) return VFVM_ERR_ARG;
  return infer_sides_impl(m, nsamples, f_dev, sides_dev, eps, out_dev, true);
}

// average device time (ms) of one inference hidden layer (k_layer_infer, not the last)
// over `rows` rows of the current hidden state
int vfvm_mpnn_time_layer(vfvm_mpnn *m, int64_t rows, int reps, double *avg_ms) {
  if (!m || rows < 1 || reps < 1 || !avg_ms) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    if (rows % m->n != 0) throw Error(VFVM_ERR_ARG, "rows must be a whole number of samples");
    hipStream_t st = m->ctx->stream;
    ensure_cap(*m, rows);
    const unsigned grid = (unsigned)std::min<int64_t>((nb(rows, 64) + 7) / 8 * 8, 2048);
    auto once = [&]() {
      hipLaunchKernelGGL(k_layer_infer, dim3(grid), dim3(TB), 0, st, rows, m->n, (const int32_t *)m->gptr.p,
                         (const int32_t *)m->gcol.p, (const float *)m->gw.p, (const float *)m->hf.p,
                         (const bf16_t *)m->Wb.p, (const float *)m->theta.p + m->off_b[0], m->dh.p,
                         (const float *)nullptr, (const float *)nullptr, (float *)nullptr);
    };
    hipLaunchKernelGGL(k_fill_f, dim3(nb(rows * WID, 256)), dim3(256), 0, st, rows * WID, m->hf.p, 0.5f);
    once();
    hipEvent_t e0, e1;
    VFVM_HIP_CHECK(hipEventCreate(&e0));
    VFVM_HIP_CHECK(hipEventCreate(&e1));
    VFVM_HIP_CHECK(hipEventRecord(e0, st));
    for (int k = 0; k < reps; k++) once();
    VFVM_HIP_CHECK(hipEventRecord(e1, st));
    VFVM_HIP_CHECK(hipEventSynchronize(e1));
    float ms = 0;
    VFVM_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *avg_ms = (double)ms / reps;
    return VFVM_OK;
  });
}

int vfvm_mpnn_loss_grad(vfvm_mpnn *m, int64_t nsamples, const float *features, const float *targets, float *loss,
                        float *grad) {
  if (!m || !features || !targets || nsamples < 1) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    hipStream_t st = m->ctx->stream;
    const int64_t rows = nsamples * m->n;
    ensure_cap(*m, rows);
    copy_in(m->x, features, (size_t)rows * NFEAT, st);
    copy_in(m->target, targets, (size_t)rows, st);
    expand(*m, m->x.p, m->x16.p, nsamples);
    forward(*m, rows);
    const float lv = backward(*m, rows);
    if (loss) *loss = lv;
    if (grad) {
      m->grad.download(grad, (size_t)m->np, st);
      VFVM_HIP_CHECK(hipStreamSynchronize(st));
    }
    return VFVM_OK;
  });
}

int vfvm_mpnn_train(vfvm_mpnn *m, int64_t nsamples, const float *features, const float *targets, int64_t epochs,
                    int64_t batch, float lr, float *final_loss) {
  if (!m || !features || !targets || nsamples < 1 || batch < 1 || epochs < 1) return VFVM_ERR_ARG;
  return mguard(m->ctx, [&]() {
    hipStream_t st = m->ctx->stream;
    const int64_t n = m->n;
    // the whole training set (with its smoothed context channels) stays resident on the device
    DevBuf<float> X, X16, T;
    X.upload(features, (size_t)nsamples * n * NFEAT, st);
    X16.alloc((size_t)nsamples * n * KPAD);
    const int64_t ech = std::max<int64_t>(1, (int64_t(1) << 22) / n);
    for (int64_t s0 = 0; s0 < nsamples; s0 += ech)
      expand(*m, X.p + s0 * n * NFEAT, X16.p + s0 * n * KPAD, std::min(ech, nsamples - s0));
    X.release();
    T.upload(targets, (size_t)nsamples * n, st);
    const int64_t B = std::min(batch, nsamples);
    ensure_cap(*m, B * n);
    std::vector<int64_t> order((size_t)nsamples);
    for (int64_t k = 0; k < nsamples; k++) order[k] = k;
    std::mt19937_64 rng(1234567u + (uint64_t)m->adam_t);
    double last = 0.0;
    for (int64_t ep = 0; ep < epochs; ep++) {
      std::shuffle(order.begin(), order.end(), rng);
      double acc = 0.0;
      int64_t nbat = 0;
      for (int64_t b0 = 0; b0 + B <= nsamples; b0 += B) {
        for (int64_t q = 0; q < B; q++) {
          const int64_t sidx = order[b0 + q];
          VFVM_HIP_CHECK(hipMemcpyAsync(m->x16.p + q * n * KPAD, X16.p + sidx * n * KPAD, sizeof(float) * n * KPAD,
                                        hipMemcpyDeviceToDevice, st));
          VFVM_HIP_CHECK(hipMemcpyAsync(m->target.p + q * n, T.p + sidx * n, sizeof(float) * n,
                                        hipMemcpyDeviceToDevice, st));
        }
        forward(*m, B * n);
        acc += backward(*m, B * n);
        nbat++;
        m->adam_t++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - std::pow(b1, (float)m->adam_t), c2 = 1.f - std::pow(b2, (float)m->adam_t);
        hipLaunchKernelGGL(k_adam, dim3(nb(m->np, 256)), dim3(256), 0, st, m->np, m->theta.p, (const float *)m->grad.p,
                           m->adam_m.p, m->adam_v.p, lr, b1, b2, 1e-8f, c1, c2);
        refresh_bf16(*m);
      }
      last = nbat ? acc / nbat : 0.0;
    }
    VFVM_HIP_CHECK(hipStreamSynchronize(st));
    if (final_loss) *final_loss = (float)last;
    return VFVM_OK;
  });
}

}  // extern "C"
