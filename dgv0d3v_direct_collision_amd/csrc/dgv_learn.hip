// dgv_learn.hip -- learned surrogate of the collision operator Q(f).
//
// An MLP maps a VDF (reference node order, scaled by 1/f_scale) to Q(f)/q_scale:
//   h_0 = x,  z_l = h_l W_l^T + b_l,  h_{l+1} = GELU(z_l)  (l < L-1),  y = z_{L-1}.
// Weights and activations are BF16 on the matrix cores (v_mfma_f32_16x16x32_bf16,
// FP32 accumulation); master weights, Adam moments, biases and pre-activations
// are FP32.  The output is scaled back to FP64 and projected onto the
// complement of the collision invariants psi = 1, u, v, w, |u|^2 in the
// w-weighted inner product, so the surrogate's Q conserves density, momentum
// and energy to FP64 rounding.  The direct evaluator is the surrogate's judge:
// on a set of probe cells the batched FP64 engine gives each row's residual,
// and rows whose residual exceeds the tolerance receive the direct Q.
//
// Every matrix product has the form C[m][n] = sum_k A[m][k] B[n][k] with both
// operands K-contiguous, so one kernel serves all of them:
//   forward       z  = h  . Wf^T     A = h   [B][in],   B = Wf [out][in]
//   input grad    dh = dz . Wb^T     A = dz  [B][out],  B = Wb [in][out]
//   weight grad   dW = dz^T . h      A = dzT [out][B],  B = hT [in][B]
// The epilogues write each activation in both orientations (h and hT, dz and
// dzT) and the Adam kernel writes both weight orientations (Wf and Wb).
// Widths are padded to multiples of 128 with zero weights, which stay zero.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "dgv_internal.h"

namespace dgv {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// GELU with the exact normal CDF and its derivative
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// ---------------------------------------------------------------------------------
// C[s][m][n] = sum_{k in chunk s} A[m][k] B[n][k].  Block tile GT x GT, k step 64, four
// waves each owning a quadrant of 16 x 16 MFMA tiles.  A training step's products
// are small (256 x 1024 x 3456 and the like), so what bounds them is the latency of
// a K step's loads over a handful of steps on a part of the chip: the K steps go
// straight to LDS, GT_RING - 1 of them in flight, and small products take tiles of
// 64 (four times the workgroups).  The tile does not enter the order of an element's
// sum.  Rows are 128 bytes of LDS; the 16-byte piece c of row r lies at c ^ (r % 8), so that
// the sixteen rows of a matrix operand read different banks.
// Requirements (checked by the host): M, N multiples of GT_PAD, K and kchunk
// multiples of 64, lda and ldb multiples of 8.
constexpr int GT_PAD = 128, GT_K = 64, kGradRing = 3;

template <int GT>
constexpr int gt_tiles() { return GT / 32; }   // MFMA tiles of a wave in each direction

// One workgroup's tile at (m0, n0) over nst K steps from kb0, in acc; sm holds GT_RING steps
template <int GT, int GT_RING>
__device__ __forceinline__ void gemm_tile(int m0, int n0, int kb0, int nst, const uint16_t* __restrict__ A, int64_t lda,
                                          const uint16_t* __restrict__ B, int64_t ldb, uint16_t (*sm)[2 * GT * GT_K],
                                          f4_t (&acc)[gt_tiles<GT>()][gt_tiles<GT>()]) {
  constexpr int kWaveLoads = GT / 16;   // a wave's loads per K step: 8 rows each of the 2 GT rows of A and B
  constexpr int TI = gt_tiles<GT>();
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 1) * (GT / 2), wn = (wave & 1) * (GT / 2);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TI; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
  // waves 0, 1 load the rows of A, waves 2, 3 those of B; lane l the piece of row l / 8
  // that belongs at position l % 8
  const int row0 = 8 * kWaveLoads * (wave & 1) + (lane >> 3), piece = (lane & 7) ^ (lane >> 3);
  const uint16_t* src = (wave < 2 ? A + (int64_t)(m0 + row0) * lda : B + (int64_t)(n0 + row0) * ldb) + kb0 + 8 * piece;
  const int64_t step8 = 8 * (wave < 2 ? lda : ldb);
  const uint32_t base = lds_addr(&sm[0][0]) + (uint32_t)wave * kWaveLoads * 8 * GT_K * 2;
  auto issue = [&](int st) {
    const uint32_t d = base + (uint32_t)(st % GT_RING) * (2 * GT * GT_K * 2);
#pragma unroll
    for (int j = 0; j < kWaveLoads; ++j) lds_load16(src + j * step8 + (int64_t)st * GT_K, d + j * 1024);
  };
  for (int st = 0; st < GT_RING - 1 && st < nst; ++st) issue(st);
  for (int st = 0; st < nst; ++st) {
    // the step has landed (only later steps are still in flight), and the LDS reads of the
    // step before are done in every wave: its buffer is free for the step GT_RING - 1 ahead
    const int later = min(nst - 1 - st, GT_RING - 2);
    if (later >= 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * kWaveLoads) : "memory");
    else if (later == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kWaveLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (st + GT_RING - 1 < nst) issue(st + GT_RING - 1);
    const uint16_t* sA = sm[st % GT_RING];
    const uint16_t* sB = sA + GT * GT_K;
#pragma unroll
    for (int kk = 0; kk < GT_K; kk += 32) {
      bf16x8_t af[TI], bv[TI];
      const int ko = ((kk / 8 + (lane >> 4)) ^ (lane & 7)) * 8;
#pragma unroll
      for (int t = 0; t < TI; ++t) {
        af[t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(sA + (wm + 16 * t + (lane & 15)) * GT_K + ko));
        bv[t] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(sB + (wn + 16 * t + (lane & 15)) * GT_K + ko));
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bv[j], acc[i][j], 0, 0, 0);
    }
  }
  static_assert(GT_RING == 3 || GT_RING == 4, "the waits count up to two later steps");
}

template <int GT, int GT_RING>
__global__ __launch_bounds__(256) void k_gemm_nt(int M, int N, int K, int kchunk, const uint16_t* __restrict__ A,
                                                 int64_t lda, const uint16_t* __restrict__ B, int64_t ldb,
                                                 float* __restrict__ C) {
  constexpr int TI = gt_tiles<GT>();
  __shared__ __attribute__((aligned(16))) uint16_t sm[GT_RING][2 * GT * GT_K];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * GT, m0 = blockIdx.y * GT;
  const int kb0 = blockIdx.z * kchunk;
  const int wm = (wave >> 1) * (GT / 2), wn = (wave & 1) * (GT / 2);
  f4_t acc[TI][TI];
  gemm_tile<GT, GT_RING>(m0, n0, kb0, (min(K, kb0 + kchunk) - kb0) / GT_K, A, lda, B, ldb, sm, acc);
  // output layout of the 16 x 16 FP32 tile: lane holds rows 4 (lane / 16) + e of column lane % 16
  float* Cs = C + (int64_t)blockIdx.z * M * N;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TI; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + e;
        const int n = n0 + wn + 16 * j + (lane & 15);
        Cs[(int64_t)m * N + n] = acc[i][j][e];
      }
}

// ---------------------------------------------------------------------------------
// Epilogues over tiles of 64 rows x 16 columns of an M x N result, 256 threads:
// thread (c, rg) handles column n0 + c of rows m0 + rg + 16 i.  The partial sums of a
// thread's four rows are in flight together, and the tile is narrow because the
// results are small (256 x 1024: 256 workgroups): what bounds the kernel is the latency
// of its loads.  Transposed copies and column sums go through LDS.  Column sums run
// over the rows g, g + 4, ... in order for g = 0 .. 3, then over g.
// (Tiles of 64 x 64 with one row's loads at a time took 15-27 us for 256 x 1024 and
// 256 x 3456 results, and the loss was a pass of its own, 9 us.)
enum { EPI_GELU = 0, EPI_BWD_GELU = 1, EPI_LOSS = 2, EPI_OUT = 3 };

struct EpiArgs {
  const float* part;   // [S][M][N] partial sums
  int S, M, N;
  const float* bias;   // [N] (forward)
  const float* zin;    // [M][N] pre-activation (backward)
  float* zout;         // [M][N] pre-activation (GELU)
  uint16_t* h;         // [M][N] BF16: GELU(z) or dz
  uint16_t* ht;        // [N][M] BF16 transposed copy
  float* dbpart;       // [M / 64][N] column sums of dz (backward, loss)
  // rows of the caller, [mvalid][ld] doubles, nvalid columns: the target Q (LOSS,
  // t = (float)(q scale), dz = gscale (y - t)) or the output (OUT, q = scale y)
  double* q;
  int64_t ld;
  int mvalid, nvalid;
  double scale;
  float gscale;
  double* losspart;    // LOSS: the tile's sum of squared differences
};

// Column tile of a workgroup: workgroups go to the eight XCDs in turn, so each XCD takes a
// run of neighbouring tiles (gridDim.x is a multiple of 8), whose halves of a 128-byte line meet in its L2
__device__ __forceinline__ int xcd_column() { return (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8); }

template <int MODE>
__global__ __launch_bounds__(256) void k_epilogue(EpiArgs a) {
  constexpr bool DZ = MODE == EPI_BWD_GELU || MODE == EPI_LOSS;
  __shared__ alignas(8) uint16_t tile[16][68];   // [column][row]; 136-byte rows keep 8-byte reads aligned
  __shared__ float dzs[DZ ? 64 : 1][17];
  __shared__ float cs[4][16];
  __shared__ double red[MODE == EPI_LOSS ? 256 : 1];
  const int n0 = xcd_column() * 16, m0 = blockIdx.y * 64;
  const int c = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int64_t MN = (int64_t)a.M * a.N;
  int64_t idx[4];
  float other[4];   // the rows' pre-activations or targets, loaded beside the partial sums
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + rg + 16 * i, n = n0 + c;
    idx[i] = (int64_t)m * a.N + n;
    other[i] = 0.f;
    if constexpr (MODE == EPI_BWD_GELU) other[i] = a.zin[idx[i]];
    if constexpr (MODE == EPI_LOSS)
      if (m < a.mvalid && n < a.nvalid) other[i] = (float)(a.q[(int64_t)m * a.ld + n] * a.scale);
  }
  // partials in a fixed order: four running sums (k mod 4), then ((0 + 1) + (2 + 3))
  float q[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) q[i][j] = 0.f;
  int k = 0;
  for (; k + 4 <= a.S; k += 4)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) q[i][j] += a.part[(int64_t)(k + j) * MN + idx[i]];
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (k + j < a.S) {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i][j] += a.part[(int64_t)(k + j) * MN + idx[i]];
    }
  const float bias = DZ && MODE != EPI_LOSS ? 0.f : a.bias[n0 + c];
  double sq = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = rg + 16 * i, m = m0 + r, n = n0 + c;
    const float s = (q[i][0] + q[i][1]) + (q[i][2] + q[i][3]);
    if constexpr (MODE == EPI_GELU) {
      const float z = s + bias;
      a.zout[idx[i]] = z;
      const uint16_t hb = f2bf(gelu(z));
      a.h[idx[i]] = hb;
      tile[c][r] = hb;
    } else if constexpr (MODE == EPI_OUT) {
      const float y = s + bias;
      if (m < a.mvalid && n < a.nvalid) a.q[(int64_t)m * a.ld + n] = a.scale * (double)y;
    } else {
      float dz;
      if constexpr (MODE == EPI_LOSS) {
        const float y = s + bias;
        const float d = (m < a.mvalid && n < a.nvalid) ? y - other[i] : 0.f;
        sq += (double)d * (double)d;
        dz = a.gscale * d;
      } else {
        dz = s * gelu_d(other[i]);
      }
      const uint16_t hb = f2bf(dz);
      a.h[idx[i]] = hb;
      tile[c][r] = hb;
      dzs[r][c] = dz;
    }
  }
  if constexpr (MODE == EPI_OUT) return;
  if constexpr (MODE == EPI_LOSS) red[threadIdx.x] = sq;
  __syncthreads();
  *reinterpret_cast<uint2*>(a.ht + (int64_t)(n0 + rg) * a.M + m0 + 4 * c) = *reinterpret_cast<const uint2*>(&tile[rg][4 * c]);
  if constexpr (DZ) {
    if (rg < 4) {
      float colsum = dzs[rg][c];
      for (int i = 1; i < 16; ++i) colsum += dzs[rg + 4 * i][c];
      cs[rg][c] = colsum;
    }
    __syncthreads();
    if (rg == 0) a.dbpart[(int64_t)blockIdx.y * a.N + n0 + c] = ((cs[0][c] + cs[1][c]) + cs[2][c]) + cs[3][c];
  }
  if constexpr (MODE == EPI_LOSS) {
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) a.losspart[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = red[0];
  }
}

// out[0] = sum of part[0..n) in a fixed order, times scale, by one workgroup of 256
__device__ __forceinline__ void sum_fixed(const double* __restrict__ part, int n, double scale, double* red, double* out) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0] * scale;
}

struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;  // c1 = 1 / (1 - b1^t), c2 = 1 / (1 - b2^t)
};

// The moments' products are contracted explicitly, weights and biases each their way, so
// that a step's bits do not depend on what the compiler fuses around them.
template <bool BIAS = false>
__device__ __forceinline__ float adam_update(float g, float& w, float& m, float& v, const AdamArgs& h) {
  m = BIAS ? fmaf(h.b1, m, (1.f - h.b1) * g) : fmaf(1.f - h.b1, g, h.b1 * m);
  v = BIAS ? fmaf(h.b2, v, (1.f - h.b2) * g * g) : fmaf((1.f - h.b2) * g, g, h.b2 * v);
  w = w - h.lr * (m * h.c1) / (sqrtf(v * h.c2) + h.eps);
  return w;
}

constexpr int kGradPitch = 68;   // floats per row of a gradient tile in LDS: 16-byte reads aligned, banks spread

// Adam on a 64 x 64 tile of a weight matrix [O][I], its gradient in LDS (and written
// to G): the master weights, the moments and the BF16 copies Wf [O][I] and
// Wb [I][O].  A thread owns four consecutive columns of four rows: 16-byte
// loads and stores, and all twelve loads in flight before the first update.
// tile: [column][row] of the tile's BF16 weights; rows of 68 halves (136 bytes)
// keep the 8-byte reads of the transposed write aligned.
__device__ __forceinline__ void adam_tile(int i0, int o0, int O, int I, const float* sg, float* __restrict__ G,
                                          float* __restrict__ W, float* __restrict__ m, float* __restrict__ v,
                                          uint16_t* __restrict__ Wf, uint16_t* __restrict__ Wb, const AdamArgs& h,
                                          uint16_t (*tile)[68]) {
  const int c4 = threadIdx.x & 15, rg = threadIdx.x >> 4;   // columns 4 c4 .. 4 c4 + 3, rows rg + 16 k
  float4 g[4], w[4], mm[4], vv[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int64_t idx = (int64_t)(o0 + rg + 16 * k) * I + i0 + 4 * c4;
    w[k] = *reinterpret_cast<const float4*>(W + idx);
    mm[k] = *reinterpret_cast<const float4*>(m + idx);
    vv[k] = *reinterpret_cast<const float4*>(v + idx);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = rg + 16 * k;
    const int64_t idx = (int64_t)(o0 + r) * I + i0 + 4 * c4;
    g[k] = *reinterpret_cast<const float4*>(sg + r * kGradPitch + 4 * c4);
    *reinterpret_cast<float4*>(G + idx) = g[k];
    adam_update(g[k].x, w[k].x, mm[k].x, vv[k].x, h);
    adam_update(g[k].y, w[k].y, mm[k].y, vv[k].y, h);
    adam_update(g[k].z, w[k].z, mm[k].z, vv[k].z, h);
    adam_update(g[k].w, w[k].w, mm[k].w, vv[k].w, h);
    *reinterpret_cast<float4*>(W + idx) = w[k];
    *reinterpret_cast<float4*>(m + idx) = mm[k];
    *reinterpret_cast<float4*>(v + idx) = vv[k];
    const uint16_t b0 = f2bf(w[k].x), b1 = f2bf(w[k].y), b2 = f2bf(w[k].z), b3 = f2bf(w[k].w);
    *reinterpret_cast<uint2*>(Wf + idx) = make_uint2((uint32_t)b0 | ((uint32_t)b1 << 16), (uint32_t)b2 | ((uint32_t)b3 << 16));
    tile[4 * c4 + 0][r] = b0;
    tile[4 * c4 + 1][r] = b1;
    tile[4 * c4 + 2][r] = b2;
    tile[4 * c4 + 3][r] = b3;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int ii = rg + 16 * k;   // column i0 + ii: rows o0 + 4 c4 .. o0 + 4 c4 + 3
    *reinterpret_cast<uint2*>(Wb + (int64_t)(i0 + ii) * O + o0 + 4 * c4) =
        *reinterpret_cast<const uint2*>(&tile[ii][4 * c4]);
  }
}

// A layer's gradient and update, one launch: the workgroups [0, ntile) take 64 x 64
// tiles of the weights -- the gradient dW = dz^T h over the batch on the matrix cores,
// kept in G, then Adam -- the next (O + 255) / 256 the bias -- its gradient, the
// column sums dbpart[t][O] over t in order, then Adam -- and, with losspart, one more
// adds the loss.  update = 0: gradients only.  Bound by the weights' 32 bytes (weights
// and moments read and written, gradient and BF16 copies written; 3456 x 1024: 113 MB).
// (As separate launches the product and Adam took 8 + 18 us at 3456 x 1024 and a gap,
// the bias sums, bias updates and loss sum 3-4 us each and their gaps, seven times a step
// of a network with two hidden layers.)
struct BiasArgs {
  const float* dbpart;
  int T;
  float *g, *w, *m, *v;
  const double* losspart;
  int nloss;
  double loss_scale;
  double* loss;
};

__global__ __launch_bounds__(256) void k_grad_update(int O, int I, int K, const uint16_t* __restrict__ dZt,
                                                     const uint16_t* __restrict__ Ht, float* __restrict__ G,
                                                     float* __restrict__ W, float* __restrict__ m,
                                                     float* __restrict__ v, uint16_t* __restrict__ Wf,
                                                     uint16_t* __restrict__ Wb, int update, AdamArgs h, BiasArgs a) {
  constexpr int GT = 64, TI = gt_tiles<GT>();
  __shared__ __attribute__((aligned(16))) uint16_t sm[kGradRing][2 * GT * GT_K];
  static_assert(sizeof(sm) >= 64 * kGradPitch * sizeof(float) + 64 * 68 * sizeof(uint16_t), "the gradient and weight tiles take the K steps' place");
  const int ntile = (O / GT) * (I / GT), nb = (O + 255) / 256;
  const int t = blockIdx.x;
  if (t < ntile) {
    const int i0 = t % (I / GT) * GT, o0 = t / (I / GT) * GT;
    f4_t acc[TI][TI];
    gemm_tile<GT, kGradRing>(o0, i0, 0, K / GT_K, dZt, K, Ht, K, sm, acc);
    __syncthreads();   // every wave is done with the K steps
    float* sg = reinterpret_cast<float*>(&sm[0][0]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * (GT / 2), wn = (wave & 1) * (GT / 2);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TI; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) sg[(wm + 16 * i + 4 * (lane >> 4) + e) * kGradPitch + wn + 16 * j + (lane & 15)] = acc[i][j][e];
    __syncthreads();
    if (update) {
      adam_tile(i0, o0, O, I, sg, G, W, m, v, Wf, Wb, h, reinterpret_cast<uint16_t(*)[68]>(sg + 64 * kGradPitch));
    } else {
      const int c4 = threadIdx.x & 15, rg = threadIdx.x >> 4;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *reinterpret_cast<float4*>(G + (int64_t)(o0 + rg + 16 * k) * I + i0 + 4 * c4) =
            *reinterpret_cast<const float4*>(sg + (rg + 16 * k) * kGradPitch + 4 * c4);
    }
    return;
  }
  if (t < ntile + nb) {
    const int n = (t - ntile) * 256 + threadIdx.x;
    if (n >= O) return;
    float s = 0.f;
    for (int k = 0; k < a.T; ++k) s += a.dbpart[(int64_t)k * O + n];
    a.g[n] = s;
    if (update) {
      float ww = a.w[n], mm = a.m[n], vv = a.v[n];
      adam_update<true>(s, ww, mm, vv, h);
      a.w[n] = ww;
      a.m[n] = mm;
      a.v[n] = vv;
    }
    return;
  }
  sum_fixed(a.losspart, a.nloss, a.loss_scale, reinterpret_cast<double*>(&sm[0][0]), a.loss);
}

// BF16 copies of master weights [O][I]: Wf [O][I] and Wb [I][O]
__global__ __launch_bounds__(256) void k_weights_bf16(int O, int I, const float* __restrict__ W,
                                                      uint16_t* __restrict__ Wf, uint16_t* __restrict__ Wb) {
  __shared__ uint16_t tile[64][66];
  const int i0 = blockIdx.x * 64, o0 = blockIdx.y * 64;
  const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
  for (int k = 0; k < 16; ++k) {
    const int r = rg + 4 * k;
    const int64_t idx = (int64_t)(o0 + r) * I + i0 + c;
    const uint16_t hb = f2bf(W[idx]);
    Wf[idx] = hb;
    tile[c][r] = hb;
  }
  __syncthreads();
  for (int k = 0; k < 16; ++k) {
    const int rr = rg + 4 * k;
    Wb[(int64_t)(i0 + rr) * O + o0 + c] = tile[rr][c];
  }
}

// Rows of f (FP64, [nrows][ld]) -> x = f / f_scale as BF16 [Mp][Kp] and [Kp][Mp],
// zero outside nrows x N.  Tiles of 64 rows x 16 columns, as the epilogues.
__global__ __launch_bounds__(256) void k_rows_in(const double* __restrict__ F, int64_t ld, int nrows, int N,
                                                 double inv_scale, int Mp, int Kp, uint16_t* __restrict__ X,
                                                 uint16_t* __restrict__ Xt) {
  __shared__ alignas(8) uint16_t tile[16][68];
  const int k0 = xcd_column() * 16, m0 = blockIdx.y * 64;
  const int c = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int k = k0 + c;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = rg + 16 * i, m = m0 + r;
    const float x = (m < nrows && k < N) ? (float)(F[(int64_t)m * ld + k] * inv_scale) : 0.f;
    const uint16_t hb = f2bf(x);
    X[(int64_t)m * Kp + k] = hb;
    tile[c][r] = hb;
  }
  __syncthreads();
  *reinterpret_cast<uint2*>(Xt + (int64_t)(k0 + rg) * Mp + m0 + 4 * c) = *reinterpret_cast<const uint2*>(&tile[rg][4 * c]);
}

// The valid [nrows][n] part of a padded matrix, dense
__global__ void k_rows_dense(const float* __restrict__ P, int64_t pitch, int64_t n, int64_t total, float* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = P[i / n * pitch + i % n];
}

// One block per row: D[m][n] = F[m][n] - fm[n] (D dense, N per row) and
// rs[m] = sqrt(mean_n D[m][n]^2), summed in a fixed order.
__global__ __launch_bounds__(256) void k_rows_minus(const double* __restrict__ F, int64_t ld, int N,
                                                    const double* __restrict__ fm, double* __restrict__ D,
                                                    double* __restrict__ rs) {
  __shared__ double red[256];
  const int m = blockIdx.x;
  double acc = 0.0;
  for (int k = threadIdx.x; k < N; k += 256) {
    const double x = F[(int64_t)m * ld + k] - fm[k];
    D[(int64_t)m * N + k] = x;
    acc = fma(x, x, acc);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) rs[m] = sqrt(red[0] / N);
}

// D[m][n] /= rs[m] (zero rows stay zero)
__global__ void k_rows_unit(double* __restrict__ D, int nrows, int N, const double* __restrict__ rs) {
  const int64_t n = (int64_t)nrows * N, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const double r = rs[i / N];
    D[i] = r > 0.0 ? D[i] / r : 0.0;
  }
}

// Q[m][n] = rs[m]^2 Q[m][n] + Lq[m][n] + qfm[n] (Lq dense, N per row)
__global__ void k_rows_combine(double* __restrict__ Q, int64_t ld, int nrows, int N, const double* __restrict__ rs,
                               const double* __restrict__ Lq, const double* __restrict__ qfm) {
  const int64_t n = (int64_t)nrows * N, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const int64_t m = i / N, k = i - m * N;
    const double r = rs[m];
    Q[m * ld + k] = fma(r * r, Q[m * ld + k], Lq[i] + qfm[k]);
  }
}

struct Chol5 {
  double L[25];
};

// FP64 projection of each row onto the complement of psi = 1,u,v,w,|u|^2 in the
// w-weighted inner product: q -= sum_k lam_k psi_k with G lam = (sum_i w_i psi_k q_i).
// One block per row; moments summed in a fixed order.
__global__ __launch_bounds__(256) void k_project_rows(double* __restrict__ q, int64_t ld, int N,
                                                      const double* __restrict__ u, const double* __restrict__ v,
                                                      const double* __restrict__ w, const double* __restrict__ gw,
                                                      Chol5 C) {
  __shared__ double red[5][256];
  __shared__ double lam[5];
  double* row = q + (int64_t)blockIdx.x * ld;
  double s[5] = {0, 0, 0, 0, 0};
  for (int i = threadIdx.x; i < N; i += 256) {
    const double x = gw[i] * row[i];
    const double uu = u[i], vv = v[i], ww = w[i];
    s[0] += x;
    s[1] += x * uu;
    s[2] += x * vv;
    s[3] += x * ww;
    s[4] += x * (uu * uu + vv * vv + ww * ww);
  }
  for (int k = 0; k < 5; ++k) red[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st)
      for (int k = 0; k < 5; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double y[5], x[5];
    for (int i = 0; i < 5; ++i) {
      double a = red[i][0];
      for (int k = 0; k < i; ++k) a -= C.L[i * 5 + k] * y[k];
      y[i] = a / C.L[i * 5 + i];
    }
    for (int i = 4; i >= 0; --i) {
      double a = y[i];
      for (int k = i + 1; k < 5; ++k) a -= C.L[k * 5 + i] * x[k];
      x[i] = a / C.L[i * 5 + i];
    }
    for (int k = 0; k < 5; ++k) lam[k] = x[k];
  }
  __syncthreads();
  const double l0 = lam[0], l1 = lam[1], l2 = lam[2], l3 = lam[3], l4 = lam[4];
  for (int i = threadIdx.x; i < N; i += 256) {
    const double uu = u[i], vv = v[i], ww = w[i];
    row[i] = row[i] - (l0 + l1 * uu + l2 * vv + l3 * ww + l4 * (uu * uu + vv * vv + ww * ww));
  }
}

// rows [nrows][ld] -> packed batch layout P[node * stride + r] (64 x 64 tiles)
__global__ __launch_bounds__(256) void k_rows_to_packed(const double* __restrict__ F, int64_t ld, int nrows, int N,
                                                        double* __restrict__ P, int64_t stride) {
  __shared__ double tile[64][65];
  const int n0 = blockIdx.x * 64, m0 = blockIdx.y * 64;
  const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
  for (int i = 0; i < 16; ++i) {
    const int r = rg + 4 * i;
    const int m = m0 + r, n = n0 + c;
    tile[c][r] = (m < nrows && n < N) ? F[(int64_t)m * ld + n] : 0.0;
  }
  __syncthreads();
  for (int i = 0; i < 16; ++i) {
    const int rr = rg + 4 * i;
    const int n = n0 + rr, m = m0 + c;
    if (n < N && m < nrows) P[(int64_t)n * stride + m] = tile[rr][c];
  }
}

// Residual of each row over the probe nodes: ||q_sur - q_dir|| / ||q_dir||,
// q_dir in the packed layout.  One block per row, fixed-order sums.
__global__ __launch_bounds__(256) void k_probe_residual(const double* __restrict__ q, int64_t ld,
                                                        const double* __restrict__ P, int64_t stride,
                                                        const int32_t* __restrict__ nodes, int nn,
                                                        double* __restrict__ res) {
  __shared__ double r0[256], r1[256];
  const int m = blockIdx.x;
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < nn; i += 256) {
    const int64_t node = nodes[i];
    const double d = P[node * stride + m];
    const double e = q[(int64_t)m * ld + node] - d;
    a += e * e;
    b += d * d;
  }
  r0[threadIdx.x] = a;
  r1[threadIdx.x] = b;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) {
      r0[threadIdx.x] += r0[threadIdx.x + st];
      r1[threadIdx.x] += r1[threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) res[m] = r1[0] > 0.0 ? sqrt(r0[0] / r1[0]) : (r0[0] > 0.0 ? INFINITY : 0.0);
}

}  // namespace dgv

// ===================================================================================
// host side

namespace {

using namespace dgv;

int round_up(int x, int m) { return ((x + m - 1) / m) * m; }

struct SurLayer {
  int in = 0, out = 0, inp = 0, outp = 0;
  float *W = nullptr, *mW = nullptr, *vW = nullptr, *G = nullptr;      // [outp][inp] FP32
  float *b = nullptr, *mb = nullptr, *vb = nullptr, *gb = nullptr;     // [outp]
  uint16_t *Wf = nullptr, *Wb = nullptr;                               // BF16 [outp][inp], [inp][outp]
};

struct Gemm {
  int M, N, K, S, kchunk;
};

// Split-K: about 512 workgroups, but at least 8 K steps per workgroup, so that
// the FP32 partials (S x M x N, summed by the epilogue) stay a small multiple of
// the output.
Gemm plan_gemm(int M, int N, int K) {
  Gemm g{M, N, K, 1, K};
  const int tiles = (M / GT_PAD) * (N / GT_PAD);
  const int kt = K / GT_K;
  const int S = std::max(1, std::min(kt / 8, (512 + tiles - 1) / tiles));
  g.kchunk = ((kt + S - 1) / S) * GT_K;
  g.S = (K + g.kchunk - 1) / g.kchunk;
  return g;
}

}  // namespace

struct dgv_surrogate {
  dgv_ctx* ctx = nullptr;
  int device = 0;
  int L = 0, batch = 0, Bp = 0;
  std::vector<SurLayer> layers;
  std::vector<uint16_t*> H, Ht;  // H[l]: input of layer l, BF16 [Bp][inp_l] and [inp_l][Bp]
  std::vector<float*> Z;         // Z[l], l < L-1: pre-activation [Bp][outp_l]
  uint16_t* dZ[2] = {nullptr, nullptr};
  uint16_t* dZt[2] = {nullptr, nullptr};
  float* part = nullptr;
  int64_t part_elems = 0;
  float* dbpart[2] = {nullptr, nullptr};   // column sums of dz, of the layer and of the one before it
  double* losspart = nullptr;
  double* h_loss = nullptr;                // pinned: the kernel that adds the loss writes it there
  int64_t step = 0;
  double f_scale = 1.0, q_scale = 1.0;
  Chol5 chol{};
  // judge / fallback
  dgv_batch* judge = nullptr;
  int32_t* d_probe_nodes = nullptr;
  int nprobe_nodes = 0;
  double* d_res = nullptr;
  std::vector<int32_t> probe_cells;
  // decomposition mode: Q(f) = Q(fm) + L(Df) + Q(Df) with Df = f - fm and L the
  // context's linearised operator at fm; the network gives Q(Df) / s^2 from
  // Df / s, s the root mean square of the row's Df (Q(Df) is quadratic in Df)
  int decomp = 0;
  int64_t decomp_gen = 0;        // the linearised operator's build count at set time
  double* d_df = nullptr;        // batch x N: Df rows of a chunk, then Df / s
  double* d_lin = nullptr;       // batch x N: L(Df) rows
  double* d_qfm = nullptr;       // N: Q(fm)
  double* d_rs = nullptr;        // batch: s per row
};

namespace {

int serr(dgv_surrogate* s, int code, const std::string& m) {
  return set_error(s ? s->ctx : nullptr, code, m);
}
#define SHIP(s, call)                                                                                    \
  do {                                                                                                   \
    hipError_t e_ = (call);                                                                              \
    if (e_ != hipSuccess) return serr((s), DGV_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int64_t kSmallTiles = 512;

int launch_gemm(dgv_surrogate* s, const Gemm& g, const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb,
                float* C) {
  if (g.M % GT_PAD || g.N % GT_PAD || g.K % GT_K || g.kchunk % GT_K || lda % 8 || ldb % 8 || lda < g.K || ldb < g.K)
    return serr(s, DGV_ERR_ARG, "matrix product shape does not fit the tiling");
  // tiles of 64 while they fit two to a CU at once, else the 128 that read half as much
  // (forward pass of 64 rows, 729-300-300-729: 0.029 ms with 64, 0.038 with 128; 256 rows,
  // 3375-1024-1024-3375: 0.052 and 0.057; 1024 rows, 19683-2048-2048-19683: 0.643 and 0.530.
  // With tiles of 128, one K step in flight and the older epilogues: 0.071, 0.108, 0.576)
  const int64_t n64 = (int64_t)(g.N / 64) * (g.M / 64) * g.S;
  if (n64 <= kSmallTiles)
    hipLaunchKernelGGL((k_gemm_nt<64, 4>), dim3(g.N / 64, g.M / 64, g.S), dim3(256), 0, s->ctx->stream, g.M, g.N, g.K,
                       g.kchunk, A, lda, B, ldb, C);
  else
    hipLaunchKernelGGL((k_gemm_nt<128, 4>), dim3(g.N / 128, g.M / 128, g.S), dim3(256), 0, s->ctx->stream, g.M, g.N,
                       g.K, g.kchunk, A, lda, B, ldb, C);
  return DGV_OK;
}

// the network on the loaded rows; the last layer's epilogue is out's (LOSS or OUT)
int forward(dgv_surrogate* s, EpiArgs out, int out_mode) {
  hipStream_t st = s->ctx->stream;
  for (int l = 0; l < s->L; ++l) {
    const SurLayer& ly = s->layers[l];
    const Gemm g = plan_gemm(s->Bp, ly.outp, ly.inp);
    int rc = launch_gemm(s, g, s->H[l], ly.inp, ly.Wf, ly.inp, s->part);
    if (rc) return rc;
    EpiArgs a = l + 1 < s->L ? EpiArgs{} : out;
    a.part = s->part;
    a.S = g.S;
    a.M = s->Bp;
    a.N = ly.outp;
    a.bias = ly.b;
    const dim3 grid(ly.outp / 16, s->Bp / 64);
    if (l + 1 < s->L) {
      a.zout = s->Z[l];
      a.h = s->H[l + 1];
      a.ht = s->Ht[l + 1];
      hipLaunchKernelGGL(k_epilogue<EPI_GELU>, grid, dim3(256), 0, st, a);
    } else if (out_mode == EPI_LOSS) {
      hipLaunchKernelGGL(k_epilogue<EPI_LOSS>, grid, dim3(256), 0, st, a);
    } else {
      hipLaunchKernelGGL(k_epilogue<EPI_OUT>, grid, dim3(256), 0, st, a);
    }
  }
  SHIP(s, hipGetLastError());
  return DGV_OK;
}

int load_rows(dgv_surrogate* s, const double* d_f, int64_t ld, int nrows) {
  const SurLayer& l0 = s->layers[0];
  hipLaunchKernelGGL(k_rows_in, dim3(l0.inp / 16, s->Bp / 64), dim3(256), 0, s->ctx->stream, d_f, ld, nrows, l0.in,
                     1.0 / s->f_scale, s->Bp, l0.inp, s->H[0], s->Ht[0]);
  SHIP(s, hipGetLastError());
  return DGV_OK;
}

// The network's part of a prediction (no projection) or, with project, the
// prediction projected onto the complement of the collision invariants.
int predict_chunk(dgv_surrogate* s, const double* d_f, int64_t ld, int nrows, double* d_q, int project) {
  int rc = load_rows(s, d_f, ld, nrows);
  if (rc) return rc;
  EpiArgs a{};
  a.q = d_q;
  a.ld = ld;
  a.mvalid = nrows;
  a.nvalid = s->layers[s->L - 1].out;
  a.scale = s->q_scale;
  if ((rc = forward(s, a, EPI_OUT))) return rc;
  if (project) {
    const dgv_ctx* c = s->ctx;
    hipLaunchKernelGGL(k_project_rows, dim3(nrows), dim3(256), 0, c->stream, d_q, ld, (int)c->g.N, c->d_u, c->d_v,
                       c->d_w, c->d_gwts, s->chol);
  }
  SHIP(s, hipGetLastError());
  return DGV_OK;
}

// Decomposition mode: the linearised operator must be the one the mode was set
// with (PrepareFMA_DGV rebuilds it at a new Maxwellian, an A-array change drops it).
int decomp_check(dgv_surrogate* s) {
  if (!s->decomp) return DGV_OK;
  const LinearState& L = s->ctx->lin;
  if (!L.fma_valid || L.nprepare != s->decomp_gen)
    return serr(s, DGV_ERR_STATE, "the linearised operator changed since the decomposition mode was set");
  return DGV_OK;
}

// Q of nrows rows of f: the network's output, or in decomposition mode
// Q(fm) + L(Df) + s^2 net(Df / s); then the projection when asked for.
int predict_rows(dgv_surrogate* s, const double* d_f, int64_t ld, int nrows, double* d_q, int project) {
  if (!s->decomp) return predict_chunk(s, d_f, ld, nrows, d_q, project);
  if (nrows == 0) return DGV_OK;
  dgv_ctx* c = s->ctx;
  const int N = (int)c->g.N;
  const int64_t n = (int64_t)nrows * N;
  const unsigned nbk = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 1 << 20));
  hipLaunchKernelGGL(k_rows_minus, dim3(nrows), dim3(256), 0, c->stream, d_f, ld, N, c->lin.d_vec[0], s->d_df,
                     s->d_rs);
  SHIP(s, hipGetLastError());
  int rc = eval_linear_dev(c, s->d_df, N, s->d_lin, N, nrows);
  if (rc) return rc;
  hipLaunchKernelGGL(k_rows_unit, dim3(nbk), dim3(256), 0, c->stream, s->d_df, nrows, N, s->d_rs);
  SHIP(s, hipGetLastError());
  if ((rc = predict_chunk(s, s->d_df, N, nrows, d_q, 0))) return rc;
  hipLaunchKernelGGL(k_rows_combine, dim3(nbk), dim3(256), 0, c->stream, d_q, ld, nrows, N, s->d_rs, s->d_lin,
                     s->d_qfm);
  if (project)
    hipLaunchKernelGGL(k_project_rows, dim3(nrows), dim3(256), 0, c->stream, d_q, ld, N, c->d_u, c->d_v, c->d_w,
                       c->d_gwts, s->chol);
  SHIP(s, hipGetLastError());
  return DGV_OK;
}

void free_surrogate(dgv_surrogate* s) {
  for (SurLayer& l : s->layers) {
    for (float* p : {l.W, l.mW, l.vW, l.G, l.b, l.mb, l.vb, l.gb}) hipFree(p);
    hipFree(l.Wf);
    hipFree(l.Wb);
  }
  for (auto p : s->H) hipFree(p);
  for (auto p : s->Ht) hipFree(p);
  for (auto p : s->Z) hipFree(p);
  for (int i = 0; i < 2; ++i) { hipFree(s->dZ[i]); hipFree(s->dZt[i]); }
  hipFree(s->part); hipFree(s->dbpart[0]); hipFree(s->dbpart[1]); hipFree(s->losspart); hipHostFree(s->h_loss);
  hipFree(s->d_probe_nodes); hipFree(s->d_res);
  hipFree(s->d_df); hipFree(s->d_lin); hipFree(s->d_qfm); hipFree(s->d_rs);
  if (s->judge) dgv_batch_destroy(s->judge);
}

}  // namespace

extern "C" {

int dgv_sur_create(dgv_ctx* ctx, const int32_t* widths, int32_t nlayers, int32_t batch, uint64_t seed,
                   dgv_surrogate** out) {
  if (!ctx || !widths || !out || nlayers < 1 || batch < 1) { set_global_error("dgv_sur_create: bad argument"); return DGV_ERR_ARG; }
  *out = nullptr;
  if (widths[0] != ctx->g.N || widths[nlayers] != ctx->g.N)
    return set_error(ctx, DGV_ERR_ARG, "the first and last widths must equal the number of nodes");
  for (int l = 0; l <= nlayers; ++l)
    if (widths[l] < 1) return set_error(ctx, DGV_ERR_ARG, "widths must be positive");
  double L25[25];
  if (gram_cholesky(ctx->g, L25)) return set_error(ctx, DGV_ERR_GRID, "Gram matrix of the invariants is singular");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  dgv_surrogate* s = new dgv_surrogate();
  s->ctx = ctx;
  s->device = ctx->device;
  s->L = nlayers;
  s->batch = batch;
  s->Bp = round_up(batch, 128);
  std::memcpy(s->chol.L, L25, sizeof(L25));
  auto fail = [&](int code, const std::string& m) { free_surrogate(s); delete s; return set_error(ctx, code, m); };
  auto dalloc = [&](void** p, size_t bytes) { return hipMalloc(p, std::max<size_t>(bytes, 16)) == hipSuccess; };
  s->layers.resize(nlayers);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.f, 1.f);
  int maxw = 0;
  s->part_elems = 1;
  for (int l = 0; l < nlayers; ++l) {
    SurLayer& ly = s->layers[l];
    ly.in = widths[l];
    ly.out = widths[l + 1];
    ly.inp = round_up(ly.in, 128);
    ly.outp = round_up(ly.out, 128);
    maxw = std::max({maxw, ly.inp, ly.outp});
    const size_t nw = (size_t)ly.outp * ly.inp;
    bool ok = dalloc((void**)&ly.W, 4 * nw) && dalloc((void**)&ly.mW, 4 * nw) && dalloc((void**)&ly.vW, 4 * nw) &&
              dalloc((void**)&ly.G, 4 * nw) && dalloc((void**)&ly.b, 4 * ly.outp) &&
              dalloc((void**)&ly.mb, 4 * ly.outp) && dalloc((void**)&ly.vb, 4 * ly.outp) &&
              dalloc((void**)&ly.gb, 4 * ly.outp) && dalloc((void**)&ly.Wf, 2 * nw) && dalloc((void**)&ly.Wb, 2 * nw);
    if (!ok) return fail(DGV_ERR_NOMEM, "hipMalloc(surrogate weights) failed");
    // W ~ N(0, 1/fan_in), the last layer scaled by 0.1; padded entries zero
    std::vector<float> W(nw, 0.f);
    const float sd = (l + 1 == nlayers ? 0.1f : 1.0f) / std::sqrt((float)ly.in);
    for (int o = 0; o < ly.out; ++o)
      for (int i = 0; i < ly.in; ++i) W[(size_t)o * ly.inp + i] = sd * nd(rng);
    hipStream_t st = ctx->stream;   // everything in stream order: the context's stream ignores the null stream
    if (hipMemcpyAsync(ly.W, W.data(), 4 * nw, hipMemcpyHostToDevice, st) != hipSuccess ||
        hipMemsetAsync(ly.mW, 0, 4 * nw, st) || hipMemsetAsync(ly.vW, 0, 4 * nw, st) ||
        hipMemsetAsync(ly.G, 0, 4 * nw, st) || hipMemsetAsync(ly.b, 0, 4 * ly.outp, st) ||
        hipMemsetAsync(ly.mb, 0, 4 * ly.outp, st) || hipMemsetAsync(ly.vb, 0, 4 * ly.outp, st) ||
        hipMemsetAsync(ly.gb, 0, 4 * ly.outp, st) || hipStreamSynchronize(st))
      return fail(DGV_ERR_HIP, "surrogate initialisation failed");
    hipLaunchKernelGGL(k_weights_bf16, dim3(ly.inp / 64, ly.outp / 64), dim3(256), 0, ctx->stream, ly.outp, ly.inp,
                       ly.W, ly.Wf, ly.Wb);
    const Gemm f = plan_gemm(s->Bp, ly.outp, ly.inp);
    const Gemm d = plan_gemm(s->Bp, ly.inp, ly.outp);
    s->part_elems = std::max({s->part_elems, (int64_t)f.S * f.M * f.N, (int64_t)d.S * d.M * d.N});
  }
  s->H.assign(nlayers, nullptr);
  s->Ht.assign(nlayers, nullptr);
  s->Z.assign(std::max(nlayers - 1, 1), nullptr);
  for (int l = 0; l < nlayers; ++l) {
    const size_t n = (size_t)s->Bp * s->layers[l].inp;
    if (!dalloc((void**)&s->H[l], 2 * n) || !dalloc((void**)&s->Ht[l], 2 * n))
      return fail(DGV_ERR_NOMEM, "hipMalloc(activations) failed");
    if (l + 1 < nlayers && !dalloc((void**)&s->Z[l], 4 * (size_t)s->Bp * s->layers[l].outp))
      return fail(DGV_ERR_NOMEM, "hipMalloc(activations) failed");
  }
  const size_t nmax = (size_t)s->Bp * maxw;
  bool ok = dalloc((void**)&s->dZ[0], 2 * nmax) &&
            dalloc((void**)&s->dZ[1], 2 * nmax) && dalloc((void**)&s->dZt[0], 2 * nmax) &&
            dalloc((void**)&s->dZt[1], 2 * nmax) && dalloc((void**)&s->part, 4 * (size_t)s->part_elems) &&
            dalloc((void**)&s->dbpart[0], 4 * (size_t)(s->Bp / 64) * maxw) &&
            dalloc((void**)&s->dbpart[1], 4 * (size_t)(s->Bp / 64) * maxw) &&
            dalloc((void**)&s->losspart, 8 * (size_t)(s->Bp / 64) * (maxw / 16)) &&
            hipHostMalloc((void**)&s->h_loss, sizeof(double), 0) == hipSuccess &&
            dalloc((void**)&s->d_res, 8 * (size_t)s->Bp);
  if (!ok) return fail(DGV_ERR_NOMEM, "hipMalloc(surrogate buffers) failed");
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(ctx->stream) != hipSuccess)
    return fail(DGV_ERR_HIP, "surrogate initialisation kernels failed");
  *out = s;
  return DGV_OK;
}

void dgv_sur_destroy(dgv_surrogate* s) {
  if (!s) return;
  // the context may already be destroyed (a caller's finaliser order): use the
  // device recorded at creation and wait for the whole device, not the context's stream
  hipSetDevice(s->device);
  hipDeviceSynchronize();
  free_surrogate(s);
  delete s;
}

int dgv_sur_set_scales(dgv_surrogate* s, double f_scale, double q_scale) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (!(f_scale > 0) || !(q_scale > 0)) return serr(s, DGV_ERR_ARG, "scales must be positive");
  s->f_scale = f_scale;
  s->q_scale = q_scale;
  return DGV_OK;
}

int dgv_sur_layer_shape(const dgv_surrogate* s, int32_t layer, int32_t* in, int32_t* out) {
  if (!s || layer < 0 || layer >= s->L) { set_global_error("bad surrogate or layer"); return DGV_ERR_ARG; }
  if (in) *in = s->layers[layer].in;
  if (out) *out = s->layers[layer].out;
  return DGV_OK;
}

static int layer_copy(dgv_surrogate* s, int32_t layer, float* W, float* b, const float* Wd, const float* bd,
                      bool to_device) {
  if (!s || layer < 0 || layer >= s->L) { set_global_error("bad surrogate or layer"); return DGV_ERR_ARG; }
  SurLayer& ly = s->layers[layer];
  SHIP(s, hipSetDevice(s->ctx->device));
  SHIP(s, hipStreamSynchronize(s->ctx->stream));
  const size_t rowb = sizeof(float) * ly.in, pitch = sizeof(float) * ly.inp;
  hipStream_t st = s->ctx->stream;
  if (to_device) {
    if (W) SHIP(s, hipMemcpy2DAsync(const_cast<float*>(Wd), pitch, W, rowb, rowb, ly.out, hipMemcpyHostToDevice, st));
    if (b) SHIP(s, hipMemcpyAsync(const_cast<float*>(bd), b, sizeof(float) * ly.out, hipMemcpyHostToDevice, st));
  } else {
    // rows without padding are one copy; padded ones are made dense on the device first,
    // as many at a time as the partial sums' buffer holds (a pitched copy of 1024 x 3375
    // weights took 38 ms)
    const int64_t rows = pitch == rowb ? ly.out : std::min<int64_t>(ly.out, s->part_elems / ly.in);
    for (int64_t r = 0; W && r < ly.out; r += rows) {
      const int64_t n = std::min<int64_t>(rows, ly.out - r) * ly.in;
      const float* src = Wd + r * ly.inp;
      if (pitch != rowb) {
        hipLaunchKernelGGL(k_rows_dense, dim3(stride_blocks(n, 256)), dim3(256), 0, st, src, (int64_t)ly.inp,
                           (int64_t)ly.in, n, s->part);
        SHIP(s, hipGetLastError());
        src = s->part;
      }
      SHIP(s, hipMemcpyAsync(W + r * ly.in, src, sizeof(float) * n, hipMemcpyDeviceToHost, st));
    }
    if (b) SHIP(s, hipMemcpyAsync(b, bd, sizeof(float) * ly.out, hipMemcpyDeviceToHost, st));
  }
  SHIP(s, hipStreamSynchronize(st));
  return DGV_OK;
}

int dgv_sur_get_layer(dgv_surrogate* s, int32_t layer, float* W, float* b) {
  return s ? layer_copy(s, layer, W, b, layer >= 0 && layer < s->L ? s->layers[layer].W : nullptr,
                        layer >= 0 && layer < s->L ? s->layers[layer].b : nullptr, false)
           : layer_copy(s, layer, W, b, nullptr, nullptr, false);
}

int dgv_sur_set_layer(dgv_surrogate* s, int32_t layer, const float* W, const float* b) {
  if (!s || layer < 0 || layer >= s->L) { set_global_error("bad surrogate or layer"); return DGV_ERR_ARG; }
  SurLayer& ly = s->layers[layer];
  int rc = layer_copy(s, layer, const_cast<float*>(W), const_cast<float*>(b), ly.W, ly.b, true);
  if (rc) return rc;
  hipLaunchKernelGGL(k_weights_bf16, dim3(ly.inp / 64, ly.outp / 64), dim3(256), 0, s->ctx->stream, ly.outp, ly.inp,
                     ly.W, ly.Wf, ly.Wb);
  SHIP(s, hipGetLastError());
  SHIP(s, hipStreamSynchronize(s->ctx->stream));
  return DGV_OK;
}

int dgv_sur_get_grad(dgv_surrogate* s, int32_t layer, float* dW, float* db) {
  if (!s || layer < 0 || layer >= s->L) { set_global_error("bad surrogate or layer"); return DGV_ERR_ARG; }
  return layer_copy(s, layer, dW, db, s->layers[layer].G, s->layers[layer].gb, false);
}

int dgv_sur_train_step(dgv_surrogate* s, const double* d_f, const double* d_q, int64_t ld, int32_t nrows, double lr,
                       double* loss) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (!d_f || !d_q || nrows < 1 || nrows > s->batch || ld < s->ctx->g.N || !(lr >= 0))
    return serr(s, DGV_ERR_ARG, "train_step: bad argument");
  SHIP(s, hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  int rc = load_rows(s, d_f, ld, nrows);
  if (rc) return rc;
  const SurLayer& lo = s->layers[s->L - 1];
  const double inv_count = 1.0 / ((double)nrows * lo.out);
  int cur = 0;
  EpiArgs e{};
  e.q = const_cast<double*>(d_q);
  e.ld = ld;
  e.mvalid = nrows;
  e.nvalid = lo.out;
  e.scale = 1.0 / s->q_scale;
  e.gscale = (float)(2.0 * inv_count);
  e.h = s->dZ[cur];
  e.ht = s->dZt[cur];
  e.dbpart = s->dbpart[cur];
  e.losspart = s->losspart;
  if ((rc = forward(s, e, EPI_LOSS))) return rc;
  ++s->step;
  AdamArgs h;
  h.lr = (float)lr;
  h.b1 = 0.9f;
  h.b2 = 0.999f;
  h.eps = 1e-8f;
  h.c1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)s->step)));
  h.c2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)s->step)));
  for (int l = s->L - 1; l >= 0; --l) {
    SurLayer& ly = s->layers[l];
    if (l > 0) {  // gradient of the layer's input, through GELU of the previous layer
      const Gemm g = plan_gemm(s->Bp, ly.inp, ly.outp);
      if ((rc = launch_gemm(s, g, s->dZ[cur], ly.outp, ly.Wb, ly.outp, s->part))) return rc;
      EpiArgs a{};
      a.part = s->part;
      a.S = g.S;
      a.M = s->Bp;
      a.N = ly.inp;
      a.zin = s->Z[l - 1];
      a.h = s->dZ[cur ^ 1];
      a.ht = s->dZt[cur ^ 1];
      a.dbpart = s->dbpart[cur ^ 1];
      hipLaunchKernelGGL(k_epilogue<EPI_BWD_GELU>, dim3(ly.inp / 16, s->Bp / 64), dim3(256), 0, st, a);
    }
    const bool last = l + 1 == s->L;   // its launch adds the loss too
    const BiasArgs ba{s->dbpart[cur], s->Bp / 64, ly.gb, ly.b, ly.mb, ly.vb, s->losspart,
                      (lo.outp / 16) * (s->Bp / 64), inv_count, s->h_loss};
    const int nwg = (ly.inp / 64) * (ly.outp / 64) + (ly.outp + 255) / 256 + (last ? 1 : 0);
    hipLaunchKernelGGL(k_grad_update, dim3((unsigned)nwg), dim3(256), 0, st, ly.outp, ly.inp, s->Bp, s->dZt[cur],
                       s->Ht[l], ly.G, ly.W, ly.mW, ly.vW, ly.Wf, ly.Wb, lr > 0 ? 1 : 0, h, ba);
    cur ^= 1;
  }
  SHIP(s, hipGetLastError());
  if (loss) {
    SHIP(s, hipStreamSynchronize(st));
    *loss = *(volatile double*)s->h_loss;
  }
  return DGV_OK;
}

int dgv_sur_predict(dgv_surrogate* s, const double* d_f, int64_t ld, int64_t nrows, double* d_q, int32_t project) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (!d_f || !d_q || nrows < 0 || ld < s->ctx->g.N) return serr(s, DGV_ERR_ARG, "predict: bad argument");
  SHIP(s, hipSetDevice(s->ctx->device));
  if (int rc = decomp_check(s)) return rc;
  for (int64_t r = 0; r < nrows; r += s->batch) {
    const int nb = (int)std::min<int64_t>(s->batch, nrows - r);
    int rc = predict_rows(s, d_f + r * ld, ld, nb, d_q + r * ld, project);
    if (rc) return rc;
  }
  return DGV_OK;
}

int dgv_sur_set_decomposition(dgv_surrogate* s, int32_t on) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (!on) {
    s->decomp = 0;
    return DGV_OK;
  }
  dgv_ctx* c = s->ctx;
  if (s->layers.front().in != c->g.N || s->layers.back().out != c->g.N)
    return serr(s, DGV_ERR_ARG, "decomposition mode needs node-sized input and output layers");
  if (!c->lin.fma_valid) return serr(s, DGV_ERR_STATE, "no linearised operator (PrepareFMA)");
  SHIP(s, hipSetDevice(c->device));
  const size_t bytes = sizeof(double) * (size_t)s->batch * (size_t)c->g.N;
  struct { double** p; size_t n; } bufs[] = {{&s->d_df, bytes}, {&s->d_lin, bytes},
                                             {&s->d_qfm, sizeof(double) * (size_t)c->g.N},
                                             {&s->d_rs, sizeof(double) * (size_t)s->batch}};
  for (auto& b : bufs)
    if (!*b.p && hipMalloc(b.p, b.n) != hipSuccess) {
      *b.p = nullptr;
      (void)hipGetLastError();
      return serr(s, DGV_ERR_NOMEM, "hipMalloc(decomposition buffers) failed");
    }
  // Q(fm), the part of the split that the reference's run_mode 1 leaves out
  int rc = eval_q_dev(c, c->lin.d_vec[0], s->d_qfm, 1.0);
  if (rc) return rc;
  SHIP(s, hipStreamSynchronize(c->stream));
  s->decomp = 1;
  s->decomp_gen = c->lin.nprepare;
  return DGV_OK;
}

int dgv_sur_set_probe_cells(dgv_surrogate* s, const int32_t* cells, int32_t ncells) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (ncells < 1 || !cells) return serr(s, DGV_ERR_ARG, "at least one probe cell is needed");
  SHIP(s, hipSetDevice(s->ctx->device));
  const Grid& g = s->ctx->g;
  std::vector<int32_t> cl(cells, cells + ncells);
  std::sort(cl.begin(), cl.end());
  cl.erase(std::unique(cl.begin(), cl.end()), cl.end());
  for (int32_t c : cl)
    if (c < 0 || c >= g.ncells) return serr(s, DGV_ERR_INDEX, "probe cell outside the grid");
  if (s->judge && batch_stale(s->judge)) {   // the A-array changed: judge with the current one
    dgv_batch_destroy(s->judge);
    s->judge = nullptr;
  }
  if (!s->judge) {
    std::vector<int32_t> goi(s->batch, 0);
    dgv_ctx* grids[1] = {s->ctx};
    int rc = dgv_batch_create(grids, 1, goi.data(), s->batch, DGV_FP64, &s->judge);
    if (rc) return serr(s, rc, std::string("judge batch: ") + dgv_last_error(nullptr));
  }
  int rc = dgv_batch_set_probe_cells(s->judge, cl.data(), (int32_t)cl.size());
  if (rc) return serr(s, rc, std::string("judge probe plan: ") + dgv_last_error(nullptr));
  std::vector<int32_t> nodes;
  for (int32_t c : cl)
    for (int l = 0; l < g.D; ++l) nodes.push_back(c * g.D + l);
  hipFree(s->d_probe_nodes);
  s->d_probe_nodes = nullptr;
  SHIP(s, hipMalloc(&s->d_probe_nodes, sizeof(int32_t) * nodes.size()));
  SHIP(s, hipMemcpyAsync(s->d_probe_nodes, nodes.data(), sizeof(int32_t) * nodes.size(), hipMemcpyHostToDevice,
                         s->ctx->stream));
  SHIP(s, hipStreamSynchronize(s->ctx->stream));
  s->nprobe_nodes = (int)nodes.size();
  s->probe_cells = cl;
  return DGV_OK;
}

int dgv_sur_eval(dgv_surrogate* s, const double* d_f, int64_t ld, int64_t nrows, double* d_q, double tol,
                 double* residual, int32_t* fallback, int64_t* nfallback) {
  if (!s) { set_global_error("null surrogate"); return DGV_ERR_ARG; }
  if (!d_f || !d_q || nrows < 0 || ld < s->ctx->g.N || !(tol >= 0)) return serr(s, DGV_ERR_ARG, "eval: bad argument");
  if (!s->judge || s->nprobe_nodes == 0) return serr(s, DGV_ERR_STATE, "no probe cells set");
  SHIP(s, hipSetDevice(s->ctx->device));
  if (int rc = decomp_check(s)) return rc;
  if (batch_stale(s->judge)) {   // the A-array changed since the probe plan: rebuild it on the current one
    const std::vector<int32_t> cl = s->probe_cells;
    int rc = dgv_sur_set_probe_cells(s, cl.data(), (int32_t)cl.size());
    if (rc) return rc;
  }
  dgv_ctx* ctx = s->ctx;
  double *jf = nullptr, *jq = nullptr;
  int64_t off = 0, stride = 0;
  int rc = dgv_batch_device_buffers(s->judge, &jf, &jq);
  if (!rc) rc = dgv_batch_layout(s->judge, 0, &off, &stride, nullptr);
  if (rc) return serr(s, rc, dgv_last_error(nullptr));
  std::vector<double> res(s->batch);
  int64_t nfb = 0;
  for (int64_t r = 0; r < nrows; r += s->batch) {
    const int nb = (int)std::min<int64_t>(s->batch, nrows - r);
    const double* F = d_f + r * ld;
    double* Q = d_q + r * ld;
    // the residual compares like with like: the network's Q before the
    // projection against the direct Q; the kept rows are projected after it
    if ((rc = predict_rows(s, F, ld, nb, Q, 0))) return rc;
    hipLaunchKernelGGL(k_rows_to_packed, dim3((unsigned)((ctx->g.N + 63) / 64), (unsigned)((nb + 63) / 64)), dim3(256),
                       0, ctx->stream, F, ld, nb, (int)ctx->g.N, jf + off, stride);
    SHIP(s, hipGetLastError());
    SHIP(s, hipStreamSynchronize(ctx->stream));
    if ((rc = dgv_batch_eval_q_probe(s->judge))) return serr(s, rc, dgv_last_error(nullptr));
    hipLaunchKernelGGL(k_probe_residual, dim3(nb), dim3(256), 0, ctx->stream, Q, ld, jq + off, stride,
                       s->d_probe_nodes, s->nprobe_nodes, s->d_res);
    SHIP(s, hipGetLastError());
    hipLaunchKernelGGL(k_project_rows, dim3(nb), dim3(256), 0, ctx->stream, Q, ld, (int)ctx->g.N, ctx->d_u, ctx->d_v,
                       ctx->d_w, ctx->d_gwts, s->chol);
    SHIP(s, hipGetLastError());
    SHIP(s, hipMemcpyAsync(res.data(), s->d_res, sizeof(double) * nb, hipMemcpyDeviceToHost, ctx->stream));
    SHIP(s, hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < nb; ++i) {
      const bool fb = !(res[i] <= tol);
      if (residual) residual[r + i] = res[i];
      if (fallback) fallback[r + i] = fb ? 1 : 0;
      if (fb) {
        ++nfb;
        if ((rc = eval_q_dev(ctx, F + (int64_t)i * ld, Q + (int64_t)i * ld, 1.0))) return rc;
      }
    }
  }
  SHIP(s, hipStreamSynchronize(ctx->stream));
  if (nfallback) *nfallback = nfb;
  return DGV_OK;
}

int dgv_sur_time_predict(dgv_surrogate* s, const double* d_f, int64_t ld, int64_t nrows, double* d_q, int32_t niter,
                         double* ms_per_call) {
  if (!s || niter < 1) { set_global_error("bad argument"); return DGV_ERR_ARG; }
  dgv_ctx* ctx = s->ctx;
  SHIP(s, hipSetDevice(ctx->device));
  SHIP(s, hipEventRecord(ctx->ev[0], ctx->stream));
  for (int i = 0; i < niter; ++i) {
    int rc = dgv_sur_predict(s, d_f, ld, nrows, d_q, 1);
    if (rc) return rc;
  }
  SHIP(s, hipEventRecord(ctx->ev[1], ctx->stream));
  SHIP(s, hipEventSynchronize(ctx->ev[1]));
  float ms = 0;
  SHIP(s, hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
  if (ms_per_call) *ms_per_call = ms / niter;
  return DGV_OK;
}

}  // extern "C"
