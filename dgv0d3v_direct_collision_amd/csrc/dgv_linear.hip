// dgv_linear.hip -- the decomposition and linearised regimes on the device.
//
//   PrepareFMA_DGV        collision_mod.f90:377-464   dense fmA = (1/w_i) sum A fm  (N x N)
//   EvalCollisionLinear   collision_mod.f90:346-359   fc = 2 f . fmA (GEMV, HBM bound)
//   CheckSolutionMode_DGV spat_oper_mod.f90:195-272   regime switch on |f - f_M|_1
//   SpatialOperSH_DGV     spat_oper_mod.f90:28-68     run_mode 0 / 1 / 2
//
// fmA lives in HBM row-major over its first index: element fmA(r, i) (row r =
// the node the record's f_M factor does NOT multiply, column i = the output
// node) is at d_fma[r * N + i].  Column i of the reference's array is the
// stride-N sequence; the GEMV reads rows (contiguous in i) and the build writes
// each lane's 27 columns of one cell contiguously.
//
// Build, deterministic and without atomics: the entries of the tile (column
// cell c, row cell c + e) receive
//   term 1: sum over blocks with a = e, pairs (s, q):  T[l] fm[c+b][q]
//   term 2: sum over blocks with b = e, pairs (p, s):  T[l] fm[c+a][p]
// (the reference's two scatter-adds per record, lines 447-448), then the
// division by w_i (line 458).  For one (e, s) that is a matrix product over all
// those pairs, 27 basis functions by the column cells: its list of (pair, offset of
// the partner's fm) is laid out once per A-array, and fm is read from a copy with
// a halo of zeros around the grid, so that partners off the grid add nothing.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <vector>

#include "dgv_internal.h"

namespace dgv {

typedef double ld2 __attribute__((ext_vector_type(2)));
typedef double ld4 __attribute__((ext_vector_type(4)));

// The column cells of one row offset e (their box), for the workgroup's four rows
// s = 4 sgroup .. and 64 of the cells
struct FmaItem {
  int32_t e[3], sgroup;
  int32_t lo[3], ext[3];
  int32_t ncells, chunk;   // chunk < 0: empty slot
  int32_t elin, pad;       // index of e among the (2 M - 1) offsets per dimension
};

// The grid with a halo of M - 1 cells of zeros on every side
struct FmaDims {
  int32_t Mu, Mv, Mw;
  __host__ __device__ int eu() const { return 3 * Mu - 2; }
  __host__ __device__ int ev() const { return 3 * Mv - 2; }
  __host__ __device__ int ew() const { return 3 * Mw - 2; }
  __host__ __device__ int64_t ncext() const { return (int64_t)eu() * ev() * ew(); }
};

// One workgroup per block in turn: idx[(block) D D + p D + q] = the pair (p, q) of the block, or -1
__global__ __launch_bounds__(256) void k_pair_index(int D, int64_t nblocks, const BlockHdr* __restrict__ blocks,
                                                    const double* __restrict__ pairs, int16_t* __restrict__ idx) {
  __shared__ int16_t t[64 * 64];
  const int DD = D * D;
  for (int64_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
    const BlockHdr* B = blocks + b;
    for (int i = threadIdx.x; i < DD; i += blockDim.x) t[i] = -1;
    __syncthreads();
    const int n = B->seg[D];
    const double* P = pairs + B->pbeg * (D + 1);
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      const int code = (int)(__double_as_longlong(P[(int64_t)k * (D + 1) + D]) & 0xffff);
      t[(code >> 8) * D + (code & 255)] = (int16_t)k;
    }
    __syncthreads();
    int16_t* out = idx + b * DD;
    for (int i = threadIdx.x; i < DD; i += blockDim.x) out[i] = t[i];
    __syncthreads();   // the table is read
  }
}

int launch_pair_index(dgv_ctx* ctx, int16_t* d_idx) {
  const int64_t nb = (int64_t)ctx->pb.blocks.size();
  if (nb > 0)
    hipLaunchKernelGGL(k_pair_index, dim3(loop_blocks(nb)), dim3(256), 0, ctx->stream, ctx->g.D, nb, ctx->pb.d_blocks,
                       ctx->pb.d_pairs, d_idx);
  DGV_HIP(ctx, hipGetLastError());
  return DGV_OK;
}

// fm with its halo, node of the cell outer: X[t][cell of the extended grid]; a last
// plane t = D of zeros is the partner of the lists' padding
__global__ void k_fma_halo(FmaDims g, int D, const double* __restrict__ fm, double* __restrict__ X) {
  const int64_t nc = g.ncext(), n = nc * (D + 1), step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const int t = (int)(i / nc);
    const int64_t c = i - t * nc;
    const int w = (int)(c % g.ew()) - (g.Mw - 1), v = (int)(c / g.ew() % g.ev()) - (g.Mv - 1),
              u = (int)(c / ((int64_t)g.ew() * g.ev())) - (g.Mu - 1);
    const bool in = t < D && u >= 0 && u < g.Mu && v >= 0 && v < g.Mv && w >= 0 && w < g.Mw;
    X[i] = in ? fm[(int64_t)((u * g.Mv + v) * g.Mw + w) * D + t] : 0.0;
  }
}

// One workgroup per row offset e: the entries (pair, byte offset in X of the
// partner relative to the column cell) of every s, blocks in list order, pairs in
// the order of the partner's node.  Without `desc` only counts them.
template <int D>
__global__ __launch_bounds__(256) void k_fma_lists(FmaDims g, const int32_t* __restrict__ p1, const int32_t* __restrict__ l1,
                                                   const int32_t* __restrict__ p2, const int32_t* __restrict__ l2,
                                                   const BlockHdr* __restrict__ blocks,
                                                   const double* __restrict__ pairs, uint32_t zero_pair,
                                                   const int64_t* __restrict__ beg, uint2* __restrict__ desc,
                                                   uint32_t* __restrict__ cnt) {
  __shared__ int32_t tab[D * D];
  __shared__ uint32_t off[D];
  const int64_t e = blockIdx.x;
  const int nc = (int)g.ncext();
  auto xoff = [&](const int8_t* o, int t) {
    return (uint32_t)((t * nc + (o[0] * g.ev() + o[1]) * g.ew() + o[2]) * 8);
  };
  if (threadIdx.x < D) off[threadIdx.x] = 0;
  __syncthreads();
  for (int k = p1[e]; k < p1[e + 1]; ++k) {
    const BlockHdr& B = blocks[l1[k]];
    if (desc)
      for (int j = threadIdx.x; j < B.npairs; j += 256) {
        const int code = (int)(__double_as_longlong(pairs[(B.pbeg + j) * (D + 1) + D]) & 0xffff);
        const int s = code >> 8;
        desc[beg[e * D + s] + off[s] + (j - B.seg[s])] = make_uint2((uint32_t)(B.pbeg + j), xoff(B.b, code & 255));
      }
    __syncthreads();
    if (threadIdx.x < D) off[threadIdx.x] += B.seg[threadIdx.x + 1] - B.seg[threadIdx.x];
    __syncthreads();
  }
  for (int k = p2[e]; k < p2[e + 1]; ++k) {
    const BlockHdr& B = blocks[l2[k]];
    for (int i = threadIdx.x; i < D * D; i += 256) tab[i] = -1;
    __syncthreads();
    for (int j = threadIdx.x; j < B.npairs; j += 256) {
      const int code = (int)(__double_as_longlong(pairs[(B.pbeg + j) * (D + 1) + D]) & 0xffff);
      tab[(code >> 8) * D + (code & 255)] = j;
    }
    __syncthreads();
    if (threadIdx.x < D) {
      const int s = threadIdx.x;
      uint32_t r = off[s];
      for (int p = 0; p < D; ++p) {
        const int j = tab[p * D + s];
        if (j < 0) continue;
        if (desc) desc[beg[e * D + s] + r] = make_uint2((uint32_t)(B.pbeg + j), xoff(B.a, p));
        ++r;
      }
      off[s] = r;
    }
    __syncthreads();
  }
  if (threadIdx.x < D) {
    const int64_t i = e * D + threadIdx.x;
    if (!desc) {
      cnt[i] = off[threadIdx.x];
    } else {   // the list's end: a pair of zero coefficients, the plane of zeros
      for (int64_t k = beg[i] + off[threadIdx.x]; k < beg[i + 1]; ++k) desc[k] = make_uint2(zero_pair, (uint32_t)(D * nc * 8));
    }
  }
}

// One wave per (e, s, 64 column cells): A = 16 basis functions x 4 pairs, B = 4 pairs
// x 16 cells of v_mfma_f64_16x16x4_f64, two row tiles and CT column tiles.  The list
// entries are two rings ahead, the operands one.  The gathers of fm bound it (seven
// loads per eight products, matrix cores busy 52 %), and half the products meet the
// halo's zeros: 65 ms at 27^3 nodes against 148 ms with one lane per cell and
// scalar coefficients.
constexpr int kFmaRing = 4;                  // also the lists' padding in steps
constexpr int kFmaListPad = 4 * 2 * kFmaRing;   // entries past the last list that the rings read

template <int D, int CT>
__device__ __forceinline__ void fma_walk(int64_t nsteps, const uint2* __restrict__ list, const double* __restrict__ pairs,
                                         const double* __restrict__ X, const uint32_t (&xb)[4], int jj, int kk,
                                         ld4 (&acc)[(D + 15) / 16][4]) {
  constexpr int RT = (D + 15) / 16, R = kFmaRing;
  uint2 d[R];
  double a[R][RT], b[R][CT];
  auto entry = [&](int u, int64_t i) { d[u] = list[4 * i + kk]; };
  auto operands = [&](int u) {
    const double* T = pairs + (int64_t)d[u].x * (D + 1) + jj;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) a[u][rt] = T[16 * rt];   // rows past D: dropped on output
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      b[u][ct] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(X) + (uint32_t)(xb[ct] + d[u].y));
  };
#pragma unroll
  for (int u = 0; u < R; ++u) entry(u, u);
#pragma unroll
  for (int u = 0; u < R; ++u) {
    operands(u);
    entry(u, u + R);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int64_t i = 0; i < nsteps; i += R) {   // lists are padded to whole rounds
#pragma unroll
    for (int u = 0; u < R; ++u) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][rt], b[u][ct], acc[rt][ct], 0, 0, 0);
      // loads in slot order: the waits count them
      __builtin_amdgcn_sched_barrier(0);
      operands(u);
      entry(u, i + u + 2 * R);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int D>
__global__ __launch_bounds__(256, 2) void k_fma_build(const FmaItem* __restrict__ items, FmaDims g,
                                                      const int64_t* __restrict__ beg, const uint2* __restrict__ desc,
                                                      const double* __restrict__ pairs, const double* __restrict__ X,
                                                      const double* __restrict__ gwts, int64_t N,
                                                      double* __restrict__ out) {
  constexpr int RT = (D + 15) / 16;
  const FmaItem& it = items[blockIdx.x];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int s = it.sgroup * 4 + wave, chunk = it.chunk;
  if (chunk < 0 || s >= D) return;
  const int kk = lane >> 4, jj = lane & 15;
  const int ncols = min(64, it.ncells - chunk * 64);
  const int ct_n = (ncols + 15) / 16;
  uint32_t xb[4];
  int32_t cell[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    const int c = chunk * 64 + 16 * ct + jj;
    int r = c < it.ncells ? c : chunk * 64;   // idle columns follow the chunk's first cell
    const int cw = it.lo[2] + r % it.ext[2];
    r /= it.ext[2];
    const int cv = it.lo[1] + r % it.ext[1];
    r /= it.ext[1];
    const int cu = it.lo[0] + r;
    cell[ct] = c < it.ncells ? (cu * g.Mv + cv) * g.Mw + cw : -1;
    xb[ct] = (uint32_t)((((cu + g.Mu - 1) * g.ev() + cv + g.Mv - 1) * g.ew() + cw + g.Mw - 1) * 8);
  }
  ld4 acc[RT][4];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) acc[rt][ct] = ld4{0.0, 0.0, 0.0, 0.0};
  const int64_t b0 = beg[(int64_t)it.elin * D + s], b1 = beg[(int64_t)it.elin * D + s + 1];
  const uint2* list = desc + b0;
  const int64_t nsteps = (b1 - b0) / 4;
  if (nsteps > 0) {
    switch (ct_n) {
      case 1: fma_walk<D, 1>(nsteps, list, pairs, X, xb, jj, kk, acc); break;
      case 2: fma_walk<D, 2>(nsteps, list, pairs, X, xb, jj, kk, acc); break;
      case 3: fma_walk<D, 3>(nsteps, list, pairs, X, xb, jj, kk, acc); break;
      default: fma_walk<D, 4>(nsteps, list, pairs, X, xb, jj, kk, acc); break;
    }
  }
  const int de = (it.e[0] * g.Mv + it.e[1]) * g.Mw + it.e[2];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    if (cell[ct] < 0) continue;
    const int64_t row = (int64_t)(cell[ct] + de) * D + s, col = (int64_t)cell[ct] * D;
    double* o = out + row * N + col;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int l = 16 * rt + 4 * k + kk;   // FP64 output layout
        if (l < D) o[l] = acc[rt][ct][k] / gwts[col + l];
      }
  }
}

// fc = 2 f . fmA for nv vectors on the matrix cores: C[v][i] = sum_r f[v][r] fmA[r][i]
// with v_mfma_f64_16x16x4_f64, A = 16 vectors x 4 rows r (from LDS), B = 4 rows x 16
// columns i, straight from fmA (a lane's two columns are one 16-byte load, a row's
// 32 columns 256 contiguous bytes).  A workgroup of four waves takes 128 columns, 16
// VT vectors and a chunk of rows; the chunks' sums are added in order by k_fma_sum.
// One pass serves up to kLinVec vectors: up to about 50 the reading of fmA bounds it,
// above them the matrix cores.  27^3 nodes (3.1 GB): 2 vectors 0.53 ms (5.8 TB/s), 32
// 0.63, 64 0.97, 128 1.86, 256 3.66 ms (54 TFLOP/s); a pass over fmA per 8 vectors
// on the vector units took 0.61, 3.1, 6.2, 12.3 and 24.7 ms.  (Tiles of 128 vectors, 3.45 ms, leave
// no registers for the running sums; with one wave per SIMD they take 4.16 ms.)
// rows of fmA per LDS tile of f (32 and 64 rows for the smaller vector tiles: 1-3 %
// slower at 27^3 nodes, no faster at 15^3)
constexpr int kLinRows = 16;
constexpr int kLinCols = 128;    // columns per workgroup
// rows whose products are added in one chain before they join the running sum (a chunk in one chain, about
// 1500 rows at 27^3 nodes, is 1.6 to 2 times as far from extended precision as chunks of 256; chains of
// 256 / 128 / 64: 9.1 / 5.2 / 5.2e-16 there for one vector, 256 vectors 3.65 / 3.66 / 3.71 ms)
constexpr int kLinSum = 128;
constexpr int kLinVec = 256;     // vectors per pass

template <int VT>
__global__ __launch_bounds__(256, 2) void k_fma_rows(int64_t N, int nv, int colblocks, int vblocks, int64_t chunk,
                                                     const double* __restrict__ fma, const double* __restrict__ f,
                                                     int64_t ldf, double* __restrict__ part) {
  constexpr int BM = 16 * VT, P = kLinRows + 2;   // LDS pitch: 16 vectors x 2 rows cover the 64 banks once
  constexpr int NL = BM * kLinRows / 256;         // f values per thread and tile
  constexpr int KS = kLinRows / 4;
  __shared__ double fs[2][BM * P];
  // the vector blocks of one (column block, chunk) read the same fmA: neighbours on one XCD
  const int w = blockIdx.x, x = w & 7, y = w >> 3;
  const int vb = y % vblocks, pos = (y / vblocks) * 8 + x;
  const int cb = pos % colblocks;
  const int64_t ck = pos / colblocks;
  const int64_t r0 = ck * chunk, r1 = min(N, r0 + chunk);
  if (r0 >= r1) return;   // the grid is padded to whole groups of eight
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kk = lane >> 4, jj = lane & 15;
  const int64_t col = (int64_t)cb * kLinCols + wave * 32 + 2 * jj;
  const int64_t cl = min(col, N - 2);            // the last columns' pair is read inside the row
  const int v0 = vb * BM;
  // this thread's f elements of a tile: vectors fr + FR i, row fc
  constexpr int FR = 256 / kLinRows;
  const int fr = threadIdx.x / kLinRows, fc = threadIdx.x % kLinRows;
  double fv[NL];
  auto fload = [&](int64_t r) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int v = v0 + fr + FR * i;
      fv[i] = (v < nv && r + fc < r1) ? f[(int64_t)v * ldf + r + fc] : 0.0;
    }
  };
  auto fstore = [&](int b) {
#pragma unroll
    for (int i = 0; i < NL; ++i) fs[b][(fr + FR * i) * P + fc] = fv[i];
  };
  ld2 bt[2][KS];
  auto bload = [&](int b, int64_t r) {
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const double* p = fma + min(r + 4 * k + kk, N - 1) * N + cl;   // chunks but the last are whole tiles
      __builtin_memcpy(&bt[b][k], p, 16);
    }
    if (r + kLinRows > N) {   // no rows: zeros, as an infinite last row would not vanish against a zero of f
#pragma unroll
      for (int k = 0; k < KS; ++k)
        if (r + 4 * k + kk >= N) bt[b][k] = ld2{0.0, 0.0};
    }
  };
  ld4 sum[VT][2], acc[VT][2];
#pragma unroll
  for (int t = 0; t < VT; ++t) sum[t][0] = sum[t][1] = ld4{0.0, 0.0, 0.0, 0.0};
  fload(r0);
  bload(0, r0);
  auto tile = [&](int b, int64_t r) {   // b: this tile's buffers (constant after unrolling)
    fstore(b);
    __syncthreads();
    if (r + kLinRows < r1) {
      fload(r + kLinRows);
      bload(b ^ 1, r + kLinRows);
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      double a[VT];
#pragma unroll
      for (int t = 0; t < VT; ++t) a[t] = fs[b][(16 * t + jj) * P + 4 * k + kk];
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        acc[t][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], bt[b][k][0], acc[t][0], 0, 0, 0);
        acc[t][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], bt[b][k][1], acc[t][1], 0, 0, 0);
      }
    }
  };
  for (int64_t rs = r0; rs < r1; rs += kLinSum) {
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[t][0] = acc[t][1] = ld4{0.0, 0.0, 0.0, 0.0};
    for (int64_t r = rs; r < min(r1, rs + kLinSum); r += 2 * kLinRows) {
      tile(0, r);
      if (r + kLinRows < r1) tile(1, r + kLinRows);
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) {
      sum[t][0] += acc[t][0];
      sum[t][1] += acc[t][1];
    }
  }
  // output layout: element e of lane jj + 16 kk is row (vector) 4 e + kk, columns col, col + 1
  double* out = part + ck * nv * N;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int v = v0 + 16 * t + 4 * e + kk;
      if (v >= nv) continue;
      if (col < N) out[(int64_t)v * N + col] = cl == col ? sum[t][0][e] : sum[t][1][e];
      if (col + 1 < N) out[(int64_t)v * N + col + 1] = sum[t][1][e];
    }
}

// One vector on the vector units: no rows of zeros to multiply (15^3 nodes: 19.8
// us against 22.8; 27^3 nodes the same, both at the card's read rate).  Adds a
// column's rows one after the other, as the matrix cores do: the sums are the
// same to the last bit.
__global__ __launch_bounds__(256) void k_fma_gemv(int64_t N, int64_t chunk, const double* __restrict__ fma,
                                                  const double* __restrict__ f, double* __restrict__ part) {
  constexpr int kU = 16;     // row loads in flight per thread
  constexpr int kF = 256;    // rows of f in LDS
  static_assert(kF % kLinSum == 0 && kLinSum % kU == 0, "chains end where the tiles do");
  __shared__ double fs[kF];
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.y * chunk, r1 = min(N, r0 + chunk);
  const double* col = fma + (i < N ? i : N - 1);
  double sum = 0.0;
  for (int64_t b = r0; b < r1; b += kF) {
    const int nr = (int)min((int64_t)kF, r1 - b);
    __syncthreads();
    fs[threadIdx.x] = (int)threadIdx.x < nr ? f[b + threadIdx.x] : 0.0;
    __syncthreads();
    double acc = 0.0;
    int r = 0;
    for (; r + kU <= nr; r += kU) {
      double m[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) m[u] = col[(b + r + u) * N];
#pragma unroll
      for (int u = 0; u < kU; ++u) acc = __fma_rn(fs[r + u], m[u], acc);
      if ((r + kU) % kLinSum == 0) {
        sum += acc;
        acc = 0.0;
      }
    }
    for (; r < nr; ++r) acc = __fma_rn(fs[r], col[(b + r) * N], acc);
    sum += acc;
  }
  if (i < N) part[(int64_t)blockIdx.y * N + i] = sum;
}

__global__ void k_fma_sum(int64_t N, int nchunk, int nv, const double* __restrict__ part, double* __restrict__ fc,
                          int64_t ldq) {
  const int64_t n = N * nv, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += step) {
    double s = 0.0;
    int c = 0;
    for (; c + 8 <= nchunk; c += 8) {   // eight loads in flight, added in order
      double x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = part[(int64_t)(c + i) * n + t];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += x[i];
    }
    for (; c < nchunk; ++c) s += part[(int64_t)c * n + t];
    const int64_t v = t / N;
    fc[v * ldq + (t - v * N)] = 2.0 * s;
  }
}

// How a pass over nv vectors is cut: vector tiles per workgroup (0: k_fma_gemv) and
// chunks of rows.  The chunks depend on N alone, so that a vector's result does not
// depend on how many are passed with it: about two rounds of workgroups for one
// vector tile, 256 rows at least.
struct LinPlan {
  int vt, vblocks, colblocks, nchunk;
  int64_t chunk;
};
static LinPlan lin_plan(int64_t N, int nv) {
  LinPlan p;
  p.vt = nv == 1 ? 0 : nv <= 16 ? 1 : nv <= 32 ? 2 : 4;
  p.vblocks = p.vt == 0 ? 1 : (nv + 16 * p.vt - 1) / (16 * p.vt);
  p.colblocks = (int)((N + kLinCols - 1) / kLinCols);
  const int64_t s = std::max<int64_t>(1, std::min<int64_t>(N / 256, 2048 / p.colblocks));
  p.chunk = ((N + s - 1) / s + kLinRows - 1) / kLinRows * kLinRows;
  p.nchunk = (int)((N + p.chunk - 1) / p.chunk);
  return p;
}

// maxwelveldist (distributions_mod.f90:83-94) at every node
__global__ void k_maxwell(int64_t n, double T, double u0, double v0, double w0, double dens,
                          const double* __restrict__ u, const double* __restrict__ v,
                          const double* __restrict__ w, double* __restrict__ out) {
  const double pi = 3.14159265358979323846264338327950288;
  const double beta = sqrt(pi * T) * (pi * T);
  const double tt = T > 0.0000001 ? T : 0.0000001;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const double du = u[i] - u0, dv = v[i] - v0, dw = w[i] - w0;
    out[i] = dens * exp(-(du * du + dv * dv + dw * dw) / tt) / beta;
  }
}

// sum |a - b| w, fixed-order two-level reduction (256 blocks, then one thread)
constexpr int kL1Blocks = 256;

__global__ __launch_bounds__(256) void k_l1_part(int64_t n, const double* __restrict__ a,
                                                 const double* __restrict__ b, const double* __restrict__ w,
                                                 double* __restrict__ part) {
  __shared__ double red[256];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)kL1Blocks * 256)
    s += fabs(a[i] - b[i]) * w[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_l1_final(const double* __restrict__ part, double* __restrict__ out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double s = 0.0;
  for (int b = 0; b < kL1Blocks; ++b) s += part[b];
  out[0] = s;
}

__global__ void k_sub(int64_t n, const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) out[i] = a[i] - b[i];
}

// out = (x + y) * scale, or x * scale when y is null
__global__ void k_sum_scale(int64_t n, const double* __restrict__ x, const double* __restrict__ y, double scale,
                            double* __restrict__ out) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step)
    out[i] = (y ? x[i] + y[i] : x[i]) * scale;
}

// ---------------------------------------------------------------------------

void free_linear(dgv_ctx* ctx) {
  LinearState& L = ctx->lin;
  hipFree(L.d_fma); hipFree(L.d_items); hipFree(L.d_beg); hipFree(L.d_desc); hipFree(L.d_halo);
  hipFree(L.d_part);
  L.d_fma = nullptr; L.d_items = nullptr; L.d_beg = nullptr; L.d_desc = nullptr; L.d_halo = nullptr;
  L.d_part = nullptr;
  L.part_vec = 0;
  L.nitems = 0;
  L.fma_valid = false;
  L.run_mode = 0;
}

void free_linear_vectors(dgv_ctx* ctx) {
  LinearState& L = ctx->lin;
  for (int k = 0; k < 5; ++k) { hipFree(L.d_vec[k]); L.d_vec[k] = nullptr; }
}

static int ensure_vectors(dgv_ctx* ctx) {
  LinearState& L = ctx->lin;
  if (L.d_vec[0]) return DGV_OK;
  for (int k = 0; k < 5; ++k) {
    const size_t nb = sizeof(double) * (k == 4 ? 2 * kL1Blocks : std::max<int64_t>(ctx->g.N, 1));
    if (hipMalloc(&L.d_vec[k], nb) != hipSuccess) {
      free_linear_vectors(ctx);
      return set_error(ctx, DGV_ERR_NOMEM, "hipMalloc(linearised-regime vectors) failed");
    }
  }
  return DGV_OK;
}

// The lists of every (e, s) and the work items (once per A-array).
template <int D>
static int build_fma_plan(dgv_ctx* ctx) {
  LinearState& L = ctx->lin;
  const Grid& g = ctx->g;
  const PairBlock& pb = ctx->pb;
  const FmaDims dims{g.Mu, g.Mv, g.Mw};
  const int M[3] = {g.Mu, g.Mv, g.Mw};
  const int64_t ne = (int64_t)(2 * M[0] - 1) * (2 * M[1] - 1) * (2 * M[2] - 1);
  if (pb.npairs >= (int64_t)UINT32_MAX || dims.ncext() * (D + 1) * 8 > (int64_t)INT32_MAX)
    return set_error(ctx, DGV_ERR_UNSUPPORTED, "PrepareFMA: grid or A-array too large");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  // block lists by offset (a for term 1, b for term 2), blocks in layout order
  auto elin = [&](const int8_t* o) {
    return ((int64_t)(o[0] + M[0] - 1) * (2 * M[1] - 1) + (o[1] + M[1] - 1)) * (2 * M[2] - 1) + (o[2] + M[2] - 1);
  };
  const int64_t nb = (int64_t)pb.blocks.size();
  std::vector<int32_t> ptr[2], list[2];
  for (int t = 0; t < 2; ++t) {
    ptr[t].assign(ne + 1, 0);
    for (const BlockHdr& B : pb.blocks) ptr[t][elin(t ? B.b : B.a) + 1]++;
    for (int64_t e = 0; e < ne; ++e) ptr[t][e + 1] += ptr[t][e];
    list[t].resize(std::max<int64_t>(nb, 1));
    std::vector<int32_t> at(ptr[t].begin(), ptr[t].end() - 1);
    for (int64_t k = 0; k < nb; ++k) list[t][at[elin(t ? pb.blocks[k].b : pb.blocks[k].a)]++] = (int32_t)k;
  }
  // items: every (row cell, column cell) pair of the grid belongs to one e, so the
  // whole operator is written, zeros included
  std::vector<FmaItem> items;
  std::vector<int64_t> epairs(ne, 0);
  for (const BlockHdr& B : pb.blocks) {
    epairs[elin(B.a)] += B.npairs;
    epairs[elin(B.b)] += B.npairs;
  }
  constexpr int NS = (D + 3) / 4, kXcd = 8;
  std::vector<FmaItem> col[kXcd];
  std::vector<int64_t> order(ne);
  std::vector<FmaItem> proto(ne);
  int64_t k = 0;
  for (int e0 = -(M[0] - 1); e0 < M[0]; ++e0)
    for (int e1 = -(M[1] - 1); e1 < M[1]; ++e1)
      for (int e2 = -(M[2] - 1); e2 < M[2]; ++e2, ++k) {
        FmaItem it{};
        const int e[3] = {e0, e1, e2};
        it.ncells = 1;
        for (int d = 0; d < 3; ++d) {
          it.e[d] = e[d];
          it.lo[d] = std::max(0, -e[d]);
          it.ext[d] = std::min(M[d], M[d] - e[d]) - it.lo[d];
          it.ncells *= it.ext[d];
        }
        it.elin = (int32_t)k;
        proto[k] = it;
        order[k] = k;
      }
  // an offset's items read the same coefficients: one XCD's L2 (workgroup i runs on
  // XCD i % 8), the heaviest offsets first
  auto work = [&](int64_t e) { return epairs[e] * ((proto[e].ncells + 15) / 16) + 64 * (int64_t)proto[e].ncells; };
  std::stable_sort(order.begin(), order.end(), [&](int64_t x, int64_t y) { return work(x) > work(y); });
  int64_t xload[kXcd] = {};
  for (int64_t e : order) {
    const int x = (int)(std::min_element(xload, xload + kXcd) - xload);
    FmaItem it = proto[e];
    for (int sg = 0; sg < NS; ++sg)
      for (int c = 0; c * 64 < it.ncells; ++c) {
        it.sgroup = sg;
        it.chunk = c;
        col[x].push_back(it);
      }
    xload[x] += work(e);
  }
  size_t nslot = 0;
  for (auto& v : col) nslot = std::max(nslot, v.size());
  FmaItem none{};
  none.chunk = -1;
  items.assign(nslot * kXcd, none);
  for (int x = 0; x < kXcd; ++x)
    for (size_t i = 0; i < col[x].size(); ++i) items[i * kXcd + x] = col[x][i];
  L.nitems = (int64_t)items.size();
  int32_t *d_ptr[2] = {}, *d_list[2] = {};
  uint32_t* d_cnt = nullptr;
  auto drop = [&]() {
    for (int t = 0; t < 2; ++t) { hipFree(d_ptr[t]); hipFree(d_list[t]); }
    hipFree(d_cnt);
  };
  auto release = [&]() {   // a call that fails leaves no part of the plan
    drop();
    hipFree(L.d_items); hipFree(L.d_beg); hipFree(L.d_desc); hipFree(L.d_halo);
    L.d_items = nullptr; L.d_beg = nullptr; L.d_desc = nullptr; L.d_halo = nullptr;
  };
  auto nomem = [&]() {
    release();
    return set_error(ctx, DGV_ERR_NOMEM, "hipMalloc(fmA plan) failed");
  };
  bool ok = hipMalloc(&L.d_beg, sizeof(int64_t) * (ne * D + 1)) == hipSuccess &&
            hipMalloc(&d_cnt, sizeof(uint32_t) * ne * D) == hipSuccess &&
            hipMalloc(&L.d_halo, sizeof(double) * dims.ncext() * (D + 1)) == hipSuccess;
  for (int t = 0; t < 2; ++t)
    ok = ok && hipMalloc(&d_ptr[t], sizeof(int32_t) * (ne + 1)) == hipSuccess &&
         hipMalloc(&d_list[t], sizeof(int32_t) * list[t].size()) == hipSuccess;
  if (!ok) return nomem();
  hipStream_t st = ctx->stream;
  hipError_t e = hipSuccess;
  for (int t = 0; t < 2 && e == hipSuccess; ++t) {
    e = hipMemcpyAsync(d_ptr[t], ptr[t].data(), sizeof(int32_t) * (ne + 1), hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
      e = hipMemcpyAsync(d_list[t], list[t].data(), sizeof(int32_t) * list[t].size(), hipMemcpyHostToDevice, st);
  }
  std::vector<uint32_t> cnt(ne * D);
  std::vector<int64_t> beg(ne * D + 1, 0);
  auto lists = [&](uint2* desc) {
    hipLaunchKernelGGL(k_fma_lists<D>, dim3((unsigned)ne), dim3(256), 0, st, dims, d_ptr[0], d_list[0], d_ptr[1],
                       d_list[1], pb.d_blocks, pb.d_pairs, (uint32_t)pb.npairs, L.d_beg, desc, d_cnt);
    return hipGetLastError();
  };
  if (e == hipSuccess) e = lists(nullptr);
  if (e == hipSuccess) e = hipMemcpyAsync(cnt.data(), d_cnt, sizeof(uint32_t) * ne * D, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e == hipSuccess) {
    constexpr int64_t round = 4 * kFmaRing;
    for (int64_t i = 0; i < ne * D; ++i) beg[i + 1] = beg[i] + (cnt[i] + round - 1) / round * round;
    if (hipMalloc(&L.d_desc, sizeof(uint2) * (beg[ne * D] + kFmaListPad)) != hipSuccess ||
        hipMalloc(&L.d_items, sizeof(FmaItem) * std::max<size_t>(items.size(), 1)) != hipSuccess)
      return nomem();
    // past the last list: pair 0, read ahead and never multiplied
    e = hipMemsetAsync(L.d_desc + beg[ne * D], 0, sizeof(uint2) * kFmaListPad, st);
    if (e == hipSuccess) e = hipMemcpyAsync(L.d_beg, beg.data(), sizeof(int64_t) * beg.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
      e = hipMemcpyAsync(L.d_items, items.data(), sizeof(FmaItem) * items.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = lists(L.d_desc);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
  }
  if (e != hipSuccess) {
    release();
    return set_error(ctx, DGV_ERR_HIP, std::string("fmA plan: ") + hipGetErrorString(e));
  }
  drop();
  return DGV_OK;
}

int prepare_fma_dev(dgv_ctx* ctx, const double* d_fm) {
  if (!ctx->has_a) return set_error(ctx, DGV_ERR_STATE, "no A-array set");
  LinearState& L = ctx->lin;
  const Grid& g = ctx->g;
  const int D = g.D;
  if (D != 8 && D != 27) return set_error(ctx, DGV_ERR_UNSUPPORTED, "PrepareFMA: 2 or 3 nodes per dimension only");
  int rc = L.d_items ? DGV_OK : D == 27 ? build_fma_plan<27>(ctx) : build_fma_plan<8>(ctx);
  if (rc) return rc;
  rc = ensure_vectors(ctx);
  if (rc) return rc;
  const int64_t N = g.N;
  if (!L.d_fma && hipMalloc(&L.d_fma, sizeof(double) * (size_t)N * N) != hipSuccess) {
    L.d_fma = nullptr;
    return set_error(ctx, DGV_ERR_NOMEM, "hipMalloc(fmA, N x N doubles) failed");
  }
  if (d_fm != L.d_vec[0])
    DGV_HIP(ctx, hipMemcpyAsync(L.d_vec[0], d_fm, sizeof(double) * N, hipMemcpyDeviceToDevice, ctx->stream));
  const FmaDims dims{g.Mu, g.Mv, g.Mw};
  hipLaunchKernelGGL(k_fma_halo, dim3(stride_blocks(dims.ncext() * (D + 1), 256)), dim3(256), 0, ctx->stream, dims, D,
                     L.d_vec[0], L.d_halo);
  if (D == 27)
    hipLaunchKernelGGL(k_fma_build<27>, dim3((unsigned)L.nitems), dim3(256), 0, ctx->stream, L.d_items, dims, L.d_beg,
                       L.d_desc, ctx->pb.d_pairs, L.d_halo, ctx->d_gwts, N, L.d_fma);
  else
    hipLaunchKernelGGL(k_fma_build<8>, dim3((unsigned)L.nitems), dim3(256), 0, ctx->stream, L.d_items, dims, L.d_beg,
                       L.d_desc, ctx->pb.d_pairs, L.d_halo, ctx->d_gwts, N, L.d_fma);
  DGV_HIP(ctx, hipGetLastError());
  L.fma_valid = true;
  L.nprepare++;
  return DGV_OK;
}

// The buffer of the chunks' sums, for passes of at least kLinVecMin vectors and of all nvec
// (up to kLinVec, 0.5 GB at 27^3 nodes) where there is memory for them.  It does not grow
// while the stream is captured: more passes over fmA give the same results to the last bit.
constexpr int kLinVecMin = 8;
static int ensure_partials(dgv_ctx* ctx, int nvec) {
  LinearState& L = ctx->lin;
  const int want = std::min(std::max(nvec, kLinVecMin), kLinVec);
  if (L.part_vec >= want) return DGV_OK;
  if (L.d_part) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return DGV_OK;
    DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));   // earlier passes are done with it
  }
  const int64_t N = ctx->g.N;
  // the chunks depend on N alone
  auto alloc = [&](int nv, double** p) {
    return hipMalloc(p, sizeof(double) * (size_t)std::max<int64_t>((int64_t)lin_plan(N, nv).nchunk * nv * N, 1)) == hipSuccess;
  };
  double* p = nullptr;
  int got = want;
  if (!alloc(want, &p)) {
    (void)hipGetLastError();
    if (L.d_part) return DGV_OK;
    got = kLinVecMin;
    if (want == got || !alloc(got, &p)) {
      (void)hipGetLastError();
      return set_error(ctx, DGV_ERR_NOMEM, "hipMalloc(partial products) failed");
    }
  }
  hipFree(L.d_part);
  L.d_part = p;
  L.part_vec = got;
  return DGV_OK;
}

int eval_linear_dev(dgv_ctx* ctx, const double* d_f, int64_t ldf, double* d_fc, int64_t ldq, int nvec) {
  LinearState& L = ctx->lin;
  if (!L.fma_valid) return set_error(ctx, DGV_ERR_STATE, "EvalCollisionLinear: no linearised operator (PrepareFMA)");
  const int64_t N = ctx->g.N;
  if (int rc = ensure_partials(ctx, nvec)) return rc;
  for (int v0 = 0; v0 < nvec; v0 += L.part_vec) {
    const int nv = std::min(L.part_vec, nvec - v0);
    const double* f = d_f + v0 * ldf;
    const LinPlan p = lin_plan(N, nv);
    const unsigned nwg = (unsigned)(((int64_t)p.colblocks * p.nchunk + 7) / 8 * 8 * p.vblocks);
    switch (p.vt) {
      case 0:
        hipLaunchKernelGGL(k_fma_gemv, dim3((unsigned)((N + 255) / 256), p.nchunk), dim3(256), 0, ctx->stream, N,
                           p.chunk, L.d_fma, f, L.d_part);
        break;
#define DGV_LIN_CASE(VT)                                                                                        \
  case VT:                                                                                                      \
    hipLaunchKernelGGL(k_fma_rows<VT>, dim3(nwg), dim3(256), 0, ctx->stream, N, nv, p.colblocks, p.vblocks, p.chunk, \
                       L.d_fma, f, ldf, L.d_part);                                                              \
    break;
      DGV_LIN_CASE(1) DGV_LIN_CASE(2) DGV_LIN_CASE(4)
#undef DGV_LIN_CASE
    }
    hipLaunchKernelGGL(k_fma_sum, dim3(stride_blocks(N * nv, 64)), dim3(64), 0, ctx->stream, N, p.nchunk, nv,
                       L.d_part, d_fc + v0 * ldq, ldq);
  }
  DGV_HIP(ctx, hipGetLastError());
  return DGV_OK;
}

static int l1_weighted(dgv_ctx* ctx, const double* a, const double* b, double* out) {
  LinearState& L = ctx->lin;
  hipLaunchKernelGGL(k_l1_part, dim3(kL1Blocks), dim3(256), 0, ctx->stream, ctx->g.N, a, b, ctx->d_gwts, L.d_vec[4]);
  hipLaunchKernelGGL(k_l1_final, dim3(1), dim3(1), 0, ctx->stream, L.d_vec[4], L.d_vec[4] + kL1Blocks);
  DGV_HIP(ctx, hipGetLastError());
  DGV_HIP(ctx, hipMemcpyAsync(out, L.d_vec[4] + kL1Blocks, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

// CheckSolutionMode_DGV (spat_oper_mod.f90:195-272).  Vectors: d_vec[0] = fm
// (the Maxwellian fmA was built at), d_vec[1] = the new Maxwellian, d_vec[2] =
// Df = f - fm, d_vec[3] = scratch of the spatial operator.
int check_solution_mode(dgv_ctx* ctx, const double* d_f) {
  LinearState& L = ctx->lin;
  int rc = ensure_vectors(ctx);
  if (rc) return rc;
  const Grid& g = ctx->g;
  double mom[5];
  rc = device_moments(ctx, d_f, mom);  // MassCheckRec, line 236
  if (rc) return rc;
  const double dens = mom[0];
  hipLaunchKernelGGL(k_maxwell, dim3(stride_blocks(g.N, 256)), dim3(256), 0, ctx->stream, g.N, mom[4], mom[1], mom[2],
                     mom[3], dens, ctx->d_u, ctx->d_v, ctx->d_w, L.d_vec[1]);
  DGV_HIP(ctx, hipGetLastError());
  double s = 0.0;
  rc = l1_weighted(ctx, d_f, L.d_vec[1], &s);
  if (rc) return rc;
  const double l1 = s / dens;  // line 238
  L.last_l1 = l1;
  L.nchecks++;
  auto refresh_fm = [&]() -> int {  // fm = fMaxwellNew; PrepareFMA_DGV
    DGV_HIP(ctx, hipMemcpyAsync(L.d_vec[0], L.d_vec[1], sizeof(double) * g.N, hipMemcpyDeviceToDevice, ctx->stream));
    return prepare_fma_dev(ctx, L.d_vec[0]);
  };
  auto l1_fm = [&](double* v) -> int {
    double t = 0.0;
    int r = l1_weighted(ctx, L.d_vec[0], L.d_vec[1], &t);
    *v = t / dens;
    return r;
  };
  if (l1 < L.decomp_lev) {
    switch (L.run_mode) {
      case 0:
        if ((rc = refresh_fm())) return rc;
        L.run_mode = l1 < L.linear_lev ? 2 : 1;
        break;
      case 1: {
        double e = 0.0;
        if ((rc = l1_fm(&e))) return rc;
        L.last_l1_fm = e;
        if (e > L.linear_lev / 2.0 && (rc = refresh_fm())) return rc;
        if (l1 < L.linear_lev) L.run_mode = 2;
        break;
      }
      case 2: {
        double e = 0.0;
        if ((rc = l1_fm(&e))) return rc;
        L.last_l1_fm = e;
        if (e > L.linear_lev / 2.0 && (rc = refresh_fm())) return rc;
        if (l1 > L.linear_lev) L.run_mode = 1;
        break;
      }
      default:
        return set_error(ctx, DGV_ERR_STATE, "CheckSolutionMode_DGV: cannot process the value of run_mode");
    }
    hipLaunchKernelGGL(k_sub, dim3(stride_blocks(g.N, 256)), dim3(256), 0, ctx->stream, g.N, d_f, L.d_vec[0],
                       L.d_vec[2]);  // Df = f - fm
    DGV_HIP(ctx, hipGetLastError());
  } else {
    L.run_mode = 0;
  }
  return DGV_OK;
}

// SpatialOperSH_DGV (spat_oper_mod.f90:28-68): the regime check (when switching
// is enabled), then run_mode 0: Q(f); 1: L(Df) + Q(Df); 2: L(Df); times scale.
int spatial_oper_device(dgv_ctx* ctx, const double* d_f, double* d_out, double scale) {
  LinearState& L = ctx->lin;
  if (!(L.decomp_lev > 0.0)) {
    L.run_mode = 0;
    return eval_q_dev(ctx, d_f, d_out, scale);
  }
  int rc = check_solution_mode(ctx, d_f);
  if (rc) return rc;
  const int64_t N = ctx->g.N;
  const unsigned nblk = stride_blocks(N, 256);
  switch (L.run_mode) {
    case 0:
      return eval_q_dev(ctx, d_f, d_out, scale);
    case 1: {
      const int save = ctx->project;
      ctx->project = 0;
      rc = eval_linear_dev(ctx, L.d_vec[2], N, L.d_vec[3], N, 1);
      if (!rc) rc = eval_q_dev(ctx, L.d_vec[2], d_out, 1.0);
      ctx->project = save;
      if (rc) return rc;
      hipLaunchKernelGGL(k_sum_scale, dim3(nblk), dim3(256), 0, ctx->stream, N, d_out, L.d_vec[3], scale, d_out);
      break;
    }
    case 2:
      rc = eval_linear_dev(ctx, L.d_vec[2], N, d_out, N, 1);
      if (rc) return rc;
      hipLaunchKernelGGL(k_sum_scale, dim3(nblk), dim3(256), 0, ctx->stream, N, d_out, (const double*)nullptr, scale,
                         d_out);
      break;
    default:
      return set_error(ctx, DGV_ERR_STATE, "SpatialOperSH_DGV: cannot process the value of run_mode");
  }
  DGV_HIP(ctx, hipGetLastError());
  if (ctx->project) return device_project(ctx, d_out);
  return DGV_OK;
}

}  // namespace dgv

using namespace dgv;

#define LIN_CHECK(ctx, n)                                                            \
  do {                                                                               \
    if (!(ctx)) return DGV_ERR_ARG;                                                  \
    if ((n) != (ctx)->g.N) return set_error((ctx), DGV_ERR_ARG, "array size mismatch"); \
  } while (0)

extern "C" {

int dgv_prepare_fma_dev(dgv_ctx* ctx, const double* d_fm, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!d_fm) return set_error(ctx, DGV_ERR_ARG, "null array");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  int rc = ensure_vectors(ctx);
  if (rc) return rc;
  return prepare_fma_dev(ctx, d_fm);
}

int dgv_prepare_fma(dgv_ctx* ctx, const double* fm, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!fm) return set_error(ctx, DGV_ERR_ARG, "null array");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  int rc = ensure_vectors(ctx);
  if (rc) return rc;
  DGV_HIP(ctx, hipMemcpyAsync(ctx->lin.d_vec[0], fm, sizeof(double) * n, hipMemcpyHostToDevice, ctx->stream));
  rc = prepare_fma_dev(ctx, ctx->lin.d_vec[0]);
  if (rc) return rc;
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

int dgv_eval_linear_dev(dgv_ctx* ctx, const double* d_f, int64_t ldf, double* d_fc, int64_t ldq, int64_t n,
                        int32_t nvec) {
  LIN_CHECK(ctx, n);
  if (!d_f || !d_fc || nvec < 1 || ldf < n || ldq < n) return set_error(ctx, DGV_ERR_ARG, "bad arguments");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  return eval_linear_dev(ctx, d_f, ldf, d_fc, ldq, nvec);
}

int dgv_eval_linear(dgv_ctx* ctx, const double* f, double* fc, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!f || !fc) return set_error(ctx, DGV_ERR_ARG, "null array");
  const size_t nb = sizeof(double) * n;
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMemcpyAsync(ctx->d_f, f, nb, hipMemcpyHostToDevice, ctx->stream));
  int rc = eval_linear_dev(ctx, ctx->d_f, n, ctx->d_q, n, 1);
  if (rc) return rc;
  DGV_HIP(ctx, hipMemcpyAsync(fc, ctx->d_q, nb, hipMemcpyDeviceToHost, ctx->stream));
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

int dgv_ctx_get_fma(dgv_ctx* ctx, double* fmA, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!fmA) return set_error(ctx, DGV_ERR_ARG, "null array");
  if (!ctx->lin.fma_valid) return set_error(ctx, DGV_ERR_STATE, "no linearised operator (PrepareFMA)");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  // device rows r (contiguous in i) -> the reference's column-major fmA(r, i)
  std::vector<double> rows;
  const int64_t chunk = std::max<int64_t>(1, std::min<int64_t>(n, (int64_t)(64 << 20) / (8 * n)));
  rows.resize((size_t)chunk * n);
  for (int64_t r0 = 0; r0 < n; r0 += chunk) {
    const int64_t nr = std::min(chunk, n - r0);
    DGV_HIP(ctx, hipMemcpyAsync(rows.data(), ctx->lin.d_fma + r0 * n, sizeof(double) * nr * n, hipMemcpyDeviceToHost,
                                ctx->stream));
    DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int64_t r = 0; r < nr; ++r)
      for (int64_t i = 0; i < n; ++i) fmA[(r0 + r) + n * i] = rows[r * n + i];
  }
  return DGV_OK;
}

int dgv_ctx_set_regime(dgv_ctx* ctx, int32_t run_mode, double decomp_lev, double linear_lev) {
  if (!ctx) return DGV_ERR_ARG;
  if (run_mode < 0 || run_mode > 2) return set_error(ctx, DGV_ERR_ARG, "run_mode must be 0, 1 or 2");
  // spat_oper_mod.f90:331-334: the decomposition threshold must lie above the
  // linearisation threshold (decomp_lev = 0 switches the regime check off)
  if (decomp_lev > 0 && decomp_lev <= linear_lev)
    return set_error(ctx, DGV_ERR_ARG,
                     "Decomposition treshold is lower than linearization treshhold (decomp_lev <= linear_lev)");
  if ((run_mode != 0) && !ctx->lin.fma_valid)
    return set_error(ctx, DGV_ERR_STATE, "run_mode 1 or 2 needs a linearised operator (PrepareFMA)");
  ctx->lin.run_mode = run_mode;
  ctx->lin.decomp_lev = decomp_lev;
  ctx->lin.linear_lev = linear_lev;
  if (ctx->rk_graph) { hipGraphExecDestroy(ctx->rk_graph); ctx->rk_graph = nullptr; }
  return DGV_OK;
}

int dgv_ctx_get_regime(dgv_ctx* ctx, int32_t* run_mode, double* l1_err, double* l1_err_fm, int64_t counts[2]) {
  if (!ctx) return DGV_ERR_ARG;
  if (run_mode) *run_mode = ctx->lin.run_mode;
  if (l1_err) *l1_err = ctx->lin.last_l1;
  if (l1_err_fm) *l1_err_fm = ctx->lin.last_l1_fm;
  if (counts) { counts[0] = ctx->lin.nchecks; counts[1] = ctx->lin.nprepare; }
  return DGV_OK;
}

// The Iphi integrals are the plain sums over the records: the conservation
// projection that the context may apply to every Q is held off while they run.
struct ProjectionOff {
  dgv_ctx* ctx;
  int save;
  explicit ProjectionOff(dgv_ctx* c) : ctx(c), save(c->project) { c->project = 0; }
  ~ProjectionOff() { ctx->project = save; }
};

// IphiDGV (dgvtools_mod.f90:847-877): for every node i, one basis function per
// node, Iphi(i) = 2 sum over its records of A f(xi) f(xi1) / w_i, times coef.
// On the shifted A-array these are the evaluator's Q of f, scaled.
int dgv_iphi(dgv_ctx* ctx, const double* f, double* iphi, int64_t n, double coef) {
  LIN_CHECK(ctx, n);
  if (!f || !iphi) return set_error(ctx, DGV_ERR_ARG, "null array");
  const size_t nb = sizeof(double) * n;
  const ProjectionOff plain(ctx);
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMemcpyAsync(ctx->d_f, f, nb, hipMemcpyHostToDevice, ctx->stream));
  int rc = eval_q_dev(ctx, ctx->d_f, ctx->d_q, coef);
  if (rc) return rc;
  DGV_HIP(ctx, hipMemcpyAsync(iphi, ctx->d_q, nb, hipMemcpyDeviceToHost, ctx->stream));
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

// IphiDGV_decomp (dgvtools_mod.f90:896-927): the same integrals with f split at
// its local Maxwellian fM (MassCheckRec, maxwelveldist; lines 912-914): per record
// A (fM(xi) Df(xi1) + Df(xi) fM(xi1) + Df(xi) Df(xi1)), Df = f - fM, i.e. the
// evaluator's mixed term of (Df, fM) plus its Q of Df, times coef.
int dgv_iphi_decomp(dgv_ctx* ctx, const double* f, double* iphi, int64_t n, double coef) {
  LIN_CHECK(ctx, n);
  if (!f || !iphi) return set_error(ctx, DGV_ERR_ARG, "null array");
  const size_t nb = sizeof(double) * n;
  const Grid& g = ctx->g;
  const ProjectionOff plain(ctx);
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMemcpyAsync(ctx->d_f, f, nb, hipMemcpyHostToDevice, ctx->stream));
  double mom[5];
  int rc = device_moments(ctx, ctx->d_f, mom);
  if (rc) return rc;
  double* fM = ctx->d_tmp[5];
  double* df = ctx->d_tmp[0];
  double* qd = ctx->d_tmp[1];
  const unsigned nblk = stride_blocks(g.N, 256);
  hipLaunchKernelGGL(k_maxwell, dim3(nblk), dim3(256), 0, ctx->stream, g.N, mom[4], mom[1], mom[2], mom[3], mom[0],
                     ctx->d_u, ctx->d_v, ctx->d_w, fM);
  hipLaunchKernelGGL(k_sub, dim3(nblk), dim3(256), 0, ctx->stream, g.N, ctx->d_f, fM, df);
  DGV_HIP(ctx, hipGetLastError());
  if ((rc = eval_mixed_dev(ctx, df, fM, ctx->d_q))) return rc;
  if ((rc = eval_q_dev(ctx, df, qd, 1.0))) return rc;
  hipLaunchKernelGGL(k_sum_scale, dim3(nblk), dim3(256), 0, ctx->stream, g.N, ctx->d_q, qd, coef, ctx->d_q);
  DGV_HIP(ctx, hipGetLastError());
  DGV_HIP(ctx, hipMemcpyAsync(iphi, ctx->d_q, nb, hipMemcpyDeviceToHost, ctx->stream));
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

int dgv_check_solution_mode(dgv_ctx* ctx, const double* f, double* df, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!f) return set_error(ctx, DGV_ERR_ARG, "null array");
  const size_t nb = sizeof(double) * n;
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMemcpyAsync(ctx->d_f, f, nb, hipMemcpyHostToDevice, ctx->stream));
  int rc = check_solution_mode(ctx, ctx->d_f);
  if (rc) return rc;
  if (df) {
    if (ctx->lin.run_mode != 0)
      DGV_HIP(ctx, hipMemcpyAsync(df, ctx->lin.d_vec[2], nb, hipMemcpyDeviceToHost, ctx->stream));
    else
      std::memset(df, 0, nb);  // Df is left unset by the reference in run_mode 0
  }
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

int dgv_ctx_get_fm(dgv_ctx* ctx, double* fm, int64_t n) {
  LIN_CHECK(ctx, n);
  if (!fm) return set_error(ctx, DGV_ERR_ARG, "null array");
  if (!ctx->lin.d_vec[0]) return set_error(ctx, DGV_ERR_STATE, "no Maxwellian set");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMemcpyAsync(fm, ctx->lin.d_vec[0], sizeof(double) * n, hipMemcpyDeviceToHost, ctx->stream));
  DGV_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return DGV_OK;
}

}  // extern "C"
