// dgv_quad.h -- the merged ("box") layout of the A-array and its evaluator core.
//
// Two nodes xi, xi1 are opposite corners of a box whose corners are all grid
// nodes: in each dimension one takes the lower coordinate and the other the
// upper.  The box's four diagonals are node pairs with one midpoint and one
// distance, hence one collision sphere, and with the same product of node
// weights.  The gain part of A depends on nothing else, and the loss part
// touches only pairs with a node in the canonical cell, so the D coefficients of
// a box's diagonals agree except there.  All four pairs also stay on the grid
// for the same output cells.  The evaluator's sum therefore needs one
// coefficient row per box,
//   Q[c, l] += T[l] (f f' + f f' + f f' + f f')   over the diagonals,
// a quarter of the matrix-core work and of the coefficient bytes.
//
// A "quad" is one coefficient row with up to four node pairs.  Pairs are merged
// only where every coefficient agrees to kQuadTol, so any A-array can be laid
// out this way; where few pairs merge the pair-block kernels stay in use.
//
//   quad block = the quads whose corners lie in the cells cc + (a_d or b_d), a <= b
//                in every dimension: up to eight cells, "slot" k = cell with b_d
//                where bit d of k is set (a dimension with a_d == b_d keeps bit 0);
//   step       = four quads, the K extent of v_mfma_f64_16x16x4_f64: D x 4
//                coefficients (row l holds the four quads), then per quad eight
//                16-bit LDS byte offsets, the rows of x0 y0 x1 y1 x2 y2 x3 y3 (the
//                zero row for both nodes of an absent pair).
#pragma once
#include <type_traits>

#include "dgv_internal.h"

namespace dgv {

constexpr int kQuadCols = 32;        // columns (output cells or instances) per workgroup
// doubles per staged row: a multiple of the 64 banks, so that the 16-byte reads of
// a step's four rows (which the LDS serves in mixed groups of 16 lanes) never meet
constexpr int kQuadRow = kQuadCols;
constexpr int kQuadRing = 4;         // steps of operand loads in flight per wave
constexpr int kQuadMaxWaves = 8;
// zero steps past the end: a wave reads up to kQuadRing of its steps past a block's start
constexpr int kQuadPadSteps = kQuadMaxWaves * (kQuadRing + 1);

template <int D>
constexpr uint32_t quad_step_bytes() { return D * 32 + 64; }
template <int D>
constexpr int quad_rows() { return 8 * D + 1; }
static_assert(8 * 27 * kQuadRow * 8 < 65536, "row offsets fit 16 bits");

typedef double qd4 __attribute__((ext_vector_type(4)));
typedef double qd2 __attribute__((ext_vector_type(2)));
typedef uint32_t qu4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double qel(const qd2& v, int i) { return v[i]; }
__device__ __forceinline__ double qel(double v, int) { return v; }

// One workgroup's walk over quad blocks for 16 CT columns.  The waves share the
// staged f and split a block's steps between them (wave w takes steps w, w + NW,
// ...), so every coefficient is loaded by one wave only and feeds RT x CT
// products; the waves' sums are added in LDS at the end of the item.
//   header(i)  -> QuadBlk of the walk's i-th block, i in [0, n)
//   fetch(B)   issues the loads of f (and of gm with MIX) for a block's slots
//   store(B)   writes them to LDS
// A block's f is on its way while the block before it is computed, and a ring slot
// whose last step of a block is done loads the next block's step of its number, so
// at a block's start only the LDS writes and two barriers are exposed.
// Bound by the LDS reads of the eight corner values (8 x 1 KiB per wave and step
// against 256 matrix-core cycles per SIMD) and the matrix cores together.
template <int D, bool MIX, int NW, int CT, class Header, class Fetch, class Store>
__device__ __forceinline__ void quad_walk(int n, QuadBlk cur, int s0, int s1, const double* __restrict__ steps,
                                          double* lf, double* lg, Header&& header, Fetch&& fetch, Store&& store,
                                          qd4 (&acc)[(D + 15) / 16][CT]) {
  constexpr int RT = (D + 15) / 16;
  constexpr int R = kQuadRing;
  using OpT = typename std::conditional<CT == 2, qd2, double>::type;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kk = lane >> 4, jj = lane & 15;
  uint32_t aoff[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) aoff[rt] = (uint32_t)((min(16 * rt + jj, D - 1) * 4 + kk) * 8);
  const uint32_t coff = (uint32_t)(D * 32 + kk * 16);
  const char* fl = reinterpret_cast<const char*>(lf + CT * jj);
  const char* gl = reinterpret_cast<const char*>(lg + (MIX ? CT * jj : 0));
  double ab[R][RT];
  qu4 cd[R];
  // this wave's first step of a block (an item of one block may hold a part of its steps)
  auto base = [&](const QuadBlk& B) {
    return reinterpret_cast<const char*>(steps) + (B.sbeg + s0 + wave) * (int64_t)quad_step_bytes<D>();
  };
  auto load = [&](int u, const char* p, int i) {
    const __amdgpu_buffer_rsrc_t P = ring_rsrc(p);
    const uint32_t s = (uint32_t)(NW * i) * quad_step_bytes<D>();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) ab[u][rt] = ring_f64(P, aoff[rt], s);
    cd[u] = __builtin_amdgcn_raw_buffer_load_b128(P, coff, s, 0);
  };
  OpT x[8], y[MIX ? 8 : 1];
  double bcur[CT];
  auto issue = [&](const qu4& c) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t o = (k & 1) ? c[k >> 1] >> 16 : c[k >> 1] & 0xffffu;
      x[k] = *reinterpret_cast<const OpT*>(fl + o);
      if constexpr (MIX) y[k] = *reinterpret_cast<const OpT*>(gl + o);
    }
  };
  auto finish = [&]() {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      double s;
      if constexpr (MIX) {
        s = qel(y[0], ct) * qel(x[1], ct);
        s = __fma_rn(qel(x[0], ct), qel(y[1], ct), s);
#pragma unroll
        for (int k = 2; k < 8; k += 2) {
          s = __fma_rn(qel(y[k], ct), qel(x[k + 1], ct), s);
          s = __fma_rn(qel(x[k], ct), qel(y[k + 1], ct), s);
        }
      } else {
        s = qel(x[0], ct) * qel(x[1], ct);
#pragma unroll
        for (int k = 2; k < 8; k += 2) s = __fma_rn(qel(x[k], ct), qel(x[k + 1], ct), s);
      }
      bcur[ct] = s;
    }
  };
  auto products = [&](int u) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(ab[u][rt], bcur[ct], acc[rt][ct], 0, 0, 0);
  };
  const char* pc = base(cur);
#pragma unroll
  for (int u = 0; u < R; ++u) load(u, pc, u);
  fetch(cur);
  QuadBlk nxt = header(min(1, n - 1));
  for (int bi = 0; bi < n; ++bi) {
    __syncthreads();   // the previous block's LDS reads are done
    store(cur);
    __syncthreads();
    const QuadBlk nn = header(min(bi + 2, n - 1));
    const int nw = (min(s1, cur.nst) - s0 - wave + NW - 1) / NW;   // this wave's steps
    const char* pn = base(nxt);
    issue(cd[0]);
    finish();
    __builtin_amdgcn_sched_barrier(0);   // the ring's wait ahead of the next block's loads
    if (bi + 1 < n) fetch(nxt);
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
    for (; i + 2 * R <= nw; i += R) {   // rounds whose loads all lie in the block
#pragma unroll
      for (int u = 0; u < R; ++u) {
        issue(cd[(u + 1) % R]);
        // the next step's LDS reads stay ahead of this step's products and the
        // wait for them behind (as in the pair-block kernel)
        __builtin_amdgcn_sched_barrier(0);
        products(u);
        __builtin_amdgcn_sched_barrier(0);
        load(u, pc, i + u + R);
        finish();
      }
    }
    for (bool first = i == 0; i < nw || first; i += R, first = false) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        const bool own = i + u < nw;
        if (own) {
          issue(cd[(u + 1) % R]);
          __builtin_amdgcn_sched_barrier(0);
          products(u);
          __builtin_amdgcn_sched_barrier(0);
        }
        const bool in = i + u + R < nw;
        load(u, in ? pc : pn, in ? i + u + R : u);
        if (own) finish();
      }
    }
    cur = nxt;
    nxt = nn;
    pc = pn;
  }
}

// The waves' sums of a walk, added in wave order: element (l, col) to
// out[col * D + l] for col < ncols, `more`: on top of what an earlier walk left there.
// `red` overlays the staged rows (the zero row behind them stays).
template <int D, int NW, int CT>
__device__ __forceinline__ void quad_flush(double* red, const qd4 (&acc)[(D + 15) / 16][CT], int ncols, double* out,
                                           bool more = false) {
  constexpr int RT = (D + 15) / 16;
  constexpr int S = NW <= 4 ? kQuadCols + 2 : kQuadCols;   // padded where there is room: the column sums read across rows
  static_assert(NW * D * S <= 8 * D * kQuadRow, "the sums fit the staged rows");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kk = lane >> 4, jj = lane & 15;
  __syncthreads();   // the last block's LDS reads are done
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int l = 16 * rt + 4 * e + kk;   // FP64 output layout: row 4 e + lane / 16
      if (l < D) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) red[(wave * D + l) * S + CT * jj + ct] = acc[rt][ct][e];
      }
    }
  __syncthreads();
  for (int i = threadIdx.x; i < ncols * D; i += 64 * NW) {
    const int col = i / D, l = i - col * D;
    double s = red[l * S + col];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[(w * D + l) * S + col];
    out[i] = more ? out[i] + s : s;
  }
}

}  // namespace dgv
