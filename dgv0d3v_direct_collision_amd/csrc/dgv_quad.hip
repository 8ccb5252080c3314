// dgv_quad.hip -- building and evaluating the merged layout of the A-array
// (dgv_quad.h) for one VDF.
#include <algorithm>
#include <array>
#include <climits>
#include <cmath>
#include <cstring>
#include <map>
#include <vector>

#include "dgv_quad.h"

namespace dgv {

// Coefficients of a box's diagonals come from one sphere integral and from
// products of the same node weights in different orders: at most a dozen
// roundings apart (2^-49); the merged row is their mean, which moves Q by 2e-18 to 3e-17
// (relative L2, in extended precision, 2- and 3-node grids of up to 960 nodes).
constexpr double kQuadTol = 3.6e-15;   // 2^-48
// The merged evaluator is used when it leaves at most this share of the pairs as
// quads.  One Q at 27^3 nodes: 4.7 ms with the generated A-array (0.29 of the
// pairs), 12.7 ms with no pair merged, 12.3 ms by the pair-block kernel, whose
// copy of the coefficients is there anyway; at 15^3 nodes 94, 237 and 250 us.
constexpr double kQuadShare = 0.9;

struct QuadSrc {
  int32_t blk[8];   // pair block whose xi cell takes b_d where bit d is set (or -1)
};

// The pairs of one box.  Candidate (p, q) of a quad block: the local indices of
// the box's low and high corner.  fn(entry, pair index, x offset, y offset), entry =
// 2 * diagonal + orientation, for every record present.
template <int D>
struct QuadDims {
  int su, sv, sw;
};

__device__ __forceinline__ uint32_t quad_row_off(int D, int slot, int local) {
  return (uint32_t)((slot * D + local) * kQuadRow * 8);
}

template <int D, class Fn>
__device__ __forceinline__ void quad_entries(const QuadDims<D>& g, int p, int q, int same, const QuadSrc& src,
                                             const BlockHdr* __restrict__ blocks, const int16_t* __restrict__ pidx,
                                             Fn&& fn) {
  const int P[3] = {p / (g.sv * g.sw), (p / g.sw) % g.sv, p % g.sw};
  const int Q[3] = {q / (g.sv * g.sw), (q / g.sw) % g.sv, q % g.sw};
  int nd = 0;   // dimensions in which the corners differ
  for (int d = 0; d < 3; ++d) {
    const bool cell_same = (same >> d) & 1;
    if (cell_same && P[d] > Q[d]) return;   // the box is (Q, P)'s
    if (!cell_same || P[d] != Q[d]) nd |= 1 << d;
  }
  const int flips = nd & (nd - 1);   // the first such dimension fixes which node is called x
  int diag = 0;
  for (int z = 0; z < 8; ++z) {
    if (z & ~flips) continue;
    int X[3], Y[3];
    for (int d = 0; d < 3; ++d) {
      X[d] = (z >> d) & 1 ? Q[d] : P[d];
      Y[d] = (z >> d) & 1 ? P[d] : Q[d];
    }
    const int lx = (X[0] * g.sv + X[1]) * g.sw + X[2], ly = (Y[0] * g.sv + Y[1]) * g.sw + Y[2];
    const int cx = z & ~same, cy = ~z & ~same & 7;
    const uint32_t ox = quad_row_off(D, cx, lx), oy = quad_row_off(D, cy, ly);
    for (int o = 0; o < (nd ? 2 : 1); ++o) {   // the record may be stored as (x, y) or (y, x)
      const int b = src.blk[o ? cy : cx];
      if (b < 0) continue;
      const int j = pidx[(int64_t)b * D * D + (o ? ly * D + lx : lx * D + ly)];
      if (j >= 0) fn(2 * diag + o, blocks[b].pbeg + j, ox, oy);
    }
    ++diag;
  }
}

// exclusive scan of one value per thread over 256 threads; returns the total
__device__ __forceinline__ int block_scan(int v, int& before) {
  __shared__ int s[256];
  const int t = threadIdx.x;
  s[t] = v;
  __syncthreads();
  for (int h = 1; h < 256; h <<= 1) {
    const int x = t >= h ? s[t - h] : 0;
    __syncthreads();
    s[t] += x;
    __syncthreads();
  }
  before = s[t] - v;
  const int total = s[255];
  __syncthreads();
  return total;
}

// One workgroup per quad block in turn: which records of each candidate box merge.
// assign[(block) D D + c]: 4 bits per entry, 0 = absent, else 1 + its cluster.
template <int D>
__global__ __launch_bounds__(256) void k_quad_assign(QuadDims<D> g, int64_t nq, const QuadBlk* __restrict__ qb,
                                                     const QuadSrc* __restrict__ src,
                                                     const BlockHdr* __restrict__ blocks,
                                                     const int16_t* __restrict__ pidx,
                                                     const double* __restrict__ pairs, double tol,
                                                     uint32_t* __restrict__ assign, int32_t* __restrict__ count) {
  for (int64_t b = blockIdx.x; b < nq; b += gridDim.x) {
    const QuadSrc S = src[b];
    const int same = qb[b].same;
    int mine = 0;
    for (int c = threadIdx.x; c < D * D; c += 256) {
      uint32_t a = 0;
      int ncl = 0;
      int64_t lead[8];
      int size[8];
      quad_entries<D>(g, c / D, c % D, same, S, blocks, pidx, [&](int e, int64_t pair, uint32_t, uint32_t) {
        const double* T = pairs + pair * (D + 1);
        int k = 0;
        for (; k < ncl; ++k) {
          if (size[k] == 4) continue;
          const double* L = pairs + lead[k] * (D + 1);
          bool eq = true;
          for (int l = 0; l < D && eq; ++l) {
            const double x = T[l], y = L[l];
            eq = fabs(x - y) <= tol * fmax(fabs(x), fabs(y));   // false for a NaN: never merged
          }
          if (eq) break;
        }
        if (k == ncl) {
          lead[ncl] = pair;
          size[ncl++] = 0;
        }
        ++size[k];
        a |= (uint32_t)(k + 1) << (4 * e);
      });
      assign[b * D * D + c] = a;
      mine += ncl;
    }
    int before;
    const int total = block_scan(mine, before);
    if (threadIdx.x == 0) count[b] = total;
  }
}

// One workgroup per quad block in turn: the steps, 256 candidates at a time.  Each thread
// lists its candidate's quads (their records, and the codes in place), then the
// workgroup writes the coefficients, one element of a row per thread (a thread per
// quad took 1.6 ms at 15^3 nodes, strided writes; this way 0.42 ms).
template <int D>
__global__ __launch_bounds__(256) void k_quad_write(QuadDims<D> g, int64_t nq, const QuadBlk* __restrict__ qb,
                                                    const QuadSrc* __restrict__ src,
                                                    const BlockHdr* __restrict__ blocks,
                                                    const int16_t* __restrict__ pidx,
                                                    const double* __restrict__ pairs,
                                                    const uint32_t* __restrict__ assign, char* __restrict__ steps) {
  constexpr uint32_t kNone = 0xffffffffu;
  __shared__ uint32_t rec[256 * 8][4];   // the records of the quads of 256 candidates
  for (int64_t b = blockIdx.x; b < nq; b += gridDim.x) {
    const QuadSrc S = src[b];
    const int same = qb[b].same;
    const uint32_t* A = assign + b * D * D;
    char* base = steps + qb[b].sbeg * (int64_t)quad_step_bytes<D>();
    const uint32_t zero = quad_row_off(D, 8, 0);
    auto slot_T = [&](int quad) { return reinterpret_cast<double*>(base + (int64_t)(quad >> 2) * quad_step_bytes<D>()) + (quad & 3); };
    auto slot_code = [&](int quad) {
      return reinterpret_cast<uint16_t*>(base + (int64_t)(quad >> 2) * quad_step_bytes<D>() + D * 32 + (quad & 3) * 16);
    };
    int done = 0;   // quads written before this round
    for (int c0 = 0; c0 < D * D; c0 += 256) {
      const int c = c0 + (int)threadIdx.x;
      const uint32_t a = c < D * D ? A[c] : 0;
      int n = 0;
      for (int e = 0; e < 8; ++e) n = max(n, (int)((a >> (4 * e)) & 15));
      int at;
      const int total = block_scan(n, at);
      for (int k = 1; k <= n; ++k, ++at) {
        uint16_t* code = slot_code(done + at);
        int m = 0;
        quad_entries<D>(g, c / D, c % D, same, S, blocks, pidx, [&](int e, int64_t pair, uint32_t ox, uint32_t oy) {
          if ((int)((a >> (4 * e)) & 15) != k) return;
          rec[at][m] = (uint32_t)pair;
          code[2 * m] = (uint16_t)ox;
          code[2 * m + 1] = (uint16_t)oy;
          ++m;
        });
        for (; m < 4; ++m) {
          rec[at][m] = kNone;
          code[2 * m] = code[2 * m + 1] = (uint16_t)zero;
        }
      }
      __syncthreads();
      for (int i = threadIdx.x; i < total * D; i += 256) {
        const int k = i / D, l = i - k * D;
        double t = pairs[(int64_t)rec[k][0] * (D + 1) + l];
        int m = 1;
        for (; m < 4 && rec[k][m] != kNone; ++m) t += pairs[(int64_t)rec[k][m] * (D + 1) + l];
        if (m > 1) t = m == 2 ? t * 0.5 : m == 4 ? t * 0.25 : t / 3.0;
        slot_T(done + k)[4 * l] = t;
      }
      done += total;
      __syncthreads();
    }
    // the last step's missing quads: zero rows
    for (int k = done + threadIdx.x; k < ((done + 3) & ~3); k += 256) {
      double* T = slot_T(k);
      uint16_t* code = slot_code(k);
      for (int l = 0; l < D; ++l) T[4 * l] = 0.0;
      for (int m = 0; m < 8; ++m) code[m] = (uint16_t)zero;
    }
  }
}

void free_quads(dgv_ctx* ctx) {
  if (ctx->plan.quad) free_plan(ctx);   // its items walk these blocks
  QuadLayout& Q = ctx->quad;
  hipFree(Q.d_steps); hipFree(Q.d_blocks);
  Q = QuadLayout();
}

int launch_pair_index(dgv_ctx* ctx, int16_t* d_idx);   // dgv_linear.hip

template <int D>
static int build_quads_t(dgv_ctx* ctx) {
  const Grid& g = ctx->g;
  const PairBlock& pb = ctx->pb;
  QuadLayout& Q = ctx->quad;
  hipStream_t st = ctx->stream;
  const int64_t nb = (int64_t)pb.blocks.size();
  if (pb.npairs >= (int64_t)UINT32_MAX) return DGV_OK;   // k_quad_write numbers the pairs with 32 bits
  // pair blocks by their corner cells
  struct Key { int32_t lo, hi; uint8_t bits; int32_t blk; };
  std::vector<Key> keys(nb);
  auto code = [](const int v[3]) { return ((v[0] + 512) << 20) | ((v[1] + 512) << 10) | (v[2] + 512); };
  for (int64_t k = 0; k < nb; ++k) {
    const BlockHdr& B = pb.blocks[k];
    int lo[3], hi[3], bits = 0;
    for (int d = 0; d < 3; ++d) {
      lo[d] = std::min(B.a[d], B.b[d]);
      hi[d] = std::max(B.a[d], B.b[d]);
      if (B.a[d] > B.b[d]) bits |= 1 << d;
    }
    keys[k] = {code(lo), code(hi), (uint8_t)bits, (int32_t)k};
  }
  std::sort(keys.begin(), keys.end(), [](const Key& x, const Key& y) {
    return x.lo != y.lo ? x.lo < y.lo : x.hi != y.hi ? x.hi < y.hi : x.blk < y.blk;
  });
  std::vector<QuadBlk> qb;
  std::vector<QuadSrc> src;
  std::map<std::array<int, 6>, std::vector<int32_t>> groups;
  const int M[3] = {g.Mu, g.Mv, g.Mw};
  for (int64_t i = 0; i < nb;) {
    int64_t j = i;
    QuadSrc s;
    std::fill(s.blk, s.blk + 8, -1);
    QuadBlk q;
    std::memset(&q, 0, sizeof(q));
    for (; j < nb && keys[j].lo == keys[i].lo && keys[j].hi == keys[i].hi; ++j) {
      s.blk[keys[j].bits] = keys[j].blk;
      q.npairs += pb.blocks[keys[j].blk].npairs;
    }
    std::array<int, 6> box;
    const BlockHdr& B = pb.blocks[keys[i].blk];
    for (int d = 0; d < 3; ++d) {
      q.a[d] = std::min(B.a[d], B.b[d]);
      q.b[d] = std::max(B.a[d], B.b[d]);
      if (q.a[d] == q.b[d]) q.same |= 1 << d;
      box[d] = std::max(0, -(int)q.a[d]);
      box[3 + d] = std::min(M[d], M[d] - q.b[d]) - box[d];
    }
    if (q.npairs > 0 && box[3] > 0 && box[4] > 0 && box[5] > 0) {
      groups[box].push_back((int32_t)qb.size());
      qb.push_back(q);
      src.push_back(s);
    }
    i = j;
  }
  if (qb.empty()) return DGV_OK;
  // group order; inside a group the blocks keep their (low, high) corner order
  std::vector<QuadSrc> src2;
  for (auto& kv : groups) {
    Group G;
    for (int d = 0; d < 3; ++d) { G.lo[d] = kv.first[d]; G.ext[d] = kv.first[3 + d]; }
    G.ncells = G.ext[0] * G.ext[1] * G.ext[2];
    G.bbeg = (int32_t)Q.blocks.size();
    G.npairs = 0;
    for (int32_t b : kv.second) { Q.blocks.push_back(qb[b]); src2.push_back(src[b]); G.npairs += qb[b].npairs; }
    G.bend = (int32_t)Q.blocks.size();
    Q.groups.push_back(G);
  }
  const int64_t nq = (int64_t)Q.blocks.size();
  int16_t* d_pidx = nullptr;
  QuadSrc* d_src = nullptr;
  uint32_t* d_assign = nullptr;
  int32_t* d_count = nullptr;
  auto drop = [&]() { hipFree(d_pidx); hipFree(d_src); hipFree(d_assign); hipFree(d_count); };
  auto without = [&]() {   // no memory for the merged copy: the pair-block kernels serve
    drop();
    free_quads(ctx);
    (void)hipGetLastError();
    return DGV_OK;
  };
  if (hipMalloc(&d_pidx, sizeof(int16_t) * nb * D * D) || hipMalloc(&d_src, sizeof(QuadSrc) * nq) ||
      hipMalloc(&d_assign, sizeof(uint32_t) * nq * D * D) || hipMalloc(&d_count, sizeof(int32_t) * nq) ||
      hipMalloc(&Q.d_blocks, sizeof(QuadBlk) * nq))
    return without();
  const QuadDims<D> dims{g.su, g.sv, g.sw};
  std::vector<int32_t> count(nq);
  hipError_t e = hipMemcpyAsync(d_src, src2.data(), sizeof(QuadSrc) * nq, hipMemcpyHostToDevice, st);
  if (e == hipSuccess)
    e = hipMemcpyAsync(Q.d_blocks, Q.blocks.data(), sizeof(QuadBlk) * nq, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    if (int rc = launch_pair_index(ctx, d_pidx)) {
      drop();
      free_quads(ctx);
      return rc;
    }
    hipLaunchKernelGGL(k_quad_assign<D>, dim3(loop_blocks(nq)), dim3(256), 0, st, dims, nq, Q.d_blocks, d_src, pb.d_blocks,
                       d_pidx, pb.d_pairs, kQuadTol, d_assign, d_count);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(count.data(), d_count, sizeof(int32_t) * nq, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) {
    drop();
    free_quads(ctx);
    return set_error(ctx, DGV_ERR_HIP, std::string("merged layout: ") + hipGetErrorString(e));
  }
  for (int64_t k = 0; k < nq; ++k) {
    Q.blocks[k].sbeg = Q.nsteps;
    Q.blocks[k].nst = (count[k] + 3) / 4;
    Q.nsteps += Q.blocks[k].nst;
    Q.nquads += count[k];
  }
  if (!((double)Q.nquads <= kQuadShare * (double)pb.npairs)) return without();
  const size_t bytes = (size_t)Q.nsteps * quad_step_bytes<D>(), pad = (size_t)kQuadPadSteps * quad_step_bytes<D>();
  if (hipMalloc(&Q.d_steps, bytes + pad)) return without();
  e = hipMemsetAsync((char*)Q.d_steps + bytes, 0, pad, st);
  if (e == hipSuccess)
    e = hipMemcpyAsync(Q.d_blocks, Q.blocks.data(), sizeof(QuadBlk) * nq, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_quad_write<D>, dim3(loop_blocks(nq)), dim3(256), 0, st, dims, nq, Q.d_blocks, d_src, pb.d_blocks,
                       d_pidx, pb.d_pairs, d_assign, (char*)Q.d_steps);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  drop();
  if (e != hipSuccess) {
    free_quads(ctx);
    return set_error(ctx, DGV_ERR_HIP, std::string("merged layout: ") + hipGetErrorString(e));
  }
  Q.use = true;
  return DGV_OK;
}

int build_quads(dgv_ctx* ctx) {
  free_quads(ctx);
  if (ctx->pb.npairs == 0 || ctx->pb.blocks.empty()) return DGV_OK;
  if (ctx->g.D == 27) return build_quads_t<27>(ctx);
  if (ctx->g.D == 8) return build_quads_t<8>(ctx);
  return DGV_OK;
}

// Work items of the merged layout.  With no tile set by the caller, an item
// holds what one of the chip's 512 resident workgroups gets, 96 steps (24 per wave)
// at least and 2048 at most: an item's start and its partial rows (7 KB) cost
// about 5 us, which below 96 steps no longer pays even where it fills the chip,
// and above 2048 the items of a large grid balance by number.  Q by steps per
// item: 9^3 nodes 21 / 105 / 420 steps 33 / 15.5 / 25 us; 15^3 nodes 80 / 330 / 660 /
// 1300 steps 136 / 94 / 92 / 105 us; 27^3 nodes 300 / 1200 steps 5.7 / 5.15 ms.
int build_quad_plan(dgv_ctx* ctx, int32_t ppi) {
  const QuadLayout& Q = ctx->quad;
  Plan& P = ctx->plan;
  P.pairs_per_item = ppi;
  P.quad = true;
  double total = 0;   // steps x chunks
  for (const Group& G : Q.groups) {
    int64_t n = 0;
    for (int b = G.bbeg; b < G.bend; ++b) n += Q.blocks[b].nst;
    total += (double)n * ((G.ncells + kQuadCols - 1) / kQuadCols);
  }
  // a caller's tile cuts no block finer than about its pair blocks, the least the pair-block
  // plan takes: 48 of up to 183 steps (27 nodes per cell; those of 8 are never cut)
  const double steps = ppi > 0 ? std::max(48.0, (double)ppi * (double)Q.nsteps / (double)std::max<int64_t>(ctx->pb.npairs, 1))
                               : std::min(2048.0, std::max(96.0, total / 512));
  // f is transposed first where that pays for its launch: 15^3 nodes (340 K steps)
  // 94 us with, 102 without; 9^3 nodes (22 K steps) 17.4 with, 15.2 without
  P.transpose = total >= (1 << 16);
  const int64_t target = std::max<int64_t>(1, (int64_t)steps);
  if (ppi <= 0)   // the pairs that make the same items
    P.pairs_per_item =
        (int32_t)std::min(1e9, std::ceil(steps * (double)ctx->pb.npairs / (double)std::max<int64_t>(Q.nsteps, 1)));
  struct Run { int32_t group, b0, b1, s0, s1; int64_t work; };
  std::vector<Run> runs;
  for (size_t gi = 0; gi < Q.groups.size(); ++gi) {
    const Group& G = Q.groups[gi];
    const int64_t nchunk = (G.ncells + kQuadCols - 1) / kQuadCols;
    for (int32_t b0 = G.bbeg; b0 < G.bend;) {
      const int32_t n0 = Q.blocks[b0].nst;
      if (n0 > target + target / 2) {   // cut one block
        const int32_t parts = (int32_t)((n0 + target - 1) / target);
        for (int32_t k = 0; k < parts; ++k) {
          const int32_t s0 = (int32_t)((int64_t)n0 * k / parts), s1 = (int32_t)((int64_t)n0 * (k + 1) / parts);
          runs.push_back({(int32_t)gi, b0, b0 + 1, s0, s1, (s1 - s0) * nchunk});
        }
        ++b0;
        continue;
      }
      int32_t b1 = b0 + 1;
      int64_t acc = n0;
      while (b1 < G.bend && acc + Q.blocks[b1].nst <= target) acc += Q.blocks[b1++].nst;
      runs.push_back({(int32_t)gi, b0, b1, 0, INT32_MAX, acc * nchunk});
      b0 = b1;
    }
  }
  // XCD-aware order: a run's chunks read the same steps, so they go to one XCD
  // (workgroup i is dispatched to XCD i % 8), largest runs first
  constexpr int kXcd = 8;
  std::stable_sort(runs.begin(), runs.end(), [](const Run& x, const Run& y) { return x.work > y.work; });
  std::vector<std::vector<QuadItem>> col(kXcd);
  std::vector<int64_t> load(kXcd, 0);
  for (const Run& r : runs) {
    const int c = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    const Group& G = Q.groups[r.group];
    QuadItem it{};
    it.group = r.group;
    it.blk = r.b0; it.nblk = r.b1 - r.b0; it.s0 = r.s0; it.s1 = r.s1;
    for (int d = 0; d < 3; ++d) { it.lo[d] = G.lo[d]; it.ext[d] = G.ext[d]; }
    it.ncells = G.ncells;
    it.first = Q.blocks[r.b0];
    for (int ch = 0; ch * kQuadCols < G.ncells; ++ch) {
      it.chunk = ch;
      col[c].push_back(it);
    }
    load[c] += r.work;
  }
  size_t nslot = 0;
  for (auto& v : col) nslot = std::max(nslot, v.size());
  QuadItem none{};
  none.chunk = -1;
  P.qitems.assign(nslot * kXcd, none);
  std::vector<int64_t> row0;
  std::vector<const Group*> grp;
  std::vector<int32_t> cell0;
  for (size_t rr = 0; rr < nslot; ++rr)
    for (int c = 0; c < kXcd; ++c) {
      const size_t pos = rr * kXcd + c;
      QuadItem& it = P.qitems[pos];
      if (rr < col[c].size()) it = col[c][rr];
      it.prow = (int64_t)pos * kQuadCols;
      if (it.chunk >= 0) {
        row0.push_back(it.prow);
        grp.push_back(&Q.groups[it.group]);
        cell0.push_back(it.chunk * kQuadCols);
      }
    }
  P.nrows = (int64_t)P.qitems.size() * kQuadCols;
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  DGV_HIP(ctx, hipMalloc(&P.d_qitems, sizeof(QuadItem) * std::max<size_t>(P.qitems.size(), 1)));
  DGV_HIP(ctx, hipMemcpy(P.d_qitems, P.qitems.data(), sizeof(QuadItem) * P.qitems.size(), hipMemcpyHostToDevice));
  return plan_cell_rows(ctx, row0, grp, cell0, kQuadCols);
}

// f transposed to [node of the cell][cell], for the staging reads of k_quad_eval
__global__ __launch_bounds__(256) void k_quad_transpose(int64_t ncells, int D, const double* __restrict__ f,
                                                        double* __restrict__ ft) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= ncells * D) return;
  ft[(i % D) * ncells + i / D] = f[i];
}

// One VDF: columns = 32 cells of the item's box.  A wave stages whole slots, lane
// = (column, parity of the node).  f element (cell, p) is at cell * sc + p * sp
// bytes: with f transposed the columns of one row are runs of cells along w.
template <int D, bool MIX, int NW>
__global__ __launch_bounds__(64 * NW, 2) void k_quad_eval(const QuadItem* __restrict__ items,
                                                          const QuadBlk* __restrict__ blocks,
                                                          const double* __restrict__ steps,
                                                          const double* __restrict__ f, const double* __restrict__ gm,
                                                          uint32_t sc, uint32_t sp, double* __restrict__ partial,
                                                          int Mv, int Mw) {
  constexpr int ROWS = quad_rows<D>();
  constexpr int NI = (D + 1) / 2;                 // loads per lane and slot
  constexpr int SL = (MIX ? 16 : 8) / NW;         // slot copies per wave
  static_assert(SL * NW == (MIX ? 16 : 8), "the slots divide over the waves");
  __shared__ __attribute__((aligned(16))) double lf[ROWS * kQuadRow];
  __shared__ __attribute__((aligned(16))) double lg[MIX ? ROWS * kQuadRow : 2];
  const QuadItem& it = items[blockIdx.x];
  const int chunk = it.chunk, ncells = it.ncells;
  if (chunk < 0) return;   // padding slot of the XCD-aware order
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cl = chunk * kQuadCols + (lane & 31), odd = lane >> 5;
  int r = cl < ncells ? cl : chunk * kQuadCols;   // idle columns stage the chunk's first cell (in range)
  const int cw = it.lo[2] + r % it.ext[2];
  r /= it.ext[2];
  const int cv = it.lo[1] + r % it.ext[1];
  r /= it.ext[1];
  const int cell = ((it.lo[0] + r) * Mv + cv) * Mw + cw;
  // rows odd, odd + 2, ...: the byte offset of the lane's first row (with an odd D
  // the last round's odd lanes repeat the last row), in f and in the staged rows
  const uint32_t goff = (uint32_t)cell * sc + (uint32_t)odd * sp;
  const uint32_t glast = D % 2 ? (uint32_t)cell * sc : goff;
  const uint32_t loff = (uint32_t)(odd * kQuadRow + (lane & 31)) * 8;
  const uint32_t llast = D % 2 ? (uint32_t)(lane & 31) * 8 : loff;
  for (int i = threadIdx.x; i < kQuadRow; i += 64 * NW) {
    lf[8 * D * kQuadRow + i] = 0.0;
    if constexpr (MIX) lg[8 * D * kQuadRow + i] = 0.0;
  }
  const QuadBlk* bl = blocks + it.blk;
  auto header = [&](int i) { return bl[i]; };
  double v[SL][NI];
  auto fetch = [&](const QuadBlk& B) {
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      const int sl = wave + NW * k, slot = sl & 7;
      if (slot & B.same) continue;   // the cell of a lower slot: its rows are used
      const int du = slot & 1 ? B.b[0] : B.a[0], dv = slot & 2 ? B.b[1] : B.a[1], dw = slot & 4 ? B.b[2] : B.a[2];
      const double* src = MIX && sl >= 8 ? gm : f;
      const __amdgpu_buffer_rsrc_t F =
          ring_rsrc(reinterpret_cast<const char*>(src) + (int64_t)((du * Mv + dv) * Mw + dw) * sc);
#pragma unroll
      for (int i = 0; i < NI; ++i) v[k][i] = ring_f64(F, i + 1 < NI ? goff : glast, (uint32_t)(2 * i) * sp);
    }
  };
  auto store = [&](const QuadBlk& B) {
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      const int sl = wave + NW * k, slot = sl & 7;
      if (slot & B.same) continue;
      char* dst = reinterpret_cast<char*>(MIX && sl >= 8 ? lg : lf) + slot * D * kQuadRow * 8;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        *reinterpret_cast<double*>(dst + (i + 1 < NI ? loff : llast) + 2 * i * kQuadRow * 8) = v[k][i];
    }
  };
  const int ncols = min(kQuadCols, ncells - chunk * kQuadCols);
  double* out = partial + it.prow * D;
  constexpr int RT = (D + 15) / 16;
  auto walk = [&](auto ct) {
    constexpr int CT = decltype(ct)::value;
    qd4 acc[RT][CT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[rt][c] = qd4{0.0, 0.0, 0.0, 0.0};
    quad_walk<D, MIX, NW, CT>(it.nblk, it.first, it.s0, it.s1, steps, lf, lg, header, fetch, store, acc);
    quad_flush<D, NW, CT>(lf, acc, ncols, out);
  };
  if (ncols > 16) walk(std::integral_constant<int, 2>{});
  else walk(std::integral_constant<int, 1>{});
}

// d_g != nullptr: the mixed term with g
int launch_main_quad(dgv_ctx* ctx, const double* d_f, const double* d_g, double* part) {
  const Grid& g = ctx->g;
  const QuadLayout& Q = ctx->quad;
  const Plan& P = ctx->plan;
  const unsigned n = (unsigned)P.qitems.size();
  if (n == 0) return DGV_OK;
  // Large evaluations read f transposed (one small kernel before them); small ones
  // would pay more for that launch than for strided reads of an f that is in L2.
  const double *F = d_f, *G = d_g ? d_g : d_f;
  uint32_t sc = (uint32_t)g.D * 8, sp = 8;
  if (P.transpose) {
    const unsigned nb = (unsigned)((g.N + 255) / 256);
    double* ft = ctx->d_ft;
    hipLaunchKernelGGL(k_quad_transpose, dim3(nb), dim3(256), 0, ctx->stream, g.ncells, g.D, d_f, ft);
    F = G = ft;
    if (d_g) {
      hipLaunchKernelGGL(k_quad_transpose, dim3(nb), dim3(256), 0, ctx->stream, g.ncells, g.D, d_g, ft + g.N);
      G = ft + g.N;
    }
    sc = 8;
    sp = (uint32_t)g.ncells * 8;
  }
  // 2^22 items of up to 512 threads a launch (a multiple of the XCDs, so the order holds)
  constexpr unsigned kItems = 1u << 22;
#define DGV_QUAD(DD, MM, NW)                                                                            \
  for (unsigned i = 0; i < n; i += kItems)                                                              \
  hipLaunchKernelGGL((k_quad_eval<DD, MM, NW>), dim3(std::min(kItems, n - i)), dim3(64 * NW), 0,        \
                     ctx->stream, P.d_qitems + i, Q.d_blocks, Q.d_steps, F, G, sc, sp, part, g.Mv, g.Mw)
  if (g.D == 27) {
    if (d_g) DGV_QUAD(27, true, 8);
    else DGV_QUAD(27, false, 4);
  } else {
    if (d_g) DGV_QUAD(8, true, 8);
    else DGV_QUAD(8, false, 4);
  }
#undef DGV_QUAD
  DGV_HIP(ctx, hipGetLastError());
  return DGV_OK;
}

}  // namespace dgv
