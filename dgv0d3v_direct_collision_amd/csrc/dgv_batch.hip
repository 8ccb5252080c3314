// dgv_batch.hip -- many VDFs, on one or several grids, in one persistent launch.
//
// Every instance is a VDF on one of the given grid contexts (each carrying its
// own A-array in the pair-block layout).  The values of all instances of a grid
// are packed node-major, instance-minor: F[node * Bpad + instance] with Bpad the
// instance count rounded up to 64, so that the f values one block needs for 64
// instances are one coalesced row.
//
// Work decomposition.  For an output cell c the contributing blocks are those
// whose box contains c; their list is cut into segments of about `tile` pairs.
// A work item is (grid, cell, segment, chunk of 64 instances), one wave; the
// items of all grids form one queue consumed by a persistent launch.  For each
// block of its segment the wave stages f[c+a][*][64 instances] and
// f[c+b][*][64 instances] in LDS and accumulates, on the matrix cores,
//   S[l, v] += sum_pairs T[l, pair] * f[c+a][p][v] f[c+b][q][v],
// i.e. the same contraction as the single-VDF kernel with instances in place
// of cells.  FP64: v_mfma_f64_16x16x4_f64.  FP32-compensated: the coefficients
// and f are rounded to FP32, products and the per-block sums run on
// v_mfma_f32_16x16x4_f32, and the sums of every 32 pairs are folded into an
// FP32 (hi, lo) pair with the two-sum of Knuth; the item writes hi + lo in FP64.
// FP64: two waves per item, block sums added into an FP64 running total; where the
// grids' A-arrays have a merged layout (dgv_quad.h) k_quad_batch evaluates it
// instead, for 32 instances per item.
// INT8_SPLIT: the same contraction in exact integer arithmetic (k_batch_i8).  A
// second
// kernel adds the items of each (cell, instance) in a fixed order in FP64 and
// applies 2/w (and the spatial operator's scale).
#include <algorithm>
#include <array>
#include <climits>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "dgv_quad.h"

namespace dgv {

struct BatchGridDev {
  const double* pairs64;   // npairs * (D+1) doubles
  const float* pairs32;    // npairs * (D+2) floats (FP32-compensated path): T, p and q row offsets
  const BlockHdr* blocks;
  const int32_t* blist;    // per-cell block lists, concatenated
  const double* gwts;
  // INT8_SPLIT: coefficient digits, pair codes, per-block row scales and the
  // first padded pair of each block (blocks padded to multiples of 16 pairs)
  const uint32_t* digits;
  const uint32_t* codes;
  const double* bscale;
  const int64_t* pbeg16;
  // merged layout: blist then lists quad blocks
  const QuadBlk* qblocks;
  const double* qsteps;
  int64_t foff;            // offset of this grid in the packed buffers
  int64_t eoff;            // offset of this grid in the per-(cell, instance) exponents (foff / D)
  int32_t Bpad, Mv, Mw, D;
};

// Work item: one cell's segment of blocks for up to kChunksPerItem chunks of
// 64 instances (vc0 .. vc0 + nvc - 1); chunk k of the item writes the partial
// rows prow + 64 k .. prow + 64 k + 63.  Where an item has fewer chunks than its
// workgroup has waves for (FP32 modes and INT8_SPLIT), its blocks are cut into
// `parts` shares of about equal pairs and the waves of a share take all its
// chunks; the shares' sums are added in LDS, in order.  Without the shares
// half (INT8_SPLIT, up to 64 instances) or three quarters (FP32) of the waves
// idled: 64 instances on 27^3 nodes INT8_SPLIT 757 -> 479 ms, 16 on 9^3 nodes FP32
// 0.99 -> 0.30 ms; full items are untouched.  Merged layout: one
// chunk of 32 instances, partial rows prow .. prow + 31.
constexpr int kMaxParts = 4;
struct BatchItem {
  int32_t grid, cell, b0, b1;  // blist range of the segment
  int32_t vc0, nvc;            // chunks of 64 instances
  int64_t prow;                // first partial row
  int32_t parts, cut[kMaxParts + 1];   // share p: cut[p] .. cut[p + 1]
};
// share p of an item, by scalar loads (an index into a copy of the item would put
// it in scratch memory, and the block walk with it on vector loads)
__device__ __forceinline__ int2 item_share(const BatchItem* it, int p) { return make_int2(it->cut[p], it->cut[p + 1]); }

// The batched kernels' eight work queues: items beg[q] .. beg[q + 1] - 1.  A
// queue holds whole runs of blocks (every cell's items of a run), so the
// workgroups that start on it -- those of one XCD, which the dispatcher fills
// round-robin by workgroup index -- share that run's records in their L2.
constexpr int kQueues = 8;
struct QueueBounds {
  int32_t beg[kQueues + 1];
};

// The next item for a workgroup (called by one thread; q and left are that
// thread's and start at blockIdx.x % kQueues and kQueues): its own queue
// first, then the others in turn once it is empty.  An empty queue stays empty,
// so a workgroup ends after at most one failed take per queue; -1 = no work left.
__device__ __forceinline__ int take_item(int* __restrict__ counter, const QueueBounds& QB, int& q, int& left) {
  while (left > 0) {
    const int k = atomicAdd(counter + q, 1);
    if (k < QB.beg[q + 1] - QB.beg[q]) return QB.beg[q] + k;
    q = (q + 1) % kQueues;
    --left;
  }
  return -1;
}

// One work decomposition: the items of the queue and the fixed-order reduction
// of their partial rows.  A batch keeps the plan over all cells and, on
// request, a probe plan over a chosen set of cells.
struct BatchPlan {
  bool ready = false;              // every part is built
  int32_t tile = 0;
  QueueBounds queues{};            // queue q holds items queues.beg[q] .. queues.beg[q + 1] - 1
  std::vector<BatchItem> items;
  BatchItem* d_items = nullptr;
  int64_t nrows = 0;
  double* d_partial = nullptr;
  // per (grid, cell, chunk): the partial rows in item order
  int64_t nred = 0;
  int32_t* d_red_rows = nullptr;
  int64_t* d_red_ptr = nullptr;
  int32_t* d_red_key = nullptr;    // (grid, cell, chunk) per reduction task
};

// per grid: what the batched projection needs
struct BatchProjGrid {
  const double *u, *v, *w, *gw;
  double L[25];                    // Cholesky factor of the invariants' Gram matrix
  int64_t foff, N;
  int32_t Bpad, nin;
};

}  // namespace dgv

struct dgv_batch {
  std::vector<dgv_ctx*> grids;
  std::vector<uint64_t> a_gen;     // each grid's A-array generation at creation
  int device = 0;                  // kept here: destroy must not read a grid context (it may be gone)
  int precision = DGV_FP64;
  bool quad = false;               // FP64 on the grids' merged layouts
  int32_t ninst = 0;
  std::vector<int32_t> inst_grid, inst_local;
  std::vector<int32_t> nin, Bpad;
  std::vector<int64_t> foff;       // element offset of each grid's packed block
  int64_t total = 0;               // packed elements
  double* d_f = nullptr;
  double* d_q = nullptr;
  float* d_f32 = nullptr;
  double* d_tmp[4] = {nullptr, nullptr, nullptr, nullptr};
  std::vector<int32_t*> d_blist;
  std::vector<std::vector<int64_t>> cell_ptr;  // per grid: ncells+1 offsets into blist
  std::vector<std::vector<int32_t>> h_blist;   // per grid: host copy of the per-cell block lists
  std::vector<float*> d_pairs32;
  // INT8_SPLIT: per grid, the coefficient digits (d_i8[g][0]), pair codes [1],
  // block row scales [2] and padded block starts [3]; per evaluation, f scaled
  // per (cell, instance) by a power of two (d_fhat) and the exponents (d_fexp)
  std::vector<std::array<void*, 4>> d_i8;
  double* d_fhat = nullptr;
  int32_t* d_fexp = nullptr;
  dgv::BatchGridDev* d_grids = nullptr;
  int32_t waves_per_cu = 0;
  dgv::BatchPlan plan;             // all cells
  dgv::BatchPlan probe;            // the probe cells (empty until set)
  std::vector<int32_t> probe_cells;
  dgv::BatchProjGrid* d_proj = nullptr;   // projection tables per grid
  int32_t* d_proj_task = nullptr;         // (grid, chunk) per block
  int32_t nproj_task = 0;
  int project = 0;                        // project every evaluation's Q (FP64)
  int* d_counter = nullptr;
  int32_t* d_nin = nullptr;        // instances per grid
  double* d_stage = nullptr;       // one instance's values (host copies)
  int ncu = 256;
  hipStream_t stream = nullptr;
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
  hipGraphExec_t graph = nullptr;
  int graph_key[2] = {0, 0};
  double graph_dt = 0, graph_coef = 0;
  std::string err;
};

namespace dgv {

static int berr(dgv_batch* b, int code, const std::string& m) {
  if (b) b->err = m;
  set_global_error(m);
  if (code == DGV_ERR_NOMEM) (void)hipGetLastError();   // the failed hipMalloc's sticky error
  return code;
}

// The batch keeps device pointers into its grids' A-arrays and copies made
// from them; once a grid's A-array is replaced, truncated or changed in place
// they are stale, and nothing may run on them.
bool batch_stale(const dgv_batch* b) {
  for (size_t g = 0; g < b->grids.size(); ++g)
    if (!b->grids[g]->has_a || b->grids[g]->a_gen != b->a_gen[g]) return true;
  return false;
}

static int batch_check_grids(dgv_batch* b) {
  for (size_t g = 0; g < b->grids.size(); ++g)
    if (!b->grids[g]->has_a || b->grids[g]->a_gen != b->a_gen[g])
      return berr(b, DGV_ERR_STATE, "the A-array of grid " + std::to_string(g) +
                                        " changed after the batch was created; create a new batch");
  return DGV_OK;
}
#define BHIP(b, call)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (call);                                                                    \
    if (e_ != hipSuccess) return berr((b), DGV_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef double bd4 __attribute__((ext_vector_type(4)));
#define AS1 __attribute__((address_space(1)))   // global memory: plain global loads, not flat
typedef float bf4 __attribute__((ext_vector_type(4)));

__global__ void k_to_f32(int64_t n, const double* __restrict__ a, float* __restrict__ b) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) b[i] = (float)a[i];
}

// FP32 copy of the pair records for the batched kernel: D coefficients, then
// the byte offsets p * 64 * 4 and q * 64 * 4 of the pair's rows in the staged
// f columns (64 floats per row), so that the kernel forms its LDS addresses
// with one add each.
__global__ void k_pairs_to_f32(int64_t npairs, int D, const double* __restrict__ a, float* __restrict__ b) {
  const int64_t n = npairs * (D + 2), step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    const int64_t k = i / (D + 2);
    const int l = (int)(i - k * (D + 2));
    const double* r = a + k * (D + 1);
    if (l < D) {
      b[i] = (float)r[l];
    } else {
      const int code = (int)__double_as_longlong(r[D]);
      b[i] = __int_as_float(l == D ? (code >> 8) * 256 : (code & 255) * 256);
    }
  }
}

__global__ void k_reset_counter(int* c) {
  if (blockIdx.x == 0 && threadIdx.x < kQueues) c[threadIdx.x] = 0;
}

// Knuth's two-sum: s + e == a + b exactly.
__device__ __forceinline__ void two_sum(float a, float b, float& s, float& e) {
  s = a + b;
  const float bp = s - a;
  e = (a - (s - bp)) + (b - bp);
}

// One workgroup of four waves per item; all waves walk the same blocks and
// pairs in step (a barrier per block), so the coefficient stream of a segment
// is fetched from memory once per item and served from the caches to the
// other waves.  FP32: wave w owns chunk w (64 instances, four column tiles of
// 16); the matrix-core sums of every 32 pairs are folded into an FP32
// (hi, lo) pair with two-sum.  FP64: waves 2c and 2c+1 share chunk c (32
// instances each); block sums are added into an FP64 running total.
constexpr int kWavesPerItem = 4;
constexpr int kPadPairs = 64;   // zero pairs after the FP32 coefficients (>= 4 kRing + 3)

template <bool FP32>
constexpr int chunks_per_item() { return FP32 ? 4 : 2; }

// FP32 row map of the matrix-core tiles: tile 0 holds basis functions 0..15 in
// rows 0..15; tile 1 holds function 16 + 3 (i / 4) + i % 4 in row i for
// i % 4 < 3.  Every unused row (i % 4 == 3 in tile 1, or a function past D,
// both mapped to D) then falls in accumulator element 3 of tile 1 (the FP32
// output row of element e is 4 (lane / 16) + e), which the fold skips.
template <int D>
__device__ __forceinline__ int f32_row_fn(int rt, int i) {
  static_assert(D <= 28, "tile 0 holds 16 functions, tile 1 holds 12");
  const int l = rt == 0 ? i : ((i & 3) < 3 ? 16 + 3 * (i >> 2) + (i & 3) : D);
  return min(l, D);
}

// MODE is the batch's precision: DGV_FP64, DGV_FP32_COMP (FP32 products and
// matrix-core sums, two-sum compensated FP32 accumulation of the 32-pair
// sums) or DGV_FP32_F64ACC (the same FP32 products and sums, accumulated in
// FP64 instead: two VALU instructions per element against seven).
template <int D, int MODE>
__global__ __launch_bounds__(64 * kWavesPerItem) void k_batch_mfma(const BatchItem* __restrict__ items, const QueueBounds QB,
                                                                   const BatchGridDev* __restrict__ grids,
                                                                   const double* __restrict__ f64,
                                                                   const float* __restrict__ f32,
                                                                   double* __restrict__ partial,
                                                                   int* __restrict__ counter) {
  constexpr bool FP32 = MODE != DGV_FP64;
  constexpr bool ACC64 = MODE == DGV_FP32_F64ACC;
  constexpr int RT = (D + 15) / 16;
  constexpr int CH = chunks_per_item<FP32>();    // chunks per item
  constexpr int WPC = kWavesPerItem / CH;        // waves per chunk
  constexpr int CT = 4 / WPC;                    // column tiles per wave
  using T = typename std::conditional<FP32, float, double>::type;
  using V4 = typename std::conditional<FP32, bf4, bd4>::type;
  typedef T VB __attribute__((ext_vector_type(CT)));
  static_assert(sizeof(VB) == 16, "one 16-byte LDS read per lane and step");
  __shared__ __attribute__((aligned(16))) T lf[2][CH][D * 64];   // f(c+a) | f(c+b) of each chunk
  __shared__ int s_item;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kk = lane >> 4, jj = lane & 15;
  const int ch = wave / WPC;                     // this wave's chunk within the item
  const int sub = wave % WPC;                    // its part of the chunk's staging / columns
  const int col0 = sub * 16 * CT;
  const int lcol = col0 + CT * jj;               // the lane's first instance in a staged row
  // FP32: the lane's byte offsets inside a step of 4 pairs (the coefficient of
  // its tile rows' basis functions, unused rows on the code slot D, and the
  // pair's code)
  uint32_t loffb[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) loffb[rt] = (uint32_t)((kk * (D + 2) + f32_row_fn<D>(rt, jj)) * (int)sizeof(float));
  const uint32_t coffb = (uint32_t)((kk * (D + 2) + D) * (int)sizeof(float));
  // FP64: the same inside a step of the context's pair records (D + 1 doubles each)
  uint32_t loffb64[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) loffb64[rt] = (uint32_t)((kk * (D + 1) + min(16 * rt + jj, D)) * 8);
  const uint32_t coffb64 = (uint32_t)((kk * (D + 1) + D) * 8 + 4);   // the LDS offsets (pair_code_bits)
  const V4 vzero = V4{0, 0, 0, 0};
  int q = blockIdx.x % kQueues, left = kQueues;   // this workgroup's XCD queue first
  for (;;) {
    if (tid == 0) s_item = take_item(counter, QB, q, left);
    __syncthreads();
    const int id = __builtin_amdgcn_readfirstlane(s_item);   // the workgroup's item, uniform
    __syncthreads();
    if (id < 0) return;
    const BatchItem it = items[id];
    const BatchGridDev G = grids[it.grid];
    // FP32: a wave's chunk and its share of the blocks.  Shares walk different blocks,
    // each wave on its own staged rows, so only an undivided item keeps its waves in step
    const int part = FP32 ? ch / it.nvc : 0, vc = FP32 ? ch - part * it.nvc : ch;
    const bool active = FP32 ? part < it.parts : ch < it.nvc;
    const bool in_step = !FP32 || it.parts == 1;
    const int2 share = FP32 && active ? item_share(items + id, part) : make_int2(it.b0, it.b1);
    const int Mv = G.Mv, Mw = G.Mw;
    const int c = it.cell;
    const int cw = c % Mw, cv = (c / Mw) % Mv, cu = c / (Mw * Mv);
    const int64_t vb = (int64_t)(it.vc0 + vc) * 64 + lane;   // the instance this thread stages
    V4 acc[RT][CT], hi[RT][CT], lo[RT][FP32 ? CT : 1];
    bd4 hd[RT][ACC64 ? CT : 1];   // DGV_FP32_F64ACC: the FP64 running sums
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        acc[rt][ct] = V4{0, 0, 0, 0};
        hi[rt][ct] = V4{0, 0, 0, 0};
        if constexpr (FP32) lo[rt][ct] = V4{0, 0, 0, 0};
        if constexpr (ACC64) hd[rt][ct] = bd4{0, 0, 0, 0};
      }
    T* la = lf[0][ch];
    T* lb = lf[1][ch];
    int prev_xc = -1;   // the cell whose f is in la (blocks come ordered by a)
    // fold a round's matrix-core sums into the FP32 (hi, lo) pair, or into the
    // FP64 sums (the next round's first products start a fresh sum, so acc
    // needs no clearing); element 3 of tile 1 holds only unused rows
    // (f32_row_fn) and is skipped
#define FOLD()                                                                                \
  do {                                                                                        \
    _Pragma("unroll") for (int rt = 0; rt < RT; ++rt)                                         \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct)                                         \
    _Pragma("unroll") for (int e = 0; e < (rt == 0 ? 4 : 3); ++e) {                           \
      if constexpr (ACC64) {                                                                  \
        hd[rt][ct][e] += (double)acc[rt][ct][e];                                              \
      } else {                                                                                \
        float s2_, er_;                                                                       \
        two_sum(hi[rt][ct][e], acc[rt][ct][e], s2_, er_);                                     \
        hi[rt][ct][e] = s2_;                                                                  \
        lo[rt][ct][e] += er_;                                                                 \
      }                                                                                       \
    }                                                                                         \
  } while (0)
    for (int bi = share.x; bi < share.y; ++bi) {
      const BlockHdr* B = G.blocks + G.blist[bi];
      const int xc = ((cu + B->a[0]) * Mv + (cv + B->a[1])) * Mw + (cw + B->a[2]);
      const int yc = ((cu + B->b[0]) * Mv + (cv + B->b[1])) * Mw + (cw + B->b[2]);
      const bool new_x = xc != prev_xc;
      prev_xc = xc;
      const int n = B->npairs;
      // Coefficient operand of step s (4 pairs): lane i holds T[pair 4s + i/16][16 rt + i%16]
      // (rows >= D read the pair's code slot and only feed output rows that are
      // dropped).  Both record arrays carry zero pairs past their end, so the
      // ring of kRing steps in flight reads straight ahead -- a uniform step base
      // plus the lane's fixed byte offset, no clamping; only the block's last,
      // partial step masks the pairs past its end.  The ring is filled before
      // the f staging, so the block's two memory latencies overlap.
      constexpr int kRing = 8;
      static_assert(4 * kRing + 3 <= kPairPad && 4 * kRing + 3 <= kPadPairs, "the ring reads at most 4 kRing + 3 pairs past a block");
      T ab[kRing][RT];
      int cbits[kRing];
      int qbits[FP32 ? kRing : 1];
      const __amdgpu_buffer_rsrc_t P =
          ring_rsrc(FP32 ? (const void*)(G.pairs32 + B->pbeg * (D + 2)) : (const void*)(G.pairs64 + B->pbeg * (D + 1)));
      constexpr uint32_t kStepBytes = FP32 ? 4 * (D + 2) * sizeof(float) : 4 * (D + 1) * 8;
#define LOAD32(slot, step)                                                                    \
  do {                                                                                        \
    const uint32_t s_ = kStepBytes * (uint32_t)(step);                                        \
    _Pragma("unroll") for (int rt = 0; rt < RT; ++rt) ab[slot][rt] = ring_f32(P, loffb[rt], s_); \
    ring_i32x2(P, coffb, s_, cbits[slot], qbits[slot]);                                       \
  } while (0)
#define LOAD64(slot, step)                                                                    \
  do {                                                                                        \
    const uint32_t s_ = kStepBytes * (uint32_t)(step);                                        \
    _Pragma("unroll") for (int rt = 0; rt < RT; ++rt) ab[slot][rt] = ring_f64(P, loffb64[rt], s_); \
    cbits[slot] = ring_i32(P, coffb64, s_);                                                   \
  } while (0)
      if (active && n > 0) {
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
          if constexpr (FP32) LOAD32(u, u);
          else LOAD64(u, u);
        }
      }
      if (in_step) __syncthreads();
      if (active) {
        if constexpr (FP32) {
          const float* F = f32 + G.foff;
          if (new_x) {
#pragma unroll
            for (int p = 0; p < D; ++p) la[p * 64 + lane] = F[((int64_t)xc * D + p) * G.Bpad + vb];
          }
#pragma unroll
          for (int q = 0; q < D; ++q) lb[q * 64 + lane] = F[((int64_t)yc * D + q) * G.Bpad + vb];
        } else {
          // waves 2c and 2c+1 split the rows of chunk c; all loads first
          const double* F = f64 + G.foff;
          constexpr int NS = (D + WPC - 1) / WPC;
          double sa[NS], sb[NS];
#pragma unroll
          for (int i = 0; i < NS; ++i) {
            const int p = min(sub + i * WPC, D - 1);
            if (new_x) sa[i] = F[((int64_t)xc * D + p) * G.Bpad + vb];
            sb[i] = F[((int64_t)yc * D + p) * G.Bpad + vb];
          }
#pragma unroll
          for (int i = 0; i < NS; ++i) {
            const int p = sub + i * WPC;
            if (p < D) {
              if (new_x) la[p * 64 + lane] = sa[i];
              lb[p * 64 + lane] = sb[i];
            }
          }
        }
      }
      if (in_step) __syncthreads();
      else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the wave's own LDS rows, in order
      if (!active || n == 0) continue;
      VB ra, rb;
      T bcur[CT];
      const char* la_lane = reinterpret_cast<const char*>(la + lcol);
      const char* lb_lane = reinterpret_cast<const char*>(lb + lcol);
      // the B operand of a step: LDS reads issued one step ahead of its products.
      // Column jj of tile ct is instance col0 + CT jj + ct, so a lane's CT
      // values are one 16-byte LDS read and the four pairs of a step (four
      // lane groups, different rows q) read disjoint 16-byte runs.
#define B_ISSUE_BYTES(pb, qb)                                                                 \
  do {                                                                                        \
    ra = *reinterpret_cast<const VB*>(la_lane + (pb));                                        \
    rb = *reinterpret_cast<const VB*>(lb_lane + (qb));                                        \
  } while (0)
#define STEP_MFMA(u, fresh)                                                                   \
  do {                                                                                        \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct)                                         \
    _Pragma("unroll") for (int rt = 0; rt < RT; ++rt) {                                       \
      if constexpr (FP32)                                                                     \
        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(ab[u][rt], bcur[ct],               \
                                                           (fresh) ? vzero : acc[rt][ct], 0, 0, 0); \
      else                                                                                    \
        acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(ab[u][rt], bcur[ct], acc[rt][ct], 0, 0, 0); \
    }                                                                                         \
  } while (0)
      if constexpr (FP32) {
#define FINISH32()                                                                            \
  do {                                                                                        \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct) bcur[ct] = ra[ct] * rb[ct];             \
  } while (0)
        const int nfull = n >> 2, nst = (n + 3) >> 2;
        B_ISSUE_BYTES(cbits[0], qbits[0]);
        FINISH32();
#define ROUND32(st_)                                                                           \
  do {                                                                                        \
    _Pragma("unroll") for (int u = 0; u < kRing; ++u) {                                       \
      B_ISSUE_BYTES(cbits[(u + 1) % kRing], qbits[(u + 1) % kRing]);   /* next step */         \
      __builtin_amdgcn_sched_barrier(0);   /* its LDS reads ahead of the products */         \
      STEP_MFMA(u, u == 0);   /* each round starts a fresh matrix-core sum */                 \
      __builtin_amdgcn_sched_barrier(0);   /* and the wait for them behind */                \
      LOAD32(u, (st_) + u + kRing);                                                           \
      FINISH32();                                                                             \
    }                                                                                         \
    FOLD();                                                                                   \
  } while (0)
        // full rounds, two per iteration (the folds' results alternate between
        // two register sets instead of being copied back); the ring refills
        // kRing steps ahead
        int st = 0;
        for (; st + 2 * kRing <= nfull; st += 2 * kRing) {
          ROUND32(st);
          ROUND32(st + kRing);
        }
        if (st + kRing <= nfull) {
          ROUND32(st);
          st += kRing;
        }
#undef ROUND32
        if (st < nst) {   // the last nst - st <= kRing steps, already in the ring
#pragma unroll
          for (int u = 0; u < kRing; ++u) {
            if (st + u < nst) {
              if (st + u == nfull) {   // partial step: pairs past the block's end contribute 0
                const bool ok = 4 * nfull + kk < n;
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) ab[u][rt] = ok ? ab[u][rt] : 0.0f;
              }
              B_ISSUE_BYTES(cbits[(u + 1) % kRing], qbits[(u + 1) % kRing]);
              STEP_MFMA(u, u == 0);
              FINISH32();
            }
          }
          FOLD();
        }
#undef FINISH32
      } else {
        // FP64: the context's pair array, read straight ahead like the FP32
        // copy; the sums of a block go into the running FP64 total after it.
#define ISSUE64(slot)                                                                         \
  do {                                                                                        \
    const uint32_t c_ = (uint32_t)cbits[slot];                                                \
    B_ISSUE_BYTES(c_ & 0xffffu, c_ >> 16);                                                    \
  } while (0)
#define FINISH64()                                                                            \
  do {                                                                                        \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct) bcur[ct] = ra[ct] * rb[ct];             \
  } while (0)
        const int nfull = n >> 2, nst = (n + 3) >> 2;
        ISSUE64(0);
        FINISH64();
        int st = 0;
        for (; st + kRing <= nfull; st += kRing) {
#pragma unroll
          for (int u = 0; u < kRing; ++u) {
            ISSUE64((u + 1) % kRing);
            __builtin_amdgcn_sched_barrier(0);   // LDS reads ahead of the products,
            STEP_MFMA(u, false);
            __builtin_amdgcn_sched_barrier(0);   // and the wait for them behind
            LOAD64(u, st + u + kRing);
            FINISH64();
          }
        }
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
          if (st + u < nst) {
            if (st + u == nfull) {   // partial step: records past the block's end contribute 0
              const bool ok = 4 * nfull + kk < n;
#pragma unroll
              for (int rt = 0; rt < RT; ++rt) ab[u][rt] = ok ? ab[u][rt] : (T)0;
            }
            ISSUE64((u + 1) % kRing);
            STEP_MFMA(u, false);
            FINISH64();
          }
        }
#undef FINISH64
#undef ISSUE64
      }
#undef STEP_MFMA
#undef B_ISSUE_BYTES
#undef LOAD64
#undef LOAD32
      if constexpr (!FP32) {  // two-level FP64 sum
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            hi[rt][ct] += acc[rt][ct];
            acc[rt][ct] = V4{0, 0, 0, 0};
          }
      }
    }
#undef FOLD
    // output layouts: FP64 row 4e + lane/16, FP32 row 4 (lane/16) + e
    double sum[RT][CT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (ACC64) sum[rt][ct][e] = hd[rt][ct][e];
          else if constexpr (FP32) sum[rt][ct][e] = (double)hi[rt][ct][e] + (double)lo[rt][ct][e];
          else sum[rt][ct][e] = hi[rt][ct][e];
        }
    if (FP32 && it.parts > 1) {   // the shares' sums, added by the first share's wave of the chunk
      static_assert(!FP32 || sizeof(lf) >= sizeof(double) * CH * D * 64, "the staged rows make room for the sums");
      double* slab = reinterpret_cast<double*>(&lf[0][0][0]);
      auto at = [&](int w, int rt, int ct, int e) -> double* {
        return slab + ((int64_t)w * D + f32_row_fn<D>(rt, 4 * kk + e)) * 64 + col0 + CT * jj + ct;
      };
      __syncthreads();   // every wave is done with its staged rows
      if (active && part > 0) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (f32_row_fn<D>(rt, 4 * kk + e) < D) *at(ch, rt, ct, e) = sum[rt][ct][e];
      }
      __syncthreads();
      if (part > 0) continue;
      for (int p = 1; p < it.parts; ++p)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (f32_row_fn<D>(rt, 4 * kk + e) < D) sum[rt][ct][e] += *at(vc + p * it.nvc, rt, ct, e);
    }
    if (!active) continue;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        const int v = col0 + CT * jj + ct;
        double* out = partial + (it.prow + 64 * vc + v) * D;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int l = FP32 ? f32_row_fn<D>(rt, 4 * kk + e) : 16 * rt + 4 * e + kk;
          if (l < D) out[l] = sum[rt][ct][e];
        }
      }
  }
}

// ---- INT8_SPLIT: exact integer digit products on the int8 matrix cores ----------------
//
// Per block and basis row l the coefficients are fixed point with the block-row
// exponent eA (max |T_l| < 2^eA): At = rint(T 2^(BA - eA)), |At| < 2^38, written
// as five signed base-256 digits A_0 (most significant) .. A_4.  Per output cell
// c the f of every (cell, instance) is scaled by a power of two so that its
// largest value lies in [2^14, 2^15): fh = f 2^(15 - e).  A pair's product
// x = fh(c+a, p) fh(c+b, q), |x| < 2^30, is rounded to an integer and written as
// four signed digits X_0 .. X_3 in the bytes of one dword (X_0 in the top byte):
// x + 0x80808080 is rounded to an integer by adding it to 2^52 in FP64 (the low
// 32 bits of the sum's significand are then that integer), and each byte's top
// bit is flipped.  Then At x = sum_k 256^(7-k) sum_{t+s=k} A_t X_s, and the levels k = 0..4
// (all digit products down to 256^-4 of the leading one) are accumulated exactly
// in int32 by v_mfma_i32_16x16x64_i8:
//   level 3: A dword (A_0, A_1, A_2, A_3) against the natural x dword;
//   level 4: A dword (A_1, A_2, A_3, A_4) against the natural x dword;
//   level k < 3: the first A dword against the x dword shifted right by 8 (3 - k).
// At the end of a block the five int32 sums are combined in FP64 as
// sum_k acc_k 256^(4-k) and scaled by 256^3 2^(eA - 38) 2^(e(c+a) + e(c+b) - 30)
// into the item's FP64 running sum.
// Dropped: digit products below 256^-4 of the leading one and the roundings of
// At and x, i.e. relative errors near 2^-30 per term at the block's scale.
typedef int bi4 __attribute__((ext_vector_type(4)));
typedef unsigned int bu4 __attribute__((ext_vector_type(4)));
constexpr int kI8BA = 38;                   // coefficient bits: |At| < 2^38
constexpr int kI8BX = 30;                   // product bits: |x| < 2^30
constexpr int kI8FS = 15;                   // f scaled into [2^14, 2^15)
constexpr double kI8Magic = 4503599627370496.0 + 2155905152.0;   // 2^52 + 0x80808080
static_assert(kI8BX == 2 * kI8FS, "a product of two scaled f values has 2 kI8FS bits");
static_assert(kI8BX <= 30, "|x| < 2^30 keeps x + 0x80808080 within the low 32 bits of the rounded sum");

template <int D>
constexpr int i8_dwords_per_pair() { return ((D + 15) / 16) * 16 * 2; }   // 2 dwords per tile row

// One workgroup per block: the block-row exponents, the digit dwords of every
// (pair, row) of the block padded to 16 pairs, and the pairs' LDS row offsets.
// Layout of a 16-pair step s of a block: for each row tile rt, 64 lanes x 8
// dwords, lane 16 g + i holding row i's (A_0..A_3) dwords of pairs 4 g .. 4 g + 3
// then its (A_1..A_4) dwords, i.e. the A operands of the step's MFMAs.
template <int D>
__global__ __launch_bounds__(256) void k_i8_digits(const BlockHdr* __restrict__ blocks,
                                                   const int64_t* __restrict__ pbeg16,
                                                   const double* __restrict__ pairs64,
                                                   uint32_t* __restrict__ digits, uint32_t* __restrict__ codes,
                                                   double* __restrict__ bscale) {
  constexpr int RT = (D + 15) / 16;
  const int blk = blockIdx.x;
  const int n = blocks[blk].npairs;
  const int64_t p0 = blocks[blk].pbeg;
  const int64_t o16 = pbeg16[blk];
  const int n16 = (n + 15) & ~15;
  __shared__ int emax[16 * RT];
  if (threadIdx.x < 16 * RT) emax[threadIdx.x] = INT_MIN;
  __syncthreads();
  for (int i = threadIdx.x; i < n * D; i += blockDim.x) {
    const int j = i / D, l = i - (i / D) * D;
    const double a = pairs64[(p0 + j) * (D + 1) + l];
    if (a != 0.0) {
      int e;
      frexp(a, &e);
      atomicMax(&emax[l], e);
    }
  }
  __syncthreads();
  if (threadIdx.x < 16 * RT) {
    const int l = threadIdx.x;
    // 2^(eA - 38) times 256^3, the weight of the lowest kept level (k = 4):
    // the kernel combines the level sums as sum_k acc_k 256^(4 - k)
    bscale[(int64_t)blk * 16 * RT + l] = (l < D && emax[l] != INT_MIN) ? ldexp(1.0, emax[l] - kI8BA + 24) : 0.0;
  }
  uint32_t* dblk = digits + o16 * i8_dwords_per_pair<D>();
  for (int i = threadIdx.x; i < n16 * 16 * RT; i += blockDim.x) {
    const int j = i / (16 * RT), r = i - j * (16 * RT);
    long long v = 0;
    if (j < n && r < D && emax[r] != INT_MIN) v = llrint(ldexp(pairs64[(p0 + j) * (D + 1) + r], kI8BA - emax[r]));
    int dg[5];
#pragma unroll
    for (int k = 4; k >= 0; --k) {
      const int d = (int)((v + 128) & 255) - 128;
      dg[k] = d;
      v = (v - d) >> 8;
    }
    const uint32_t w1 = (uint32_t)(uint8_t)dg[0] | ((uint32_t)(uint8_t)dg[1] << 8) |
                        ((uint32_t)(uint8_t)dg[2] << 16) | ((uint32_t)(uint8_t)dg[3] << 24);
    const uint32_t w2 = (uint32_t)(uint8_t)dg[1] | ((uint32_t)(uint8_t)dg[2] << 8) |
                        ((uint32_t)(uint8_t)dg[3] << 16) | ((uint32_t)(uint8_t)dg[4] << 24);
    const int st = j >> 4, k = j & 15, g = k >> 2, m = k & 3, rt = r >> 4, ii = r & 15;
    uint32_t* o = dblk + ((int64_t)(st * RT + rt) * 64 + 16 * g + ii) * 8;
    o[m] = w1;
    o[4 + m] = w2;
  }
  for (int j = threadIdx.x; j < n16; j += blockDim.x) {
    uint32_t c = 0;   // padded pairs: rows 0 and 0, zero digits
    if (j < n) {   // LDS byte offsets of the pair's rows p, q in a 32-instance staging buffer
      const uint32_t pq = (uint32_t)__double_as_longlong(pairs64[(p0 + j) * (D + 1) + D]) & 0xffffu;
      c = ((pq >> 8) << 8) | ((pq & 0xffu) << 24);
    }
    codes[o16 + j] = c;
  }
}

// Per (cell, instance) of one grid: e = exponent of max |f| over the cell's D
// nodes (max |f| < 2^e), fh = f 2^(15 - e) (exact), both for k_batch_i8.
template <int D>
__global__ void k_i8_fixed(int64_t ncells, int32_t Bpad, const double* __restrict__ F, double* __restrict__ Fh,
                           int32_t* __restrict__ E) {
  const int64_t n = ncells * Bpad, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += step) {
    const int64_t c = t / Bpad, v = t - c * Bpad;
    double m = 0.0;
#pragma unroll
    for (int p = 0; p < D; ++p) m = fmax(m, fabs(F[(c * D + p) * Bpad + v]));
    int e = -1000;
    if (m > 0.0) frexp(m, &e);
    E[t] = e;
#pragma unroll
    for (int p = 0; p < D; ++p) Fh[(c * D + p) * Bpad + v] = ldexp(F[(c * D + p) * Bpad + v], kI8FS - e);
  }
}

// The INT8_SPLIT evaluator.  Workgroup of four waves per item: two chunks of 64
// instances per item, two waves per chunk, 32 instances per wave (column tiles
// ct = 0, 1; column jj of tile ct = instance 2 jj + ct of the wave's 32).  A
// 16-pair step: per row tile 5 level MFMAs per column tile.
// Inside an item the waves run independently, and the block boundaries are
// hidden behind the products:
//  - the digit and code operands come through a ring of kI8Ring steps in
//    flight (per-block buffer resources).  Once a slot's last step of a block
//    has been used, the slot loads the same-numbered step of the next block, so
//    the next block's first steps are in flight before the current one ends
//    (every digit array ends with kI8Ring zero steps: the ring reads ahead);
//  - each wave stages its own 32 instances of f(c+a), f(c+b) and the block's
//    scales in LDS with direct global-to-LDS loads, double-buffered: the next
//    block's staging is issued when a block starts and has landed when the next
//    block starts, since at least a full ring of loads was issued after it and
//    the wave waits for all but that many;
//  - the block headers come through the scalar cache, two blocks ahead;
//  - the LDS reads of a step's f values are issued two steps ahead and its x
//    dwords computed one step ahead of its products (the reads after the
//    current step's products, the x dwords between them);
//  - a block's passes whose steps and loads all lie in the block run as one
//    unrolled body with no per-step test; only its last one or two passes
//    choose, per slot, between this block and the next.
constexpr int kI8Ring = 6;   // even: the x dwords alternate by step parity; 6 measured faster than 4 or 8

// s_waitcnt immediates: vector memory count n (lgkm and exp counts left free),
// and LDS/scalar count 0 (vector memory and exp left free)
__device__ __forceinline__ constexpr int i8_vmcnt(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }
constexpr int kI8LgkmZero = 15 | (7 << 4) | (3 << 14);

template <int D>
__global__ __launch_bounds__(256) void k_batch_i8(const BatchItem* __restrict__ items, const QueueBounds QB,
                                                  const BatchGridDev* __restrict__ grids,
                                                  const double* __restrict__ fhat, const int32_t* __restrict__ fexp,
                                                  double* __restrict__ partial, int* __restrict__ counter) {
  constexpr int RT = (D + 15) / 16;
  constexpr int ROWS = (D + 3) & ~3;              // staged rows: four per 1 KiB direct load
  constexpr int CT = 2, WPC = 2;
  constexpr int DW = i8_dwords_per_pair<D>();     // digit dwords per pair
  constexpr uint32_t kStepA = 16u * DW * 4u;      // digit bytes per 16-pair step
  constexpr int kRowBytes = 32 * 8;               // a staged row: the wave's 32 instances
  constexpr int kBufBytes = ROWS * kRowBytes;
  constexpr int kSlotLoads = 2 * RT + 1;          // buffer loads per ring slot
  typedef double VB __attribute__((ext_vector_type(2)));
  typedef const __attribute__((address_space(4))) int32_t* ScalarI32;
  typedef const __attribute__((address_space(4))) int64_t* ScalarI64;
  __shared__ __attribute__((aligned(16))) char s_f[4][2][2][kBufBytes];   // [wave][f(c+a) | f(c+b)][buffer]
  __shared__ __attribute__((aligned(16))) double s_sa[4][2][32];         // [wave][block parity]: row scales
  __shared__ __attribute__((aligned(16))) int s_fe[4][2][64];            // [wave][parity]: exponents of f(c+a), f(c+b)
  __shared__ int s_item;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kk = lane >> 4, jj = lane & 15;
  const int ch = wave / WPC, sub = wave % WPC;
  const int lcol = sub * 32 + 2 * jj;              // the lane's instances in the chunk: lcol, lcol + 1
  const uint32_t aoff = (uint32_t)lane * 32u;      // the lane's 8 digit dwords of a step's row tile
  const uint32_t coff = (uint32_t)kk * 16u;        // its lane group's 4 codes of a step
  const bi4 izero = bi4{0, 0, 0, 0};
  int q = blockIdx.x % kQueues, left = kQueues;   // this workgroup's XCD queue first
  for (;;) {
    if (tid == 0) s_item = take_item(counter, QB, q, left);
    __syncthreads();
    const int id = __builtin_amdgcn_readfirstlane(s_item);
    __syncthreads();
    if (id < 0) return;
    const BatchItem it = items[id];
    const int part = ch / it.nvc, vc = ch - part * it.nvc;   // the wave's share of the blocks and its chunk
    const bool active = part < it.parts;   // a chunk without work: its columns lie past the grid's instances
    const int2 share = active ? item_share(items + id, part) : make_int2(0, 0);
    const BatchGridDev G = grids[it.grid];
    const int Mv = G.Mv, Mw = G.Mw;
    const int c = it.cell;
    const int cw = c % Mw, cv = (c / Mw) % Mv, cu = c / (Mw * Mv);
    const int64_t Bpad = G.Bpad;
    const int64_t vcol0 = (int64_t)(it.vc0 + vc) * 64 + sub * 32;   // the wave's first instance
    const double* F = fhat + G.foff;
    const int32_t* FE = fexp + G.eoff;
    double tot[RT][CT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e) tot[rt][ct][e] = 0.0;
    const int nb = share.y - share.x;
    if (nb > 0) {
      const ScalarI32 blist = (ScalarI32)(G.blist + share.x);
      // a block's header: its records, step count and the cells of f(c+a), f(c+b)
      struct Hdr {
        int blk, nst, xc, yc;
        const uint32_t* A;
        const uint32_t* C;
      };
      auto header = [&](int blk) {
        Hdr h;
        h.blk = blk;
        const ScalarI32 w = (ScalarI32)(reinterpret_cast<const char*>(G.blocks + blk) + 8);
        const int w0 = w[0], w1 = w[1];   // a[0..2], b[0]; b[1..2], npairs
        const int a0 = (int8_t)w0, a1 = (int8_t)(w0 >> 8), a2 = (int8_t)(w0 >> 16);
        const int b0 = (int8_t)(w0 >> 24), b1 = (int8_t)w1, b2 = (int8_t)(w1 >> 8);
        h.nst = ((int)(int16_t)(w1 >> 16) + 15) >> 4;
        h.xc = ((cu + a0) * Mv + (cv + a1)) * Mw + (cw + a2);
        h.yc = ((cu + b0) * Mv + (cv + b1)) * Mw + (cw + b2);
        const int64_t o16 = ((ScalarI64)G.pbeg16)[blk];
        h.A = G.digits + o16 * DW;
        h.C = G.codes + o16;
        return h;
      };
      // direct loads of f rows of one cell (the wave's 32 instances) into a buffer
      auto stage_rows = [&](int cell, char* buf) {
        const double* src = F + (int64_t)cell * D * Bpad + vcol0 + 2 * jj;
        const uint32_t lb = lds_addr(buf);
#pragma unroll
        for (int i = 0; i < ROWS / 4; ++i) {
          const int p = min(4 * i + kk, D - 1);
          lds_load16(src + p * Bpad, lb + i * 1024);
        }
      };
      // ... and of a block's row scales and the exponents of its two cells
      auto stage_scales = [&](const Hdr& h, int par) {
        const char* sa = reinterpret_cast<const char*>(G.bscale + (int64_t)h.blk * 16 * RT) + ((lane * 4) & (16 * RT * 8 - 1));
        lds_load4(sa, lds_addr(&s_sa[wave][par][0]));
        const int32_t* se = FE + (int64_t)(lane < 32 ? h.xc : h.yc) * Bpad + vcol0 + (lane & 31);
        lds_load4(se, lds_addr(&s_fe[wave][par][0]));
      };
      // the cell held by each f buffer
      int tag_a0 = -1, tag_a1 = -1, tag_b0 = -1, tag_b1 = -1;
      Hdr cur = header(blist[0]);
      Hdr nxt = header(blist[min(1, nb - 1)]);
      int bq = blist[min(2, nb - 1)];   // the block after nxt
      int pa = 0, pb = 0;               // the current block's f buffers
      stage_rows(cur.xc, s_f[wave][0][0]);
      stage_rows(cur.yc, s_f[wave][1][0]);
      tag_a0 = cur.xc;
      tag_b0 = cur.yc;
      stage_scales(cur, 0);
      bi4 r1[kI8Ring][RT], r2[kI8Ring][RT];
      bu4 rc[kI8Ring];
#define I8_LOAD_R(slot, RA_, RC_, step)                                                              \
  do {                                                                                              \
    const uint32_t sa_ = kStepA * (uint32_t)(step);                                                 \
    _Pragma("unroll") for (int rt = 0; rt < RT; ++rt) {                                             \
      r1[slot][rt] = __builtin_bit_cast(bi4, __builtin_amdgcn_raw_buffer_load_b128(RA_, aoff, sa_ + rt * 2048u, 0)); \
      r2[slot][rt] =                                                                                \
          __builtin_bit_cast(bi4, __builtin_amdgcn_raw_buffer_load_b128(RA_, aoff + 16u, sa_ + rt * 2048u, 0)); \
    }                                                                                               \
    rc[slot] = __builtin_amdgcn_raw_buffer_load_b128(RC_, coff, 64u * (uint32_t)(step), 0);         \
  } while (0)
#define I8_LOAD(slot, pA, pC, step) I8_LOAD_R(slot, ring_rsrc(pA), ring_rsrc(pC), step)
      // in slot order, as in the loop (the loop's waits count loads in that order)
#pragma unroll
      for (int u = 0; u < kI8Ring; ++u) {
        I8_LOAD(u, cur.A, cur.C, u);
        __builtin_amdgcn_sched_barrier(0);
      }
      bi4 acc[5][RT][CT];
      VB fa[4], fb[4];   // f values read from LDS two steps ahead of their products
      bi4 nat[2][CT];    // the x dwords: [step parity], those of the step whose products come next
                         // and those of the step after it (the ring has an even number of slots)
      const char* la_lane;
      const char* lb_lane;
#define I8_LDS(cd_)                                                                                 \
  do {                                                                                              \
    _Pragma("unroll") for (int m = 0; m < 4; ++m) {                                                 \
      fa[m] = *reinterpret_cast<const VB*>(la_lane + ((cd_)[m] & 0xffffu));                         \
      fb[m] = *reinterpret_cast<const VB*>(lb_lane + ((cd_)[m] >> 16));                             \
    }                                                                                               \
  } while (0)
      // the x dwords of the lane's four pairs, for both column tiles, from fa / fb
#define I8_NAT(out_)                                                                                \
  do {                                                                                              \
    _Pragma("unroll") for (int m = 0; m < 4; ++m)                                                   \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct)                                               \
      (out_)[ct][m] = (int)((uint32_t)__double_as_longlong(fma(fa[m][ct], fb[m][ct], kI8Magic)) ^ 0x80808080u); \
  } while (0)
      // one step, software-pipelined over three steps: the next step's x dwords
      // (VALU) and the LDS reads of the step after it are interleaved with this
      // step's 5 x RT x CT products, so that the VALU work runs beside the
      // matrix cores
#define I8_STEP(slot, next2_slot)                                                                   \
  do {                                                                                              \
    I8_NAT(nat[((slot) + 1) & 1]);                                                                  \
    I8_LDS(rc[next2_slot]);                                                                         \
    _Pragma("unroll") for (int ct = 0; ct < CT; ++ct) {                                             \
      const bu4 u3_ = __builtin_bit_cast(bu4, nat[(slot) & 1][ct]);                                 \
      const bi4 x2_ = __builtin_bit_cast(bi4, u3_ >> 8u);                                           \
      const bi4 x1_ = __builtin_bit_cast(bi4, u3_ >> 16u);                                          \
      const bi4 x0_ = __builtin_bit_cast(bi4, u3_ >> 24u);                                          \
      _Pragma("unroll") for (int rt = 0; rt < RT; ++rt) {                                           \
        acc[3][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1[slot][rt], nat[(slot) & 1][ct], acc[3][rt][ct], 0, 0, 0); \
        acc[4][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r2[slot][rt], nat[(slot) & 1][ct], acc[4][rt][ct], 0, 0, 0); \
        acc[2][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1[slot][rt], x2_, acc[2][rt][ct], 0, 0, 0); \
        acc[1][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1[slot][rt], x1_, acc[1][rt][ct], 0, 0, 0); \
        acc[0][rt][ct] = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1[slot][rt], x0_, acc[0][rt][ct], 0, 0, 0); \
      }                                                                                             \
    }                                                                                               \
    /* interleave: one product per three VALU instructions, then the DS reads */                   \
    _Pragma("unroll") for (int g_ = 0; g_ < 5 * RT * CT; ++g_) {                                    \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                            \
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);                                            \
    }                                                                                               \
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);                                              \
  } while (0)
      for (int j = 0; j < nb; ++j) {
        // this block's staging has landed (a full ring of loads was issued after
        // it), and the previous block's LDS reads are done, so its buffers are free
        __builtin_amdgcn_s_waitcnt(i8_vmcnt(kSlotLoads * kI8Ring));
        __builtin_amdgcn_s_waitcnt(kI8LgkmZero);
        int pa_n = pa, pb_n = pb;
        if (j + 1 < nb) {
          if (nxt.xc != (pa ? tag_a1 : tag_a0)) {
            pa_n = (nxt.xc == (pa ? tag_a0 : tag_a1)) ? 1 - pa : -1;
            if (pa_n < 0) {
              pa_n = 1 - pa;
              stage_rows(nxt.xc, s_f[wave][0][pa_n]);
              if (pa_n) tag_a1 = nxt.xc; else tag_a0 = nxt.xc;
            }
          }
          if (nxt.yc != (pb ? tag_b1 : tag_b0)) {
            pb_n = (nxt.yc == (pb ? tag_b0 : tag_b1)) ? 1 - pb : -1;
            if (pb_n < 0) {
              pb_n = 1 - pb;
              stage_rows(nxt.yc, s_f[wave][1][pb_n]);
              if (pb_n) tag_b1 = nxt.yc; else tag_b0 = nxt.yc;
            }
          }
          stage_scales(nxt, (j + 1) & 1);
        }
        const Hdr nn = header(bq);
        bq = blist[min(j + 3, nb - 1)];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int k = 0; k < 5; ++k) acc[k][rt][ct] = izero;
        la_lane = s_f[wave][0][pa] + jj * 16;
        lb_lane = s_f[wave][1][pb] + jj * 16;
        const int nst = max(cur.nst, 1);
        I8_LDS(rc[0]);
        I8_NAT(nat[0]);
        I8_LDS(rc[1 % kI8Ring]);
        // every slot loads once per pass (the count of loads in flight is the
        // same on every path); past the block's end a slot loads the next
        // block's step of its own number (again, on the last partial pass).
        // The passes whose steps and loads all lie in this block come first,
        // without a per-step test or a choice of block
        int st = 0;
        {
          const __amdgpu_buffer_rsrc_t RA = ring_rsrc(cur.A), RC = ring_rsrc(cur.C);
          for (const int sA = kI8Ring * (nst / kI8Ring - 1); st < sA; st += kI8Ring) {
#pragma unroll
            for (int u = 0; u < kI8Ring; ++u) {
              I8_STEP(u, (u + 2) % kI8Ring);
              I8_LOAD_R(u, RA, RC, st + u + kI8Ring);
            }
          }
        }
        for (; st < nst; st += kI8Ring) {
#pragma unroll
          for (int u = 0; u < kI8Ring; ++u) {
            if (st + u < nst) I8_STEP(u, (u + 2) % kI8Ring);
            const int s_ = st + u + kI8Ring;
            const bool in_ = s_ < nst;
            I8_LOAD(u, in_ ? cur.A : nxt.A, in_ ? cur.C : nxt.C, in_ ? s_ : u);
          }
        }
        // the block's exact sums, combined and scaled into the FP64 running sums
        {
          const int par = j & 1;
          double sA[RT][4], sF[CT];
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) sA[rt][e] = s_sa[wave][par][16 * rt + 4 * kk + e];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
            sF[ct] = ldexp(1.0, s_fe[wave][par][2 * jj + ct] + s_fe[wave][par][32 + 2 * jj + ct] - 2 * kI8FS);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                double v = (double)acc[0][rt][ct][e];
                v = fma(v, 256.0, (double)acc[1][rt][ct][e]);
                v = fma(v, 256.0, (double)acc[2][rt][ct][e]);
                v = fma(v, 256.0, (double)acc[3][rt][ct][e]);
                v = fma(v, 256.0, (double)acc[4][rt][ct][e]);
                tot[rt][ct][e] = fma(v, sA[rt][e] * sF[ct], tot[rt][ct][e]);
              }
        }
        cur = nxt;
        nxt = nn;
        pa = pa_n;
        pb = pb_n;
      }
#undef I8_STEP
#undef I8_NAT
#undef I8_LDS
#undef I8_LOAD
#undef I8_LOAD_R
    }
    if (it.parts > 1) {   // the shares' sums, added by the first share's waves of the chunk
      // (every staged row has been waited for, so a wave's own buffers are free)
      static_assert(sizeof(s_f[0]) >= sizeof(double) * 64 * RT * CT * 4, "the staged rows make room for the sums");
      auto at = [&](int w, int rt, int ct, int e) -> double* {
        return reinterpret_cast<double*>(&s_f[w][0][0][0]) + ((rt * CT + ct) * 4 + e) * 64 + lane;
      };
      if (part > 0) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) *at(wave, rt, ct, e) = tot[rt][ct][e];
      }
      __syncthreads();
      if (part > 0) continue;
      for (int p = 1; p < it.parts; ++p)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int e = 0; e < 4; ++e) tot[rt][ct][e] += *at(wave + p * it.nvc * WPC, rt, ct, e);
    }
    if (!active) continue;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        double* out = partial + (it.prow + 64 * vc + lcol + ct) * D;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int l = 16 * rt + 4 * kk + e;   // int32 16x16 output: row 4 (lane / 16) + e
          if (l < D) out[l] = tot[rt][ct][e];
        }
      }
  }
}

// One wave per (grid, cell, chunk): lane v sums its instance's rows over the
// cell's items in order, Q = (2 s) / w * scale, written to the packed layout.
template <int D>
__global__ __launch_bounds__(64) void k_batch_reduce(int64_t ntask, const int32_t* __restrict__ key,
                                                     const int64_t* __restrict__ ptr,
                                                     const int32_t* __restrict__ rows,
                                                     const BatchGridDev* __restrict__ grids,
                                                     const double* __restrict__ partial, double scale,
                                                     double* __restrict__ q) {
  const int64_t t = blockIdx.x;
  if (t >= ntask) return;
  const int lane = threadIdx.x;
  const int g = key[3 * t], c = key[3 * t + 1], vc = key[3 * t + 2];
  const BatchGridDev G = grids[g];
  double s[D];
#pragma unroll
  for (int l = 0; l < D; ++l) s[l] = 0.0;
  for (int64_t k = ptr[t]; k < ptr[t + 1]; ++k) {
    const double* row = partial + ((int64_t)rows[k] + lane) * D;
#pragma unroll
    for (int l = 0; l < D; ++l) s[l] = s[l] + row[l];
  }
  const int64_t v = (int64_t)vc * 64 + lane;
  double* Q = q + G.foff;
#pragma unroll
  for (int l = 0; l < D; ++l) {
    const int64_t node = (int64_t)c * D + l;
    double x = (2.0 * s[l]) / G.gwts[node];
    if (scale != 1.0) x = x * scale;
    Q[node * G.Bpad + v] = x;
  }
}

// FP64 on the merged layout: persistent workgroups of four waves, an item = one
// cell's quad blocks of one run for 32 instances.  The columns of quad_walk are
// instances: a staged row is 256 contiguous bytes of the packed f.  An item is walked
// kQuadWalk blocks (up to about 3072 steps) at a time and the walks' sums are added, as the pair-block
// kernel adds block sums: in one chain of matrix-core sums the error grows with the run.  15^3 nodes, error
// against extended precision by pairs per run 16 K / 256 K / 1 M: one chain 6e-16 / 3.8e-15 / 2e-14,
// walks of 4 blocks 5 / 4 / 8e-16, of 16 5 / 6 / 6e-16; the pair-block kernel 7e-16 / 1.1e-15 / 1.6e-15.
// A walk's start and its sums cost 1 % (256 VDFs on 27^3 nodes 1154 -> 1165 ms).
template <int D>
constexpr int kQuadWalk = 3072 / (D * D / 4);
template <int D>
__global__ __launch_bounds__(256, 2) void k_quad_batch(const BatchItem* __restrict__ items, const QueueBounds QB,
                                                       const BatchGridDev* __restrict__ grids,
                                                       const double* __restrict__ f, double* __restrict__ partial,
                                                       int* __restrict__ counter, const int32_t* __restrict__ nin) {
  constexpr int NW = 4, NI = (D + 1) / 2, SL = 8 / NW, RT = (D + 15) / 16;
  __shared__ __attribute__((aligned(16))) double lf[quad_rows<D>() * kQuadRow];
  __shared__ int s_item;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int odd = lane >> 5, col = lane & 31;
  for (int i = threadIdx.x; i < kQuadRow; i += 64 * NW) lf[8 * D * kQuadRow + i] = 0.0;
  int q = blockIdx.x % kQueues, left = kQueues;   // this workgroup's XCD queue first
  for (;;) {
    if (threadIdx.x == 0) s_item = take_item(counter, QB, q, left);
    __syncthreads();
    const int id = __builtin_amdgcn_readfirstlane(s_item);
    __syncthreads();
    if (id < 0) return;
    const BatchItem& it = items[id];
    const BatchGridDev& G = grids[it.grid];
    const int Mv = G.Mv, Mw = G.Mw, cell = it.cell, ncols = min(kQuadCols, nin[it.grid] - it.vc0 * kQuadCols);
    const int32_t* list = G.blist + it.b0;
    const QuadBlk* blocks = G.qblocks;
    const uint32_t sp = (uint32_t)G.Bpad * 8;
    const double* F = f + G.foff + (int64_t)it.vc0 * kQuadCols;
    // rows odd, odd + 2, ... of the lane's column (with an odd D the last round's odd
    // lanes repeat the last row)
    const uint32_t goff = (uint32_t)odd * sp + (uint32_t)col * 8, glast = D % 2 ? (uint32_t)col * 8 : goff;
    const uint32_t loff = (uint32_t)(odd * kQuadRow + col) * 8, llast = D % 2 ? (uint32_t)col * 8 : loff;
    double v[SL][NI];
    auto fetch = [&](const QuadBlk& B) {
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        const int slot = wave + NW * k;
        if (slot & B.same) continue;   // the cell of a lower slot: its rows are used
        const int du = slot & 1 ? B.b[0] : B.a[0], dv = slot & 2 ? B.b[1] : B.a[1], dw = slot & 4 ? B.b[2] : B.a[2];
        const __amdgpu_buffer_rsrc_t R = ring_rsrc(F + (int64_t)(cell + (du * Mv + dv) * Mw + dw) * D * (sp / 8));
#pragma unroll
        for (int i = 0; i < NI; ++i) v[k][i] = ring_f64(R, i + 1 < NI ? goff : glast, (uint32_t)(2 * i) * sp);
      }
    };
    auto store = [&](const QuadBlk& B) {
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        const int slot = wave + NW * k;
        if (slot & B.same) continue;
        char* dst = reinterpret_cast<char*>(lf) + slot * D * kQuadRow * 8;
#pragma unroll
        for (int i = 0; i < NI; ++i)
          *reinterpret_cast<double*>(dst + (i + 1 < NI ? loff : llast) + 2 * i * kQuadRow * 8) = v[k][i];
      }
    };
    const int n = it.b1 - it.b0;
    auto walk = [&](auto ct) {
      constexpr int CT = decltype(ct)::value;
      for (int i0 = 0; i0 < n; i0 += kQuadWalk<D>) {
        auto header = [&](int i) { return blocks[list[i0 + i]]; };
        qd4 acc[RT][CT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[rt][c] = qd4{0.0, 0.0, 0.0, 0.0};
        quad_walk<D, false, NW, CT>(min(kQuadWalk<D>, n - i0), header(0), 0, INT_MAX, G.qsteps, lf, lf, header, fetch,
                                    store, acc);
        quad_flush<D, NW, CT>(lf, acc, ncols, partial + it.prow * D, i0 > 0);
      }
    };
    if (ncols > 16) walk(std::integral_constant<int, 2>{});
    else walk(std::integral_constant<int, 1>{});
  }
}

// One workgroup per (grid, cell, chunk of 32 instances): the items' partial rows in
// item order (contiguous reads), Q = (2 s) / w * scale to the packed layout.
template <int D>
__global__ __launch_bounds__(256) void k_quad_batch_reduce(const int32_t* __restrict__ key,
                                                           const int64_t* __restrict__ ptr,
                                                           const int32_t* __restrict__ rows,
                                                           const BatchGridDev* __restrict__ grids,
                                                           const int32_t* __restrict__ nin,
                                                           const double* __restrict__ partial, double scale,
                                                           double* __restrict__ q) {
  constexpr int NE = (kQuadCols * D + 255) / 256;
  __shared__ double t[kQuadCols * D];
  const int64_t task = blockIdx.x;
  const int g = key[3 * task], c = key[3 * task + 1], v0 = key[3 * task + 2] * kQuadCols;
  const BatchGridDev& G = grids[g];
  const int ncols = min(kQuadCols, nin[g] - v0);
  double s[NE];
#pragma unroll
  for (int i = 0; i < NE; ++i) s[i] = 0.0;
  for (int64_t k = ptr[task]; k < ptr[task + 1]; ++k) {
    const double* row = partial + (int64_t)rows[k] * D;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = (int)threadIdx.x + 256 * i;
      if (e < ncols * D) s[i] += row[e];
    }
  }
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int e = (int)threadIdx.x + 256 * i;
    if (e < ncols * D) t[e] = s[i];
  }
  __syncthreads();
  double* Q = q + G.foff + v0;
  for (int e = threadIdx.x; e < kQuadCols * D; e += 256) {
    const int l = e / kQuadCols, col = e % kQuadCols;
    if (col >= ncols) continue;
    const int64_t node = (int64_t)c * D + l;
    double x = (2.0 * t[col * D + l]) / G.gwts[node];
    if (scale != 1.0) x = x * scale;
    Q[node * G.Bpad + col] = x;
  }
}

// out = t0 + t1 + ... over the packed buffers (as k_lincomb)
struct BLinTerm {
  const double* x;
  double m1, den;
  int neg;
};
struct BLinComb {
  BLinTerm t[5];
  int n;
};
__global__ void k_blincomb(int64_t n, double* __restrict__ out, BLinComb c) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) {
    double s = 0.0;
    for (int k = 0; k < c.n; ++k) {
      double v = c.t[k].x[i];
      if (c.t[k].m1 != 1.0) v = v * c.t[k].m1;
      if (c.t[k].den != 1.0) v = v / c.t[k].den;
      if (k == 0) s = c.t[k].neg ? -v : v;
      else s = c.t[k].neg ? s - v : s + v;
    }
    out[i] = s;
  }
}

// FP64 projection of every instance's Q onto the complement of the collision
// invariants psi = 1,u,v,w,|u|^2 in the w-weighted inner product.  One block of
// 16 waves per (grid, chunk of 64 instances): lane = instance, wave k sums the
// moments over its share of the nodes, the shares are added in wave order, and
// each lane solves G lam = m with the grid's Cholesky factor and applies it.
__global__ __launch_bounds__(1024) void k_batch_project(const BatchProjGrid* __restrict__ grids,
                                                        const int32_t* __restrict__ task, double* __restrict__ q) {
  __shared__ double part[16][5][64];
  const int g = task[2 * blockIdx.x], vc = task[2 * blockIdx.x + 1];
  const BatchProjGrid G = grids[g];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int inst = vc * 64 + lane;
  double* Q = q + G.foff + inst;
  const int64_t per = (G.N + 15) / 16;
  const int64_t i0 = wave * per, i1 = min(G.N, i0 + per);
  double s[5] = {0, 0, 0, 0, 0};
  for (int64_t i = i0; i < i1; ++i) {
    const double x = G.gw[i] * Q[i * G.Bpad];
    const double uu = G.u[i], vv = G.v[i], ww = G.w[i];
    s[0] += x;
    s[1] += x * uu;
    s[2] += x * vv;
    s[3] += x * ww;
    s[4] += x * (uu * uu + vv * vv + ww * ww);
  }
  for (int k = 0; k < 5; ++k) part[wave][k][lane] = s[k];
  __syncthreads();
  double lam[5];
  {
    double m[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      double a = 0.0;
      for (int wv = 0; wv < 16; ++wv) a += part[wv][k][lane];
      m[k] = a;
    }
    double y[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      double a = m[i];
#pragma unroll
      for (int k = 0; k < i; ++k) a -= G.L[i * 5 + k] * y[k];
      y[i] = a / G.L[i * 5 + i];
    }
#pragma unroll
    for (int i = 4; i >= 0; --i) {
      double a = y[i];
#pragma unroll
      for (int k = i + 1; k < 5; ++k) a -= G.L[k * 5 + i] * lam[k];
      lam[i] = a / G.L[i * 5 + i];
    }
  }
  if (inst >= G.nin) return;
  for (int64_t i = i0; i < i1; ++i) {
    const double uu = G.u[i], vv = G.v[i], ww = G.w[i];
    Q[i * G.Bpad] = Q[i * G.Bpad] - (lam[0] + lam[1] * uu + lam[2] * vv + lam[3] * ww +
                                     lam[4] * (uu * uu + vv * vv + ww * ww));
  }
}

// rows [count][ld] <-> packed instances (node * stride + first + r), 64 x 64 tiles
__global__ __launch_bounds__(256) void k_rows_pack(double* __restrict__ rows, int64_t ld, int count, int64_t N,
                                                   double* __restrict__ packed, int64_t stride, int to_packed) {
  __shared__ double tile[64][65];
  const int64_t n0 = (int64_t)blockIdx.x * 64;
  const int r0 = blockIdx.y * 64;
  const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
  if (to_packed) {
    for (int i = 0; i < 16; ++i) {
      const int r = r0 + rg + 4 * i;
      const int64_t n = n0 + c;
      tile[rg + 4 * i][c] = (r < count && n < N) ? rows[(int64_t)r * ld + n] : 0.0;
    }
    __syncthreads();
    for (int i = 0; i < 16; ++i) {
      const int64_t n = n0 + rg + 4 * i;
      const int r = r0 + c;
      if (n < N && r < count) packed[n * stride + r] = tile[c][rg + 4 * i];
    }
  } else {
    for (int i = 0; i < 16; ++i) {
      const int64_t n = n0 + rg + 4 * i;
      const int r = r0 + c;
      tile[rg + 4 * i][c] = (n < N && r < count) ? packed[n * stride + r] : 0.0;
    }
    __syncthreads();
    for (int i = 0; i < 16; ++i) {
      const int r = r0 + rg + 4 * i;
      const int64_t n = n0 + c;
      if (r < count && n < N) rows[(int64_t)r * ld + n] = tile[c][rg + 4 * i];
    }
  }
}

static void destroy_plan(dgv_batch* b, BatchPlan& P) {
  hipFree(P.d_items); hipFree(P.d_partial); hipFree(P.d_red_rows); hipFree(P.d_red_ptr); hipFree(P.d_red_key);
  P.d_items = nullptr; P.d_partial = nullptr; P.d_red_rows = nullptr; P.d_red_ptr = nullptr; P.d_red_key = nullptr;
  P.items.clear();
  P.ready = false;
  P.nrows = 0;
  P.nred = 0;
  if (&P == &b->plan && b->graph) { hipGraphExecDestroy(b->graph); b->graph = nullptr; }
}

static int chunks_of_item(const dgv_batch* b) {   // chunks per item of the batch's kernel
  const bool fp32 = b->precision == DGV_FP32_COMP || b->precision == DGV_FP32_F64ACC;
  return b->quad ? 1 : fp32 ? chunks_per_item<true>() : chunks_per_item<false>();   // INT8_SPLIT: as FP64
}
static int shares_of_item(const dgv_batch* b, int nvc) {   // shares of an item of nvc chunks
  return b->quad || b->precision == DGV_FP64 ? 1 : chunks_of_item(b) / nvc;
}

// The run of each of a grid's quad blocks, in their own order, cut at about `tile` pairs
static std::vector<int32_t> quad_runs(const dgv_ctx* ctx, int32_t tile) {
  const QuadLayout& L = ctx->quad;
  const double per_step = (double)ctx->pb.npairs / (double)std::max<int64_t>(L.nsteps, 1);
  std::vector<int32_t> run(L.blocks.size());
  double acc = 0;
  int32_t r = 0;
  for (size_t k = 0; k < L.blocks.size(); ++k) {
    run[k] = r;
    acc += L.blocks[k].nst * per_step;
    if (acc >= tile) { ++r; acc = 0; }
  }
  return run;
}

// A merged batch's partial rows with such runs
static int64_t quad_nrows(const dgv_batch* b, int32_t tile, const std::vector<int32_t>* cells) {
  int64_t rows = 0;
  for (size_t g = 0; g < b->grids.size(); ++g) {
    if (b->nin[g] == 0) continue;
    const std::vector<int32_t> run = quad_runs(b->grids[g], tile);
    const std::vector<int64_t>& cp = b->cell_ptr[g];
    const std::vector<int32_t>& bl = b->h_blist[g];
    int64_t segs = 0;
    auto add = [&](int64_t c) {
      for (int64_t k = cp[c]; k < cp[c + 1]; ++k) segs += k + 1 == cp[c + 1] || run[bl[k + 1]] != run[bl[k]];
    };
    if (cells) {
      for (int32_t c : *cells)
        if (c >= 0 && c < b->grids[g]->g.ncells) add(c);
    } else {
      for (int64_t c = 0; c < b->grids[g]->g.ncells; ++c) add(c);
    }
    rows += segs * ((b->nin[g] + kQuadCols - 1) / kQuadCols) * kQuadCols;
  }
  return rows;
}

// Pairs per run.  Merged batch: about 2048 steps (2 MB of coefficients, shared
// through one XCD's 4 MB L2 by the cells running on it), less where a small batch
// would not give each of the 512 workgroups four items; but, up to 1 M pairs, as many as
// keep the partial sums within a quarter of the coefficients' bytes, pair blocks and
// merged rows, or 1 GB (256 VDFs on 27^3 nodes: 1165 ms and 25 GB with 2048 steps, 1160 ms
// with 64 K to 256 K pairs, there 4 GB, 1164 with 512 K, 1176 with 1 M).
// Otherwise: 4096 pairs for each wave of an item, which keeps the runs of the
// cells on one XCD close enough together to meet in L2 (27^3 nodes, 64 instances
// INT8_SPLIT: 479 ms with 1 M pairs a run, 375 with 64 K; 256 instances FP32: 1478
// and 1434), down to 1024 where the 512 workgroups would get fewer than three
// items each (9^3 nodes, 64 instances, INT8_SPLIT: 2.29 ms with one item per cell, 0.22
// with 8 K pairs a run, 0.30 with 2 K; 15^3 nodes, 256 instances, FP32: 59 ms with 1 M,
// 13.7 with 16 K, 15.0 with 2 K); but no more partial sums than a quarter of the
// coefficients' bytes or 1 GB, and at most 1 M pairs.
static int32_t auto_tile(const dgv_batch* b, const std::vector<int32_t>* cells) {
  if (!b->quad) {
    const int D = b->grids[0]->g.D;
    const int chpi = chunks_of_item(b);
    const double coef = b->precision == DGV_INT8_SPLIT ? 128.0 * ((D + 15) / 16) : b->precision == DGV_FP64 ? 8.0 * (D + 1) : 4.0 * (D + 2);
    // walk: pairs walked by the waves of all items; whole: the same if every block held every cell
    double walk = 0, whole = 0, bytes = 0, rows = 0;
    for (size_t g = 0; g < b->grids.size(); ++g) {
      if (b->nin[g] == 0) continue;
      const auto& pb = b->grids[g]->pb;
      const std::vector<int64_t>& cp = b->cell_ptr[g];
      const std::vector<int32_t>& bl = b->h_blist[g];
      double listed = 0, ncells = 0;
      auto add = [&](int64_t c) {
        ++ncells;
        for (int64_t k = cp[c]; k < cp[c + 1]; ++k) listed += pb.blocks[bl[k]].npairs;
      };
      if (cells) {
        for (int32_t c : *cells)
          if (c >= 0 && c < b->grids[g]->g.ncells) add(c);
      } else {
        for (int64_t c = 0; c < b->grids[g]->g.ncells; ++c) add(c);
      }
      const int nchunk = b->Bpad[g] / 64;
      for (int vc0 = 0; vc0 < nchunk; vc0 += chpi) {
        walk += listed / shares_of_item(b, std::min(chpi, nchunk - vc0));
        whole += ncells * (double)pb.npairs;
      }
      rows += 64.0 * nchunk * listed;   // rows times tile
      bytes += coef * (double)pb.npairs;
    }
    if (walk <= 0) return 1 << 20;
    const double per_wave = std::min(4096.0, std::max(1024.0, walk / (3 * 512.0)));
    // a cell's part of a run is about twice its share of the pairs: blocks near in
    // order lie near in space (27^3 nodes: 297 K items of 64 K pairs, 9.1e9 pairs walked)
    const double fit = 2 * rows * D * 8 / std::max(1e9, bytes / 4);
    return (int32_t)std::min(1048576.0, std::max(per_wave * whole / walk, fit));
  }
  double pairs = 0, steps = 0, items = 0;   // items: (cell, chunk) walks of a whole array
  for (size_t g = 0; g < b->grids.size(); ++g) {
    if (b->nin[g] == 0) continue;
    pairs += (double)b->grids[g]->pb.npairs;
    steps += (double)b->grids[g]->quad.nsteps;
    items += (double)(cells ? (int64_t)cells->size() : b->grids[g]->g.ncells) * ((b->nin[g] + kQuadCols - 1) / kQuadCols);
  }
  const double per_walk = steps / std::max<double>(1, (double)b->grids.size());
  const double runs = std::max(per_walk / 2048.0, 4.0 * 512.0 / std::max(items, 1.0));
  double tile = std::min(1e9, std::max(256.0, pairs / std::max<double>(1, (double)b->grids.size()) / std::max(runs, 1.0)));
  const int D = b->grids[0]->g.D;
  const double most = std::max(1e9, (pairs * (D + 1) * 8 + steps * (D * 32 + 64)) / 4);
  while (tile < (1 << 20)) {   // the rows fall about as the runs grow
    const double over = (double)quad_nrows(b, (int32_t)tile, cells) * D * 8 / most;
    if (over <= 1) break;
    tile = std::min(1048576.0, tile * std::max(1.1, over));
  }
  return (int32_t)tile;
}

// Per cell and grid: blocks whose box contains the cell, cut into segments;
// items = segments x chunks of 64 instances.  Segments are global: the grid's
// blocks in (a, b) order -- the order of every cell's list -- are cut into runs
// of about `tile` pairs, and a cell's segment k is its blocks in run k.  The
// items of one run for different cells then walk the same blocks in the same
// order, and run side by side (the queue is ordered by run, then cell), so
// the coefficient records of a block are fetched from memory once and served
// from L2 to the items running with it.  With `cells` given, only those cells
// (of every grid) are planned.
static int build_batch_plan(dgv_batch* b, BatchPlan& P, int32_t tile, const std::vector<int32_t>* cells = nullptr) {
  if (int rc = batch_check_grids(b)) return rc;
  destroy_plan(b, P);
  const bool automatic = tile <= 0;
  if (automatic) tile = auto_tile(b, cells);
  P.tile = tile;
  std::vector<BatchItem> items;
  int64_t nrows = 0;
  std::vector<int32_t> key;
  std::vector<int64_t> rptr(1, 0);
  std::vector<int32_t> rrows;
  std::vector<std::vector<int32_t>> run_of(b->grids.size());   // per grid: the run of each block
  for (size_t gi = 0; gi < b->grids.size(); ++gi) {
    if (b->nin[gi] == 0) continue;
    const dgv_ctx* ctx = b->grids[gi];
    const PairBlock& pb = ctx->pb;
    const std::vector<int64_t>& cp = b->cell_ptr[gi];
    const std::vector<int32_t>& blist = b->h_blist[gi];
    const int nchunk = b->quad ? (b->nin[gi] + kQuadCols - 1) / kQuadCols : b->Bpad[gi] / 64;
    if (b->quad) {
      run_of[gi] = quad_runs(ctx, tile);
    } else {
      std::vector<int32_t> order(pb.blocks.size());
      std::iota(order.begin(), order.end(), 0);
      std::sort(order.begin(), order.end(), [&](int32_t x, int32_t y) {
        const BlockHdr &X = pb.blocks[x], &Y = pb.blocks[y];
        for (int d = 0; d < 3; ++d) if (X.a[d] != Y.a[d]) return X.a[d] < Y.a[d];
        for (int d = 0; d < 3; ++d) if (X.b[d] != Y.b[d]) return X.b[d] < Y.b[d];
        return x < y;
      });
      run_of[gi].assign(pb.blocks.size(), 0);
      int64_t acc = 0;
      int32_t run = 0;
      for (int32_t k : order) {
        run_of[gi][k] = run;
        acc += pb.blocks[k].npairs;
        if (acc >= tile) { ++run; acc = 0; }
      }
    }
    const std::vector<int32_t>& run = run_of[gi];
    std::vector<int64_t> todo;
    if (cells) {
      for (int32_t c : *cells)
        if (c >= 0 && c < ctx->g.ncells) todo.push_back(c);
    } else {
      for (int64_t c = 0; c < ctx->g.ncells; ++c) todo.push_back(c);
    }
    for (int64_t c : todo) {
      std::vector<std::pair<int32_t, int32_t>> segs;
      int64_t s0 = cp[c];
      for (int64_t k = cp[c]; k < cp[c + 1]; ++k)
        if (k + 1 == cp[c + 1] || run[blist[k + 1]] != run[blist[k]]) {
          segs.push_back({(int32_t)s0, (int32_t)(k + 1)});
          s0 = k + 1;
        }
      const int chpi = chunks_of_item(b);
      const int width = b->quad ? kQuadCols : 64;
      for (int vc0 = 0; vc0 < nchunk; vc0 += chpi) {
        const int nvc = std::min(chpi, nchunk - vc0);
        const int parts = shares_of_item(b, nvc);
        std::vector<int64_t> first;   // first partial row of each segment's item
        for (auto& sg : segs) {
          BatchItem it{};
          it.grid = (int32_t)gi; it.cell = (int32_t)c; it.b0 = sg.first; it.b1 = sg.second;
          it.vc0 = vc0; it.nvc = nvc;
          it.prow = nrows;
          it.parts = parts;
          it.cut[0] = it.b0;
          it.cut[parts] = it.b1;
          if (parts > 1) {
            int64_t all = 0, acc = 0;
            for (int32_t k = it.b0; k < it.b1; ++k) all += pb.blocks[blist[k]].npairs;
            int p = 1;
            for (int32_t k = it.b0; k < it.b1 && p < parts; ++k) {
              acc += pb.blocks[blist[k]].npairs;
              while (p < parts && acc * parts >= all * p) it.cut[p++] = k + 1;
            }
            for (; p < parts; ++p) it.cut[p] = it.b1;
          }
          nrows += width * nvc;
          if (nrows > INT32_MAX) return berr(b, DGV_ERR_UNSUPPORTED, "too many batch work items");
          first.push_back(it.prow);
          items.push_back(it);
        }
        for (int k = 0; k < nvc; ++k) {
          key.push_back((int32_t)gi); key.push_back((int32_t)c); key.push_back(vc0 + k);
          for (int64_t r : first) rrows.push_back((int32_t)(r + width * k));
          rptr.push_back((int64_t)rrows.size());
        }
      }
    }
  }
  const int D = b->grids[0]->g.D;
  // keep the partial sums within 32 GiB: coarser segments otherwise
  if (nrows * D * 8 > ((int64_t)32 << 30) && tile < (1 << 30))
    return build_batch_plan(b, P, tile * 2, cells);
  // Execution order: by the item's run of blocks, then by cell.  Items that run
  // at the same time then stream the same coefficient records for different
  // cells (shared through L2); each item keeps its partial-sum rows, so the
  // reduction order does not depend on the execution order.
  {
    std::vector<int64_t> key1(items.size());
    for (size_t i = 0; i < items.size(); ++i) {
      const BatchItem& it = items[i];
      key1[i] = ((int64_t)it.grid << 40) | ((int64_t)run_of[it.grid][b->h_blist[it.grid][it.b0]] << 8);
    }
    std::vector<size_t> order(items.size());
    std::iota(order.begin(), order.end(), (size_t)0);
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
      if (key1[x] != key1[y]) return key1[x] < key1[y];
      return items[x].cell < items[y].cell;
    });
    std::vector<BatchItem> sorted(items.size());
    for (size_t i = 0; i < order.size(); ++i) sorted[i] = items[order[i]];
    items.swap(sorted);
    // whole runs to eight queues, each run to the queue with the fewest items
    // so far; a queue keeps its runs in order
    for (int q = 0; q <= kQueues; ++q) P.queues.beg[q] = (int32_t)items.size();
    if (!items.empty()) {
      std::vector<std::vector<BatchItem>> qs(kQueues);
      std::vector<int64_t> load(kQueues, 0);
      for (size_t i = 0; i < items.size();) {
        size_t j = i;
        const int64_t k = key1[order[i]];
        while (j < items.size() && key1[order[j]] == k) ++j;
        const int q = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        qs[q].insert(qs[q].end(), items.begin() + i, items.begin() + j);
        load[q] += (int64_t)(j - i);
        i = j;
      }
      items.clear();
      for (int q = 0; q < kQueues; ++q) {
        P.queues.beg[q] = (int32_t)items.size();
        items.insert(items.end(), qs[q].begin(), qs[q].end());
      }
      P.queues.beg[kQueues] = (int32_t)items.size();
    }
  }
  P.items.swap(items);
  P.nrows = nrows;
  P.nred = (int64_t)rptr.size() - 1;
  BHIP(b, hipMalloc(&P.d_items, sizeof(BatchItem) * std::max<size_t>(P.items.size(), 1)));
  BHIP(b, hipMemcpy(P.d_items, P.items.data(), sizeof(BatchItem) * P.items.size(), hipMemcpyHostToDevice));
  if (hipMalloc(&P.d_partial, sizeof(double) * std::max<int64_t>(P.nrows * D, 1)) != hipSuccess) {
    P.d_partial = nullptr;
    (void)hipGetLastError();
    if (automatic && tile < (1 << 20)) return build_batch_plan(b, P, 1 << 20, cells);   // the fewest rows
  }
  if (!P.d_partial)
    return berr(b, DGV_ERR_NOMEM, "hipMalloc(batch partial sums) failed");
  BHIP(b, hipMalloc(&P.d_red_rows, sizeof(int32_t) * std::max<size_t>(rrows.size(), 1)));
  BHIP(b, hipMemcpy(P.d_red_rows, rrows.data(), sizeof(int32_t) * rrows.size(), hipMemcpyHostToDevice));
  BHIP(b, hipMalloc(&P.d_red_ptr, sizeof(int64_t) * rptr.size()));
  BHIP(b, hipMemcpy(P.d_red_ptr, rptr.data(), sizeof(int64_t) * rptr.size(), hipMemcpyHostToDevice));
  BHIP(b, hipMalloc(&P.d_red_key, sizeof(int32_t) * std::max<size_t>(key.size(), 1)));
  BHIP(b, hipMemcpy(P.d_red_key, key.data(), sizeof(int32_t) * key.size(), hipMemcpyHostToDevice));
  P.ready = true;
  return DGV_OK;
}

static int batch_eval_dev(dgv_batch* b, const BatchPlan& P, const double* d_f, double* d_q, double scale,
                          bool reduce = true) {
  if (int rc = batch_check_grids(b)) return rc;
  if (!P.ready) return berr(b, DGV_ERR_STATE, "no work plan: the call that last changed it failed");
  const int D = b->grids[0]->g.D;
  const int nitems = (int)P.items.size();
  hipStream_t st = b->stream;
  if (b->precision == DGV_FP32_COMP || b->precision == DGV_FP32_F64ACC)
    hipLaunchKernelGGL(k_to_f32, dim3(stride_blocks(b->total, 256)), dim3(256), 0, st, b->total, d_f, b->d_f32);
  if (b->precision == DGV_INT8_SPLIT)
    for (size_t g = 0; g < b->grids.size(); ++g) {
      const int64_t nc = b->grids[g]->g.ncells;
      const int64_t n = nc * b->Bpad[g];
      if (n == 0) continue;
      const double* F = d_f + b->foff[g];
      double* Fh = b->d_fhat + b->foff[g];
      int32_t* E = b->d_fexp + b->foff[g] / D;
      if (D == 27)
        hipLaunchKernelGGL(k_i8_fixed<27>, dim3(stride_blocks(n, 256)), dim3(256), 0, st, nc, b->Bpad[g], F, Fh, E);
      else
        hipLaunchKernelGGL(k_i8_fixed<8>, dim3(stride_blocks(n, 256)), dim3(256), 0, st, nc, b->Bpad[g], F, Fh, E);
    }
  hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(64), 0, st, b->d_counter);
  // workgroups of four waves; waves_per_cu sets the persistent grid's size
  const int wpc = b->waves_per_cu > 0 ? b->waves_per_cu : 8;
  const unsigned nwg = (unsigned)std::max(1, std::min(nitems, b->ncu * wpc / kWavesPerItem));
  if (nitems > 0) {
    const dim3 blk(64 * kWavesPerItem);
#define DGV_BATCH_LAUNCH(DD, MM)                                                                          \
  hipLaunchKernelGGL((k_batch_mfma<DD, MM>), dim3(nwg), blk, 0, st, P.d_items, P.queues, b->d_grids, d_f, \
                     b->d_f32, P.d_partial, b->d_counter)
    if (b->quad) {
      if (D == 27)
        hipLaunchKernelGGL(k_quad_batch<27>, dim3(nwg), blk, 0, st, P.d_items, P.queues, b->d_grids, d_f,
                           P.d_partial, b->d_counter, b->d_nin);
      else
        hipLaunchKernelGGL(k_quad_batch<8>, dim3(nwg), blk, 0, st, P.d_items, P.queues, b->d_grids, d_f,
                           P.d_partial, b->d_counter, b->d_nin);
    } else if (b->precision == DGV_INT8_SPLIT) {
      if (D == 27)
        hipLaunchKernelGGL(k_batch_i8<27>, dim3(nwg), blk, 0, st, P.d_items, P.queues, b->d_grids, b->d_fhat,
                           b->d_fexp, P.d_partial, b->d_counter);
      else
        hipLaunchKernelGGL(k_batch_i8<8>, dim3(nwg), blk, 0, st, P.d_items, P.queues, b->d_grids, b->d_fhat,
                           b->d_fexp, P.d_partial, b->d_counter);
    } else if (D == 27) {
      if (b->precision == DGV_FP32_COMP) DGV_BATCH_LAUNCH(27, DGV_FP32_COMP);
      else if (b->precision == DGV_FP32_F64ACC) DGV_BATCH_LAUNCH(27, DGV_FP32_F64ACC);
      else DGV_BATCH_LAUNCH(27, DGV_FP64);
    } else {
      if (b->precision == DGV_FP32_COMP) DGV_BATCH_LAUNCH(8, DGV_FP32_COMP);
      else if (b->precision == DGV_FP32_F64ACC) DGV_BATCH_LAUNCH(8, DGV_FP32_F64ACC);
      else DGV_BATCH_LAUNCH(8, DGV_FP64);
    }
#undef DGV_BATCH_LAUNCH
  }
  if (reduce && P.nred > 0 && b->quad) {
    if (D == 27)
      hipLaunchKernelGGL(k_quad_batch_reduce<27>, dim3((unsigned)P.nred), dim3(256), 0, st, P.d_red_key, P.d_red_ptr,
                         P.d_red_rows, b->d_grids, b->d_nin, P.d_partial, scale, d_q);
    else
      hipLaunchKernelGGL(k_quad_batch_reduce<8>, dim3((unsigned)P.nred), dim3(256), 0, st, P.d_red_key, P.d_red_ptr,
                         P.d_red_rows, b->d_grids, b->d_nin, P.d_partial, scale, d_q);
  } else if (reduce && P.nred > 0) {
    if (D == 27)
      hipLaunchKernelGGL(k_batch_reduce<27>, dim3((unsigned)P.nred), dim3(64), 0, st, P.nred, P.d_red_key,
                         P.d_red_ptr, P.d_red_rows, b->d_grids, P.d_partial, scale, d_q);
    else
      hipLaunchKernelGGL(k_batch_reduce<8>, dim3((unsigned)P.nred), dim3(64), 0, st, P.nred, P.d_red_key,
                         P.d_red_ptr, P.d_red_rows, b->d_grids, P.d_partial, scale, d_q);
  }
  if (reduce && b->project && b->nproj_task > 0 && &P == &b->plan)
    hipLaunchKernelGGL(k_batch_project, dim3((unsigned)b->nproj_task), dim3(1024), 0, st, b->d_proj, b->d_proj_task,
                       d_q);
  BHIP(b, hipGetLastError());
  return DGV_OK;
}

static int blincomb(dgv_batch* b, double* out, int n, const double* const* xs, const double* m1, const double* den,
                    const int* neg) {
  BLinComb c;
  std::memset(&c, 0, sizeof(c));
  c.n = n;
  for (int k = 0; k < n; ++k) { c.t[k].x = xs[k]; c.t[k].m1 = m1[k]; c.t[k].den = den[k]; c.t[k].neg = neg[k]; }
  hipLaunchKernelGGL(k_blincomb, dim3(stride_blocks(b->total, 256)), dim3(256), 0, b->stream, b->total, out, c);
  BHIP(b, hipGetLastError());
  return DGV_OK;
}

// One Runge-Kutta step (rkmts 1..3) of every instance, the reference's
// combinations (time_integr_mod.f90:37-83) on the packed buffers.
static int batch_rk_step(dgv_batch* b, double dt, double coef, int rkmts) {
  double *f = b->d_f, *k1 = b->d_tmp[0], *k2 = b->d_tmp[1], *k3 = b->d_tmp[2], *tmp = b->d_tmp[3];
  const double ct = coef * dt;
  int rc;
#define BSOP(in, out) do { rc = batch_eval_dev(b, b->plan, in, out, ct); if (rc) return rc; } while (0)
  switch (rkmts) {
    case 1: {
      BSOP(f, k1);
      const double* x[] = {f, k1}; double m[] = {1, 1}, d[] = {1, 1}; int ng[] = {0, 0};
      return blincomb(b, f, 2, x, m, d, ng);
    }
    case 2: {
      BSOP(f, k1);
      { const double* x[] = {f, k1}; double m[] = {1, 2}, d[] = {1, 3.0}; int ng[] = {0, 0};
        if ((rc = blincomb(b, tmp, 2, x, m, d, ng))) return rc; }
      BSOP(tmp, k2);
      const double* x[] = {f, k1, k2}; double m[] = {1, 1, 3.0}, d[] = {1, 4.0, 4}; int ng[] = {0, 0, 0};
      return blincomb(b, f, 3, x, m, d, ng);
    }
    case 3: {
      BSOP(f, k1);
      { const double* x[] = {f, k1}; double m[] = {1, 1}, d[] = {1, 2.0}; int ng[] = {0, 0};
        if ((rc = blincomb(b, tmp, 2, x, m, d, ng))) return rc; }
      BSOP(tmp, k2);
      { const double* x[] = {f, k2}; double m[] = {1, 3.0}, d[] = {1, 4}; int ng[] = {0, 0};
        if ((rc = blincomb(b, tmp, 2, x, m, d, ng))) return rc; }
      BSOP(tmp, k3);
      const double* x[] = {f, k1, k2, k3}; double m[] = {1, 2, 3.0, 4}, d[] = {1, 9.0, 9.0, 9.0};
      int ng[] = {0, 0, 0, 0};
      return blincomb(b, f, 4, x, m, d, ng);
    }
  }
#undef BSOP
  return berr(b, DGV_ERR_ARG, "batched stepping supports rkmts 1..3");
}

}  // namespace dgv

using namespace dgv;

extern "C" {

int dgv_batch_create(dgv_ctx* const* grids, int32_t ngrids, const int32_t* grid_of_instance, int32_t ninstances,
                     int32_t precision, dgv_batch** out) {
  if (!out || !grids || ngrids < 1 || !grid_of_instance || ninstances < 1) {
    set_global_error("dgv_batch_create: bad argument");
    return DGV_ERR_ARG;
  }
  *out = nullptr;
  if (precision != DGV_FP64 && precision != DGV_FP32_COMP && precision != DGV_FP32_F64ACC &&
      precision != DGV_INT8_SPLIT) {
    set_global_error("precision must be DGV_FP64, DGV_FP32_COMP, DGV_FP32_F64ACC or DGV_INT8_SPLIT");
    return DGV_ERR_ARG;
  }
  const int D = grids[0] ? grids[0]->g.D : 0;
  for (int g = 0; g < ngrids; ++g) {
    if (!grids[g] || !grids[g]->has_a) { set_global_error("every grid needs an A-array"); return DGV_ERR_STATE; }
    if (grids[g]->g.D != D || (D != 27 && D != 8)) {
      set_global_error("batched evaluation needs 8 or 27 nodes per cell on every grid");
      return DGV_ERR_UNSUPPORTED;
    }
    if (grids[g]->device != grids[0]->device) { set_global_error("all grids must be on one device"); return DGV_ERR_ARG; }
  }
  dgv_batch* b = new dgv_batch();
  b->grids.assign(grids, grids + ngrids);
  for (int g = 0; g < ngrids; ++g) b->a_gen.push_back(grids[g]->a_gen);
  b->device = grids[0]->device;
  b->precision = precision;
  b->quad = precision == DGV_FP64;
  for (int g = 0; g < ngrids; ++g) b->quad = b->quad && grids[g]->quad.use;
  b->ninst = ninstances;
  b->nin.assign(ngrids, 0);
  b->inst_grid.resize(ninstances);
  b->inst_local.resize(ninstances);
  for (int i = 0; i < ninstances; ++i) {
    const int g = grid_of_instance[i];
    if (g < 0 || g >= ngrids) { delete b; set_global_error("grid_of_instance out of range"); return DGV_ERR_ARG; }
    b->inst_grid[i] = g;
    b->inst_local[i] = b->nin[g]++;
  }
  b->Bpad.resize(ngrids);
  b->foff.resize(ngrids);
  int64_t off = 0;
  for (int g = 0; g < ngrids; ++g) {
    b->Bpad[g] = ((b->nin[g] + 63) / 64) * 64;
    b->foff[g] = off;
    off += grids[g]->g.N * (int64_t)b->Bpad[g];
  }
  b->total = off;
  auto fail = [&](int code, const std::string& m) {
    dgv_batch_destroy(b);
    set_global_error(m);
    if (code == DGV_ERR_NOMEM) (void)hipGetLastError();   // the failed hipMalloc's sticky error
    return code;
  };
  if (hipSetDevice(grids[0]->device) != hipSuccess) return fail(DGV_ERR_HIP, "hipSetDevice failed");
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, grids[0]->device) == hipSuccess) b->ncu = prop.multiProcessorCount;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return fail(DGV_ERR_HIP, "stream");
  for (int i = 0; i < 3; ++i)
    if (hipEventCreate(&b->ev[i]) != hipSuccess) return fail(DGV_ERR_HIP, "event");
  const size_t nb = sizeof(double) * std::max<int64_t>(b->total, 1);
  if (hipMalloc(&b->d_f, nb) || hipMalloc(&b->d_q, nb)) return fail(DGV_ERR_NOMEM, "hipMalloc(batch buffers)");
  for (int i = 0; i < 4; ++i)
    if (hipMalloc(&b->d_tmp[i], nb)) return fail(DGV_ERR_NOMEM, "hipMalloc(batch buffers)");
  if (hipMemsetAsync(b->d_f, 0, nb, b->stream) || hipMemsetAsync(b->d_q, 0, nb, b->stream))
    return fail(DGV_ERR_HIP, "hipMemset");
  const bool fp32 = precision == DGV_FP32_COMP || precision == DGV_FP32_F64ACC;
  const bool i8 = precision == DGV_INT8_SPLIT;
  if (fp32 && hipMalloc(&b->d_f32, sizeof(float) * std::max<int64_t>(b->total, 1)))
    return fail(DGV_ERR_NOMEM, "hipMalloc(FP32 buffers)");
  if (i8 && (hipMalloc(&b->d_fhat, nb) || hipMalloc(&b->d_fexp, sizeof(int32_t) * std::max<int64_t>(b->total / D, 1))))
    return fail(DGV_ERR_NOMEM, "hipMalloc(fixed-point buffers)");
  if (hipMalloc(&b->d_counter, sizeof(int) * kQueues)) return fail(DGV_ERR_NOMEM, "hipMalloc(counter)");
  if (hipMalloc(&b->d_nin, sizeof(int32_t) * ngrids) ||
      hipMemcpy(b->d_nin, b->nin.data(), sizeof(int32_t) * ngrids, hipMemcpyHostToDevice))
    return fail(DGV_ERR_NOMEM, "hipMalloc(instance counts)");
  {
    int64_t nmax = 1;
    for (int g = 0; g < ngrids; ++g) nmax = std::max<int64_t>(nmax, grids[g]->g.N);
    if (hipMalloc(&b->d_stage, sizeof(double) * nmax)) return fail(DGV_ERR_NOMEM, "hipMalloc(staging)");
  }
  // per grid: per-cell block lists, FP32 coefficients
  std::vector<BatchGridDev> gd(ngrids);
  b->d_blist.assign(ngrids, nullptr);
  b->d_pairs32.assign(ngrids, nullptr);
  b->d_i8.assign(ngrids, {nullptr, nullptr, nullptr, nullptr});
  b->cell_ptr.assign(ngrids, {});
  b->h_blist.assign(ngrids, {});
  for (int g = 0; g < ngrids; ++g) {
    const dgv_ctx* ctx = grids[g];
    const PairBlock& pb = ctx->pb;
    std::vector<int64_t> cnt(ctx->g.ncells + 1, 0);
    const std::vector<Group>& groups = b->quad ? ctx->quad.groups : pb.groups;
    for (const Group& G : groups)
      for (int r = 0; r < G.ncells; ++r) {
        int rr = r;
        const int cw = G.lo[2] + rr % G.ext[2]; rr /= G.ext[2];
        const int cv = G.lo[1] + rr % G.ext[1]; rr /= G.ext[1];
        const int cu = G.lo[0] + rr;
        cnt[((int64_t)cu * ctx->g.Mv + cv) * ctx->g.Mw + cw + 1] += G.bend - G.bbeg;
      }
    for (int64_t c = 0; c < ctx->g.ncells; ++c) cnt[c + 1] += cnt[c];
    std::vector<int32_t> blist(cnt.back());
    std::vector<int64_t> pos(cnt.begin(), cnt.end() - 1);
    for (const Group& G : groups)
      for (int r = 0; r < G.ncells; ++r) {
        int rr = r;
        const int cw = G.lo[2] + rr % G.ext[2]; rr /= G.ext[2];
        const int cv = G.lo[1] + rr % G.ext[1]; rr /= G.ext[1];
        const int cu = G.lo[0] + rr;
        const int64_t cell = ((int64_t)cu * ctx->g.Mv + cv) * ctx->g.Mw + cw;
        for (int k = G.bbeg; k < G.bend; ++k) blist[pos[cell]++] = b->quad ? k : pb.group_blocks[k];
      }
    // each cell's blocks ordered by (a, b): runs of equal a share the staged f[c + a]
    // (quad blocks keep their own order)
    for (int64_t c = 0; c < ctx->g.ncells && !b->quad; ++c)
      std::sort(blist.begin() + cnt[c], blist.begin() + cnt[c + 1], [&](int32_t x, int32_t y) {
        const BlockHdr &X = pb.blocks[x], &Y = pb.blocks[y];
        for (int d = 0; d < 3; ++d) if (X.a[d] != Y.a[d]) return X.a[d] < Y.a[d];
        for (int d = 0; d < 3; ++d) if (X.b[d] != Y.b[d]) return X.b[d] < Y.b[d];
        return x < y;
      });
    b->cell_ptr[g] = cnt;
    if (hipMalloc(&b->d_blist[g], sizeof(int32_t) * std::max<size_t>(blist.size(), 1)) ||
        hipMemcpy(b->d_blist[g], blist.data(), sizeof(int32_t) * blist.size(), hipMemcpyHostToDevice))
      return fail(DGV_ERR_NOMEM, "block lists");
    b->h_blist[g] = blist;
    if (i8) {
      // blocks padded to multiples of 16 pairs, in block order
      std::vector<int64_t> p16(pb.blocks.size());
      int64_t tot16 = 0;
      for (size_t k = 0; k < pb.blocks.size(); ++k) {
        p16[k] = tot16;
        tot16 += (pb.blocks[k].npairs + 15) & ~15;
      }
      const int RT = (D + 15) / 16;
      const int64_t dw = (int64_t)RT * 32;   // digit dwords per pair
      auto& a = b->d_i8[g];
      const int64_t pad16 = 16 * kI8Ring;    // the ring reads up to kI8Ring steps past a block
      if (hipMalloc(&a[0], sizeof(uint32_t) * (tot16 + pad16) * dw) ||
          hipMalloc(&a[1], sizeof(uint32_t) * (tot16 + pad16)) ||
          hipMalloc(&a[2], sizeof(double) * 16 * RT * std::max<size_t>(pb.blocks.size(), 1)) ||
          hipMalloc(&a[3], sizeof(int64_t) * std::max<size_t>(p16.size(), 1)))
        return fail(DGV_ERR_NOMEM, "hipMalloc(INT8_SPLIT coefficient digits)");
      if (hipMemcpy(a[3], p16.data(), sizeof(int64_t) * p16.size(), hipMemcpyHostToDevice))
        return fail(DGV_ERR_HIP, "hipMemcpy(block starts)");
      if (hipMemsetAsync((uint32_t*)a[0] + tot16 * dw, 0, sizeof(uint32_t) * pad16 * dw, b->stream) ||
          hipMemsetAsync((uint32_t*)a[1] + tot16, 0, sizeof(uint32_t) * pad16, b->stream))
        return fail(DGV_ERR_HIP, "hipMemsetAsync(digit padding)");
      if (!pb.blocks.empty()) {
        if (D == 27)
          hipLaunchKernelGGL(k_i8_digits<27>, dim3((unsigned)pb.blocks.size()), dim3(256), 0, b->stream, pb.d_blocks,
                             (const int64_t*)a[3], pb.d_pairs, (uint32_t*)a[0], (uint32_t*)a[1], (double*)a[2]);
        else
          hipLaunchKernelGGL(k_i8_digits<8>, dim3((unsigned)pb.blocks.size()), dim3(256), 0, b->stream, pb.d_blocks,
                             (const int64_t*)a[3], pb.d_pairs, (uint32_t*)a[0], (uint32_t*)a[1], (double*)a[2]);
        if (hipGetLastError() != hipSuccess) return fail(DGV_ERR_HIP, "INT8_SPLIT digit kernel launch");
      }
    }
    if (fp32) {
      // zero pairs past the end: the kernel's load ring reads up to 4 kRing + 3
      // pairs beyond a block without clamping
      const int64_t n = pb.npairs * (D + 2), pad = (int64_t)kPadPairs * (D + 2);
      if (hipMalloc(&b->d_pairs32[g], sizeof(float) * (n + pad)))
        return fail(DGV_ERR_NOMEM, "hipMalloc(FP32 coefficients)");
      if (n > 0)
        hipLaunchKernelGGL(k_pairs_to_f32, dim3(stride_blocks(n, 256)), dim3(256), 0, b->stream, pb.npairs, D,
                           pb.d_pairs, b->d_pairs32[g]);
      if (hipMemsetAsync(b->d_pairs32[g] + n, 0, sizeof(float) * pad, b->stream))
        return fail(DGV_ERR_HIP, "hipMemsetAsync(FP32 coefficient padding)");
    }
    gd[g].qblocks = ctx->quad.d_blocks;
    gd[g].qsteps = ctx->quad.d_steps;
    gd[g].pairs64 = pb.d_pairs;
    gd[g].pairs32 = b->d_pairs32[g];
    gd[g].blocks = pb.d_blocks;
    gd[g].blist = b->d_blist[g];
    gd[g].gwts = ctx->d_gwts;
    gd[g].digits = (const uint32_t*)b->d_i8[g][0];
    gd[g].codes = (const uint32_t*)b->d_i8[g][1];
    gd[g].bscale = (const double*)b->d_i8[g][2];
    gd[g].pbeg16 = (const int64_t*)b->d_i8[g][3];
    gd[g].foff = b->foff[g];
    gd[g].eoff = b->foff[g] / D;
    gd[g].Bpad = b->Bpad[g];
    gd[g].Mv = ctx->g.Mv;
    gd[g].Mw = ctx->g.Mw;
    gd[g].D = D;
  }
  {
    std::vector<BatchProjGrid> pg(ngrids);
    std::vector<int32_t> task;
    for (int g = 0; g < ngrids; ++g) {
      const dgv_ctx* ctx = grids[g];
      pg[g].u = ctx->d_u; pg[g].v = ctx->d_v; pg[g].w = ctx->d_w; pg[g].gw = ctx->d_gwts;
      if (gram_cholesky(ctx->g, pg[g].L)) return fail(DGV_ERR_GRID, "Gram matrix of the invariants is singular");
      pg[g].foff = b->foff[g];
      pg[g].N = ctx->g.N;
      pg[g].Bpad = b->Bpad[g];
      pg[g].nin = b->nin[g];
      for (int vc = 0; vc < b->Bpad[g] / 64; ++vc) { task.push_back(g); task.push_back(vc); }
    }
    b->nproj_task = (int32_t)(task.size() / 2);
    if (hipMalloc(&b->d_proj, sizeof(BatchProjGrid) * ngrids) ||
        hipMemcpy(b->d_proj, pg.data(), sizeof(BatchProjGrid) * ngrids, hipMemcpyHostToDevice) ||
        hipMalloc(&b->d_proj_task, sizeof(int32_t) * std::max<size_t>(task.size(), 2)) ||
        hipMemcpy(b->d_proj_task, task.data(), sizeof(int32_t) * task.size(), hipMemcpyHostToDevice))
      return fail(DGV_ERR_HIP, "projection tables");
  }
  if (hipMalloc(&b->d_grids, sizeof(BatchGridDev) * ngrids) ||
      hipMemcpy(b->d_grids, gd.data(), sizeof(BatchGridDev) * ngrids, hipMemcpyHostToDevice))
    return fail(DGV_ERR_HIP, "grid table");
  if (hipStreamSynchronize(b->stream) != hipSuccess) return fail(DGV_ERR_HIP, "coefficient conversion");
  int rc = build_batch_plan(b, b->plan, 0);
  if (rc) { std::string m = b->err; dgv_batch_destroy(b); set_global_error(m); return rc; }
  *out = b;
  return DGV_OK;
}

void dgv_batch_destroy(dgv_batch* b) {
  if (!b) return;
  hipSetDevice(b->device);
  if (b->stream) hipStreamSynchronize(b->stream);
  destroy_plan(b, b->plan);
  destroy_plan(b, b->probe);
  hipFree(b->d_f); hipFree(b->d_q); hipFree(b->d_f32); hipFree(b->d_counter); hipFree(b->d_nin); hipFree(b->d_grids);
  hipFree(b->d_proj); hipFree(b->d_proj_task); hipFree(b->d_stage);
  for (int i = 0; i < 4; ++i) hipFree(b->d_tmp[i]);
  for (auto p : b->d_blist) hipFree(p);
  for (auto p : b->d_pairs32) hipFree(p);
  for (auto& a : b->d_i8)
    for (void* p : a) hipFree(p);
  hipFree(b->d_fhat); hipFree(b->d_fexp);
  for (int i = 0; i < 3; ++i)
    if (b->ev[i]) hipEventDestroy(b->ev[i]);
  if (b->stream) hipStreamDestroy(b->stream);
  delete b;
}

int dgv_batch_layout(const dgv_batch* b, int32_t instance, int64_t* offset, int64_t* stride, int64_t* total) {
  if (!b || instance < 0 || instance >= b->ninst) { set_global_error("bad batch or instance"); return DGV_ERR_ARG; }
  const int g = b->inst_grid[instance];
  if (offset) *offset = b->foff[g] + b->inst_local[instance];
  if (stride) *stride = b->Bpad[g];
  if (total) *total = b->total;
  return DGV_OK;
}

// One instance from / to a host array: a contiguous copy through a staging
// buffer and the row pack kernel (a 2-D copy of 8-byte rows would be slow).
static int batch_copy(dgv_batch* b, int32_t instance, double* host, int64_t n, bool to_device, double* dev) {
  if (!b || instance < 0 || instance >= b->ninst || !host) { set_global_error("bad argument"); return DGV_ERR_ARG; }
  const int g = b->inst_grid[instance];
  const int64_t N = b->grids[g]->g.N;
  if (n != N) return berr(b, DGV_ERR_ARG, "array length differs from the instance's node count");
  BHIP(b, hipSetDevice(b->grids[0]->device));
  double* base = dev + b->foff[g] + b->inst_local[instance];
  const dim3 grid((unsigned)((N + 63) / 64), 1);
  if (to_device) {
    BHIP(b, hipMemcpyAsync(b->d_stage, host, sizeof(double) * N, hipMemcpyHostToDevice, b->stream));
    hipLaunchKernelGGL(k_rows_pack, grid, dim3(256), 0, b->stream, b->d_stage, N, 1, N, base, (int64_t)b->Bpad[g], 1);
    BHIP(b, hipGetLastError());
  } else {
    hipLaunchKernelGGL(k_rows_pack, grid, dim3(256), 0, b->stream, b->d_stage, N, 1, N, base, (int64_t)b->Bpad[g], 0);
    BHIP(b, hipGetLastError());
    BHIP(b, hipMemcpyAsync(host, b->d_stage, sizeof(double) * N, hipMemcpyDeviceToHost, b->stream));
  }
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_set_f(dgv_batch* b, int32_t instance, const double* f, int64_t n) {
  return batch_copy(b, instance, const_cast<double*>(f), n, true, b ? b->d_f : nullptr);
}

int dgv_batch_get_q(dgv_batch* b, int32_t instance, double* q, int64_t n) {
  return batch_copy(b, instance, q, n, false, b ? b->d_q : nullptr);
}

// instances first .. first + count - 1 (all on one grid) from / to device rows
static int batch_rows(dgv_batch* b, const double* d_rows, int64_t ld, int32_t first, int32_t count, bool to_packed,
                      double* packed) {
  if (!b || !d_rows || first < 0 || count < 1 || first + count > b->ninst) {
    set_global_error("bad batch row range");
    return DGV_ERR_ARG;
  }
  const int g = b->inst_grid[first];
  for (int32_t i = first; i < first + count; ++i)
    if (b->inst_grid[i] != g || b->inst_local[i] != b->inst_local[first] + (i - first))
      return berr(b, DGV_ERR_ARG, "row copies need consecutive instances of one grid");
  const int64_t N = b->grids[g]->g.N;
  if (ld < N) return berr(b, DGV_ERR_ARG, "leading dimension below the node count");
  BHIP(b, hipSetDevice(b->grids[0]->device));
  double* base = packed + b->foff[g] + b->inst_local[first];
  hipLaunchKernelGGL(k_rows_pack, dim3((unsigned)((N + 63) / 64), (unsigned)((count + 63) / 64)), dim3(256), 0,
                     b->stream, const_cast<double*>(d_rows), ld, count, N, base, (int64_t)b->Bpad[g],
                     to_packed ? 1 : 0);
  BHIP(b, hipGetLastError());
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_set_f_rows_dev(dgv_batch* b, const double* d_rows, int64_t ld, int32_t first, int32_t count) {
  return batch_rows(b, d_rows, ld, first, count, true, b ? b->d_f : nullptr);
}

int dgv_batch_get_q_rows_dev(dgv_batch* b, double* d_rows, int64_t ld, int32_t first, int32_t count) {
  return batch_rows(b, d_rows, ld, first, count, false, b ? b->d_q : nullptr);
}

int dgv_batch_get_f_rows_dev(dgv_batch* b, double* d_rows, int64_t ld, int32_t first, int32_t count) {
  return batch_rows(b, d_rows, ld, first, count, false, b ? b->d_f : nullptr);
}

int dgv_batch_eval_q(dgv_batch* b) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  int rc = batch_eval_dev(b, b->plan, b->d_f, b->d_q, 1.0);
  if (rc) return rc;
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_set_projection(dgv_batch* b, int32_t on) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  b->project = on ? 1 : 0;
  if (b->graph) { hipGraphExecDestroy(b->graph); b->graph = nullptr; }
  return DGV_OK;
}

int dgv_batch_set_tile(dgv_batch* b, int32_t pairs_per_segment, int32_t waves_per_cu) {
  if (!b || pairs_per_segment < 0 || waves_per_cu < 0) { set_global_error("bad argument"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  BHIP(b, hipStreamSynchronize(b->stream));
  if (waves_per_cu > 0) b->waves_per_cu = waves_per_cu;
  int rc = build_batch_plan(b, b->plan, pairs_per_segment);
  if (rc) return rc;
  if (!b->probe_cells.empty()) rc = build_batch_plan(b, b->probe, b->plan.tile, &b->probe_cells);
  return rc;
}

int dgv_batch_project_invariants(dgv_batch* b) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  if (b->nproj_task > 0)
    hipLaunchKernelGGL(k_batch_project, dim3((unsigned)b->nproj_task), dim3(1024), 0, b->stream, b->d_proj,
                       b->d_proj_task, b->d_q);
  BHIP(b, hipGetLastError());
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_set_probe_cells(dgv_batch* b, const int32_t* cells, int32_t ncells) {
  if (!b || ncells < 0 || (ncells > 0 && !cells)) { set_global_error("bad argument"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  BHIP(b, hipStreamSynchronize(b->stream));
  b->probe_cells.assign(cells, cells + ncells);
  std::sort(b->probe_cells.begin(), b->probe_cells.end());
  b->probe_cells.erase(std::unique(b->probe_cells.begin(), b->probe_cells.end()), b->probe_cells.end());
  for (int32_t c : b->probe_cells)
    for (const dgv_ctx* g : b->grids)
      if (c < 0 || c >= g->g.ncells) return berr(b, DGV_ERR_INDEX, "probe cell outside a grid");
  if (ncells == 0) { destroy_plan(b, b->probe); return DGV_OK; }
  return build_batch_plan(b, b->probe, b->plan.tile, &b->probe_cells);
}

int dgv_batch_eval_q_probe(dgv_batch* b) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  if (b->probe.items.empty()) return berr(b, DGV_ERR_STATE, "no probe cells set");
  BHIP(b, hipSetDevice(b->grids[0]->device));
  int rc = batch_eval_dev(b, b->probe, b->d_f, b->d_q, 1.0);
  if (rc) return rc;
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_rk_run(dgv_batch* b, double dt, double coef, int32_t rkmts, int64_t nsteps, int use_graph) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  if (rkmts < 1 || rkmts > 3) return berr(b, DGV_ERR_ARG, "batched stepping supports rkmts 1..3");
  if (int rc = batch_check_grids(b)) return rc;   // a graph replay would not pass batch_eval_dev
  BHIP(b, hipSetDevice(b->grids[0]->device));
  if (!use_graph) {
    for (int64_t s = 0; s < nsteps; ++s) {
      int rc = batch_rk_step(b, dt, coef, rkmts);
      if (rc) return rc;
    }
    BHIP(b, hipStreamSynchronize(b->stream));
    return DGV_OK;
  }
  const bool same = b->graph && b->graph_key[0] == rkmts && b->graph_key[1] == b->plan.tile && b->graph_dt == dt &&
                    b->graph_coef == coef;
  if (!same) {
    if (b->graph) { hipGraphExecDestroy(b->graph); b->graph = nullptr; }
    hipGraph_t graph;
    BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    int rc = batch_rk_step(b, dt, coef, rkmts);
    hipError_t e = hipStreamEndCapture(b->stream, &graph);
    if (rc) return rc;
    if (e != hipSuccess) return berr(b, DGV_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&b->graph, graph, nullptr, nullptr, 0);
    hipGraphDestroy(graph);
    if (e != hipSuccess) return berr(b, DGV_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    b->graph_key[0] = rkmts;
    b->graph_key[1] = b->plan.tile;
    b->graph_dt = dt;
    b->graph_coef = coef;
  }
  for (int64_t s = 0; s < nsteps; ++s) BHIP(b, hipGraphLaunch(b->graph, b->stream));
  BHIP(b, hipStreamSynchronize(b->stream));
  return DGV_OK;
}

int dgv_batch_time_eval(dgv_batch* b, int32_t niter, double* ms_per_call, double* ms_main_kernel) {
  if (!b || niter < 1) { set_global_error("bad argument"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  BHIP(b, hipEventRecord(b->ev[0], b->stream));
  for (int i = 0; i < niter; ++i) {
    int rc = batch_eval_dev(b, b->plan, b->d_f, b->d_q, 1.0);
    if (rc) return rc;
  }
  BHIP(b, hipEventRecord(b->ev[1], b->stream));
  // the persistent main kernel alone (with its FP32 conversion and queue reset)
  for (int i = 0; i < niter && ms_main_kernel; ++i) {
    int rc = batch_eval_dev(b, b->plan, b->d_f, b->d_q, 1.0, false);
    if (rc) return rc;
  }
  BHIP(b, hipEventRecord(b->ev[2], b->stream));
  BHIP(b, hipEventSynchronize(b->ev[2]));
  float a = 0, m = 0;
  BHIP(b, hipEventElapsedTime(&a, b->ev[0], b->ev[1]));
  BHIP(b, hipEventElapsedTime(&m, b->ev[1], b->ev[2]));
  if (ms_per_call) *ms_per_call = a / niter;
  if (ms_main_kernel) *ms_main_kernel = m / niter;
  return DGV_OK;
}

int dgv_batch_merged(const dgv_batch* b, int32_t* merged) {
  if (!b || !merged) { set_global_error("null argument"); return DGV_ERR_ARG; }
  *merged = b->quad ? 1 : 0;
  return DGV_OK;
}

int dgv_batch_autotune(dgv_batch* b, int32_t* best, double* best_ms) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  BHIP(b, hipSetDevice(b->grids[0]->device));
  // small segments suit the INT8 kernel (16 K pairs: 2 % faster than 256 K at
  // 27^3), large ones the FP64 kernel; a candidate whose plan cannot be built
  // (too many work items) is skipped
  const int32_t tiles[] = {1 << 14, 1 << 15, 1 << 16, 1 << 17, 1 << 18, 1 << 19, 1 << 20, 1 << 21};
  const int32_t wpcs[] = {4, 8};
  int32_t bt = 0, bw = 0;
  double bms = 1e300;
  bool warm = false;
  for (int32_t t : tiles) {
    int rc = build_batch_plan(b, b->plan, t);
    if (rc == DGV_ERR_UNSUPPORTED) continue;
    if (rc) return rc;
    for (int32_t w : wpcs) {
      b->waves_per_cu = w;
      double ms;
      if (!warm) {
        if ((rc = batch_eval_dev(b, b->plan, b->d_f, b->d_q, 1.0))) return rc;
        warm = true;
      }
      rc = dgv_batch_time_eval(b, 1, &ms, nullptr);
      if (rc) return rc;
      if (ms < bms) { bms = ms; bt = t; bw = w; }
    }
  }
  if (bt == 0) return berr(b, DGV_ERR_UNSUPPORTED, "autotune: no segment size gives a plan");
  b->waves_per_cu = bw;
  int rc = build_batch_plan(b, b->plan, bt);
  if (rc) return rc;
  if (!b->probe_cells.empty() && (rc = build_batch_plan(b, b->probe, bt, &b->probe_cells))) return rc;
  if (best) *best = bt;
  if (best_ms) *best_ms = bms;
  return DGV_OK;
}

int dgv_batch_device_buffers(dgv_batch* b, double** d_f, double** d_q) {
  if (!b) { set_global_error("null batch"); return DGV_ERR_ARG; }
  if (d_f) *d_f = b->d_f;
  if (d_q) *d_q = b->d_q;
  return DGV_OK;
}

}  // extern "C"
