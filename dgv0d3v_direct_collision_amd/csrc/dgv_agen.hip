// dgv_agen.hip -- GPU generator of the A-array (SetA_DGV, dgvtools_mod.f90:377-681)
// for all canonical basis functions at once, written directly in the
// pair-block layout.
//
// Two nodes are opposite corners of a box of grid nodes; the box's four diagonals
// share midpoint and distance, hence the sphere and its integrals S_l, the costly
// part.  Every box is integrated once, for its main diagonal (the pair whose xi has
// the lower coordinate in every dimension), and serves its up to four pairs.
//
// Pipeline (cp = ordered cell pair X <= Y in the reference's cell order):
//   1. k_count   : per cp, pairs (xi in X, xi1 in Y, xi < xi1) passing the
//                  prefilter of lines 493-530, and main diagonals among them
//   2. host scan -> offsets; k_list writes the list of main diagonals, the pairs'
//                  (p, q) and each cp's table (p, q) -> pair
//   3. k_integrate: one thread per main diagonal, S_l (dgv_agen_math.h), then for
//                  each pair of the box the D values of A: min_sens test, weights
//                  and |g|/8                                             -> pairs;
//                  k_integrate_marked the few spheres whose records hang on rounding
//   4. k_kept + host scan + k_compact: drop pairs whose D values are all zero and
//                  emit per-cp segment tables (the block headers)
#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <numeric>

#include "dgv_agen_math.h"
#include "dgv_internal.h"

namespace dgv {

static void lagrange_monomials(const double* kap, int n, double mono[kAgenMaxS][kAgenMaxS]) {
  for (int i = 0; i < kAgenMaxS; ++i)
    for (int m = 0; m < kAgenMaxS; ++m) mono[i][m] = 0.0;
  for (int i = 0; i < n; ++i) {
    double c[kAgenMaxS + 1] = {1.0};
    int deg = 0;
    for (int j = 0; j < n; ++j) {
      if (j == i) continue;
      // multiply by (kap[j] - y) / (kap[j] - kap[i])
      const double den = kap[j] - kap[i];
      double nc[kAgenMaxS + 1] = {0};
      for (int m = 0; m <= deg; ++m) {
        nc[m] += c[m] * kap[j] / den;
        nc[m + 1] += -c[m] / den;
      }
      ++deg;
      for (int m = 0; m <= deg; ++m) c[m] = nc[m];
    }
    for (int m = 0; m < n; ++m) mono[i][m] = c[m];
  }
}

static int make_consts(const Grid& g, const dgv_agen_params& p, AgenConsts& C, std::string& err) {
  std::memset(&C, 0, sizeof(C));
  if (g.su > kAgenMaxS || g.sv > kAgenMaxS || g.sw > kAgenMaxS) {
    err = "A-array generator supports at most 4 nodes per cell per dimension";
    return DGV_ERR_UNSUPPORTED;
  }
  C.su = g.su; C.sv = g.sv; C.sw = g.sw;
  const int cc = g.ccell;
  C.u0 = g.lu[cc]; C.u1 = g.ru[cc]; C.v0 = g.lv[cc]; C.v1 = g.rv[cc]; C.w0 = g.lw[cc]; C.w1 = g.rw[cc];
  const int s[3] = {g.su, g.sv, g.sw};
  for (int d = 0; d < 3; ++d) {
    for (int i = 0; i < s[d]; ++i) C.kap[d][i] = g.gn[d][i];
    lagrange_monomials(C.kap[d], s[d], C.mono[d]);
    if (d < 2) std::memcpy(C.monol[d], C.mono[d], sizeof(C.mono[d]));
    const double h = 0.5 * (d == 0 ? C.u1 - C.u0 : d == 1 ? C.v1 - C.v0 : C.w1 - C.w0);
    for (int i = 0; i < s[d]; ++i)
      for (int m = 1; m < s[d]; ++m) C.mono[d][i][m] /= std::pow(h, m);
  }
  int nq = p.nquad > 0 ? p.nquad : 24;
  if (nq > kAgenMaxQ) { err = "nquad too large (max 48)"; return DGV_ERR_ARG; }
  C.nq = nq;
  std::vector<double> x(nq), w(nq);
  if (gauss_legendre(nq, x.data(), w.data())) { err = "Gauss-Legendre failed"; return DGV_ERR_ARG; }
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int i = 0; i < nq; ++i) {
    C.qs[i] = 0.5 * (double)pi * (x[i] + 1.0);
    C.qv[i] = 0.5 * (double)pi * w[i];
    const long double a = 0.5L * pi * (1.0L + x[i]);
    C.qx[i] = (double)(1.0L - std::cos(a));
    C.qw[i] = (double)(0.5L * pi * w[i] * std::sin(a));
  }
  C.Trad = p.Trad > 0 ? p.Trad : 100.0;
  C.moment_mode = p.moment_mode;
  if (p.moment_mode < 0 || p.moment_mode > 5) { err = "moment_mode must be 0..5"; return DGV_ERR_ARG; }
  return DGV_OK;
}

template <int SU, int SV, int SW>
DGV_HD inline int pair_raw_dispatch(const AgenConsts& C, const double x[3], const double y[3], double* raw,
                                    double* dsph) {
  return pair_raw<SU, SV, SW>(C, x, y, raw, dsph);
}

static int pair_raw_host(const AgenConsts& C, const double x[3], const double y[3], double* raw, double* dsph) {
  if (C.su == 3 && C.sv == 3 && C.sw == 3) return pair_raw<3, 3, 3>(C, x, y, raw, dsph);
  if (C.su == 2 && C.sv == 2 && C.sw == 2) return pair_raw<2, 2, 2>(C, x, y, raw, dsph);
  if (C.su == 1 && C.sv == 1 && C.sw == 1) return pair_raw<1, 1, 1>(C, x, y, raw, dsph);
  if (C.su == 4 && C.sv == 4 && C.sw == 4) return pair_raw<4, 4, 4>(C, x, y, raw, dsph);
  return -2;
}

// ---------------------------------------------------------------------------
struct NodeGeo {
  const double *u, *v, *w, *gwts;
};
struct CellDims {
  int Mv, Mw;
  int64_t nc;
};

// (xi, xi1) = nodes (X, p), (Y, q): whether xi has the lower coordinate, or the same,
// in every dimension
template <int SU, int SV, int SW>
__device__ __forceinline__ bool main_diagonal(const CellDims& d, int2 XY, int p, int q) {
  const int xc[3] = {XY.x / (d.Mv * d.Mw), XY.x / d.Mw % d.Mv, XY.x % d.Mw};
  const int yc[3] = {XY.y / (d.Mv * d.Mw), XY.y / d.Mw % d.Mv, XY.y % d.Mw};
  const int xl[3] = {p / (SV * SW), p / SW % SV, p % SW}, yl[3] = {q / (SV * SW), q / SW % SV, q % SW};
  bool ok = true;
  for (int k = 0; k < 3; ++k) ok = ok && (xc[k] < yc[k] || (xc[k] == yc[k] && xl[k] <= yl[k]));
  return ok;
}

// Candidate c of a cell pair: the nodes p = c / D, q = c % D
template <int D>
__device__ __forceinline__ bool candidate(const AgenConsts& C, int2 XY, int c, const NodeGeo& G) {
  const int p = c / D, q = c - p * D;
  if (c >= D * D || (XY.x == XY.y && q <= p)) return false;
  const int64_t i = (int64_t)XY.x * D + p, j = (int64_t)XY.y * D + q;
  const double x[3] = {G.u[i], G.v[i], G.w[i]}, y[3] = {G.u[j], G.v[j], G.w[j]};
  return pair_distance(C, x, y) >= 0.0;
}

// One wave per cp in turn: cnt = its pairs and its main diagonals
template <int SU, int SV, int SW>
__global__ __launch_bounds__(64) void k_count(AgenConsts C, CellDims dims, int64_t ncp, const int2* __restrict__ cps,
                                              NodeGeo G, uint2* __restrict__ cnt) {
  constexpr int D = SU * SV * SW;
  for (int64_t cp = blockIdx.x; cp < ncp; cp += gridDim.x) {
    const int2 XY = cps[cp];
    uint32_t n = 0, m = 0;
    for (int c0 = 0; c0 < D * D; c0 += 64) {
      const int c = c0 + (int)threadIdx.x;
      const bool ok = candidate<D>(C, XY, c, G);
      const bool main = ok && main_diagonal<SU, SV, SW>(dims, XY, c / D, c % D);
      n += __popcll(__ballot(ok));
      m += __popcll(__ballot(main));
    }
    if (threadIdx.x == 0) cnt[cp] = make_uint2(n, m);
  }
}

// ... the pairs' codes p << 8 | q in (p, q) order, each candidate's rank among them
// (-1: no pair) and the main diagonals
template <int SU, int SV, int SW>
__global__ __launch_bounds__(64) void k_list(AgenConsts C, CellDims dims, int64_t ncp, const int2* __restrict__ cps,
                                             NodeGeo G, const int64_t* __restrict__ off,
                                             const int64_t* __restrict__ moff, uint16_t* __restrict__ code,
                                             int16_t* __restrict__ rank, uint64_t* __restrict__ mains) {
  constexpr int D = SU * SV * SW;
  const int lane = threadIdx.x;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  for (int64_t cp = blockIdx.x; cp < ncp; cp += gridDim.x) {
    const int2 XY = cps[cp];
    int n = 0;
    int64_t m = moff[cp];
    const int64_t o = off[cp];
    for (int c0 = 0; c0 < D * D; c0 += 64) {
      const int c = c0 + lane;
      const bool ok = candidate<D>(C, XY, c, G);
      const bool main = ok && main_diagonal<SU, SV, SW>(dims, XY, c / D, c % D);
      const uint64_t bo = __ballot(ok), bm = __ballot(main);
      const int r = n + __popcll(bo & below);
      if (c < D * D) rank[cp * (D * D) + c] = ok ? (int16_t)r : (int16_t)-1;
      if (ok) code[o + r] = (uint16_t)((c / D) << 8 | c % D);
      if (main) mains[m + __popcll(bm & below)] = ((uint64_t)cp << 16) | ((uint64_t)(c / D) << 8) | (uint64_t)(c % D);
      n += __popcll(bo);
      m += __popcll(bm);
    }
  }
}

// The spheres' inputs: main diagonal k of the list
// (kPointwise set in the entry: integrate it point by point)
constexpr uint64_t kPointwise = (uint64_t)1 << 63;
struct Mains {
  const int2* cps;
  uint64_t* list;
};
struct Main {
  int2 XY;
  int p, q;
  double cen[3], dsph;
};
template <int SU, int SV, int SW>
__device__ __forceinline__ Main main_of(const AgenConsts& C, const Mains& M, const NodeGeo& G, int64_t k) {
  constexpr int D = SU * SV * SW;
  Main m;
  const uint64_t e = M.list[k] & ~kPointwise;
  m.p = (int)((e >> 8) & 255);
  m.q = (int)(e & 255);
  m.XY = M.cps[e >> 16];
  const int64_t i0 = (int64_t)m.XY.x * D + m.p, j0 = (int64_t)m.XY.y * D + m.q;
  const double lo[3] = {G.u[i0], G.v[i0], G.w[i0]}, hi[3] = {G.u[j0], G.v[j0], G.w[j0]};
  m.dsph = pair_distance(C, lo, hi);
  for (int d = 0; d < 3; ++d) m.cen[d] = 0.5 * (lo[d] + hi[d]);
  return m;
}

// Diagonal z of a main diagonal's box, if it is one: the pair's D values of A.  Returns
// whether one of them is too close to the cutoff for its side of it to be certain.
struct PairsOut {
  const int64_t* off;
  const int16_t* rank;
  double min_sens;
  double* pairs;
  uint8_t* keep;
};
template <int SU, int SV, int SW>
__device__ __forceinline__ bool write_diagonal(const AgenConsts& C, const CellDims& dims, const NodeGeo& G, const PairsOut& O,
                                               const Main& m, const double* S, int z) {
  constexpr int D = SU * SV * SW;
  const int2 XY = m.XY;
  const int p = m.p, q = m.q;
  const double dsph = m.dsph;
  // the box's corners: cell and local coordinates of the low and the high one
  const int lc[3] = {XY.x / (dims.Mv * dims.Mw), XY.x / dims.Mw % dims.Mv, XY.x % dims.Mw};
  const int hc[3] = {XY.y / (dims.Mv * dims.Mw), XY.y / dims.Mw % dims.Mv, XY.y % dims.Mw};
  const int ll[3] = {p / (SV * SW), p / SW % SV, p % SW}, hl[3] = {q / (SV * SW), q / SW % SV, q % SW};
  int differ = 0;
  for (int d = 0; d < 3; ++d) differ |= (lc[d] != hc[d] || ll[d] != hl[d]) << d;
  const int flips = differ & (differ - 1);   // the first dimension that differs stays: each diagonal once
  if (z & ~flips) return false;
  int ac[3], al[3], bc[3], bl[3];   // the diagonal's ends: `a` takes the high corner where bit d of z is set
  for (int d = 0; d < 3; ++d) {
    const bool f = (z >> d) & 1;
    ac[d] = f ? hc[d] : lc[d]; al[d] = f ? hl[d] : ll[d];
    bc[d] = f ? lc[d] : hc[d]; bl[d] = f ? ll[d] : hl[d];
  }
  int X = (ac[0] * dims.Mv + ac[1]) * dims.Mw + ac[2], Y = (bc[0] * dims.Mv + bc[1]) * dims.Mw + bc[2];
  int P = (al[0] * SV + al[1]) * SW + al[2], Q = (bl[0] * SV + bl[1]) * SW + bl[2];
  if (X > Y || (X == Y && P > Q)) {   // xi < xi1 in node order
    const int t = X, u = P;
    X = Y; Y = t;
    P = Q; Q = u;
  }
  const int64_t cp = (int64_t)X * dims.nc - (int64_t)X * (X - 1) / 2 + (Y - X);
  const int64_t at = O.off[cp] + O.rank[cp * (D * D) + P * D + Q];
  const int64_t i = (int64_t)X * D + P, j = (int64_t)Y * D + Q;
  const double x[3] = {G.u[i], G.v[i], G.w[i]}, y[3] = {G.u[j], G.v[j], G.w[j]};
  double raw[D];
  if (C.moment_mode == 0) {
    raw_from_sphere<SU, SV, SW>(C, x, y, S, raw);
  } else {
    const double v = raw_moment(C.moment_mode, x, y, 0.5 * dsph);
    for (int l = 0; l < D; ++l) raw[l] = v;
  }
  const double wi = G.gwts[i], wj = G.gwts[j];
  double* out = O.pairs + at * (D + 1);
  bool any = false, near = false;
  for (int l = 0; l < D; ++l) {
    near = near || near_cutoff(raw[l], O.min_sens);
    double a = 0.0;
    if (fabs(raw[l]) > O.min_sens) {  // line 641, then lines 654-659
      a = raw[l] * wj;
      a = a * wi;
      a = a * (dsph / 8.0);
      any = true;
    }
    out[l] = a;
  }
  out[D] = __longlong_as_double((long long)pair_code_bits(P, Q));
  O.keep[at] = any ? 1 : 0;
  return near;
}

// One thread per main diagonal.  FP64 arithmetic bounds it: up to 19 smooth pieces of 24
// points, each with up to four crossed lines (an inverse sine, a square root and the
// antiderivatives each).  26 ms at 15^3 nodes (0.86 M spheres, 3.2 M pairs) with the arcs
// searched, and their ends' sines and cosines taken, at every point; 3.6 ms (and 1.2 for
// the marked ones) with the arcs' ends known per piece.
// Spheres that have to be integrated point by point are marked for k_integrate_marked.
template <int SU, int SV, int SW>
__global__ __launch_bounds__(128) void k_integrate(AgenConsts C, CellDims dims, int64_t nmain, Mains M, NodeGeo G,
                                                   PairsOut O) {
  constexpr int D = SU * SV * SW;
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nmain) return;
  const Main m = main_of<SU, SV, SW>(C, M, G, k);
  double S[D];
  bool hit = false;
  if (C.moment_mode == 0) {
    if (grazing(C, m.cen, 0.5 * m.dsph) || !sphere_integrals<SU, SV, SW>(C, m.cen, 0.5 * m.dsph, S)) {
      M.list[k] |= kPointwise;
      return;
    }
#pragma unroll
    for (int l = 0; l < D; ++l) hit = hit || S[l] != 0.0;
  }
  bool near = false;
  for (int z = 0; z < 8; ++z) near = write_diagonal<SU, SV, SW>(C, dims, G, O, m, S, z) || near;
  if (hit && near) M.list[k] |= kPointwise;
}

// The marked ones: a wave looks through kMarkedRun main diagonals and takes the marked
// ones among them one after the other, its lanes the points of all pieces (a lane per
// sphere would wait 4 ms for the slowest); each basis function's sum then runs over the
// points in order, in one lane.
constexpr int kMarkedRun = 256;
template <int SU, int SV, int SW>
__global__ __launch_bounds__(64) void k_integrate_marked(AgenConsts C, CellDims dims, int64_t nmain, Mains M, NodeGeo G,
                                                          PairsOut O) {
  constexpr int D = SU * SV * SW, F = SU * SV + SW;
  static_assert(D <= 64, "a lane per basis function");
  __shared__ double pt[F][64 + 1];
  const int lane = threadIdx.x;
  for (int64_t k0 = (int64_t)blockIdx.x * kMarkedRun; k0 < min(nmain, ((int64_t)blockIdx.x + 1) * kMarkedRun); k0 += 64) {
    const bool mine = k0 + lane < nmain && (M.list[k0 + lane] & kPointwise) != 0;
    for (uint64_t todo = __ballot(mine); todo != 0; todo &= todo - 1) {
      const Main m = main_of<SU, SV, SW>(C, M, G, k0 + __builtin_ctzll(todo));
      const double r = 0.5 * m.dsph;
      double bp[20], sum = 0.0, S[D];
      const int nb = sphere_pieces(C, m.cen, r, bp), npt = nb > 1 ? (nb - 1) * C.nq : 0;
      for (int t0 = 0; t0 < npt; t0 += 64) {
        const int t = t0 + lane, p = min(t / C.nq, max(nb - 2, 0));
        double f[F];
        if (!(t < npt && bp[p + 1] > bp[p] && grazing_point<SU, SV, SW>(C, m.cen, r, bp[p], bp[p + 1], t - p * C.nq, f)))
          for (int i = 0; i < F; ++i) f[i] = 0.0;
        for (int i = 0; i < F; ++i) pt[i][lane] = f[i];
        __syncthreads();
        if (lane < D)
          for (int i = 0; i < 64; ++i) sum += pt[SU * SV + lane % SW][i] * pt[lane / SW][i];
        __syncthreads();
      }
      for (int l = 0; l < D; ++l) S[l] = __shfl(sum, l);
      if (lane < 8) write_diagonal<SU, SV, SW>(C, dims, G, O, m, S, lane);
    }
  }
}

// One wave per cp in turn: its kept pairs and, for each p, the first kept pair with
// local index of xi >= p
template <int D>
__global__ __launch_bounds__(64) void k_kept(int64_t ncp, const int64_t* __restrict__ off,
                                             const uint16_t* __restrict__ code, const uint8_t* __restrict__ keep,
                                             int32_t* __restrict__ kcnt, uint16_t* __restrict__ seg) {
  __shared__ int per[D];
  for (int64_t cp = blockIdx.x; cp < ncp; cp += gridDim.x) {
    if (threadIdx.x < D) per[threadIdx.x] = 0;
    __syncthreads();
    for (int64_t k = off[cp] + threadIdx.x; k < off[cp + 1]; k += 64)
      if (keep[k]) atomicAdd(&per[code[k] >> 8], 1);
    __syncthreads();
    if (threadIdx.x == 0) {
      uint16_t* s = seg + cp * (D + 1);
      int n = 0;
      for (int p = 0; p < D; ++p) {
        s[p] = (uint16_t)n;
        n += per[p];
      }
      s[D] = (uint16_t)n;
      kcnt[cp] = n;
    }
    __syncthreads();   // `per` is read
  }
}

// The kept pairs of each cp to their place, a workgroup per cp in turn, and the
// records per basis function (integer sums: exact whatever the order)
template <int D>
__global__ __launch_bounds__(256) void k_compact(int64_t ncp, const int64_t* __restrict__ off,
                                                 const int64_t* __restrict__ koff, const uint8_t* __restrict__ keep,
                                                 const double* __restrict__ src, double* __restrict__ out,
                                                 unsigned long long* __restrict__ cnt) {
  __shared__ int16_t from[D * D];
  __shared__ uint32_t nz[D];
  __shared__ int base[5];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x < D) nz[threadIdx.x] = 0;
  for (int64_t cp = blockIdx.x; cp < ncp; cp += gridDim.x) {
    const int64_t b = off[cp];
    const int n = (int)(off[cp + 1] - b), nk = (int)(koff[cp + 1] - koff[cp]);
    if (nk == 0) continue;
    int before = 0;
    for (int k0 = 0; k0 < n; k0 += 256) {
      const int k = k0 + (int)threadIdx.x;
      const bool ok = k < n && keep[b + k];
      const uint64_t m = __ballot(ok);
      __syncthreads();   // the last round's `base` is read
      if (lane == 0) base[wave + 1] = __popcll(m);
      __syncthreads();
      int at = before;
      for (int w = 0; w < wave; ++w) at += base[w + 1];
      if (ok) from[at + __popcll(m & (((uint64_t)1 << lane) - 1))] = (int16_t)k;
      for (int w = 0; w < 4; ++w) before += base[w + 1];
    }
    __syncthreads();
    double* o = out + koff[cp] * (D + 1);
    for (int i = threadIdx.x; i < nk * (D + 1); i += 256) {
      const int r = i / (D + 1), l = i - r * (D + 1);
      const double a = src[(b + from[r]) * (D + 1) + l];
      o[i] = a;
      if (l < D && a != 0.0) atomicAdd(&nz[l], 1u);
    }
    __syncthreads();
  }
  if (threadIdx.x < D) atomicAdd(&cnt[threadIdx.x], (unsigned long long)nz[threadIdx.x]);
}

template <int SU, int SV, int SW>
static int generate_t(dgv_ctx* ctx, const AgenConsts& C, double min_sens) {
  constexpr int D = SU * SV * SW;
  const Grid& g = ctx->g;
  const int64_t nc = g.ncells;
  // ordered cell pairs X <= Y (node ids of X precede those of Y)
  std::vector<int2> cps;
  cps.reserve((size_t)(nc * (nc + 1) / 2));
  for (int64_t X = 0; X < nc; ++X)
    for (int64_t Y = X; Y < nc; ++Y) cps.push_back(make_int2((int)X, (int)Y));
  const int64_t ncp = (int64_t)cps.size();
  int2* d_cps = nullptr;
  uint2* d_cnt = nullptr;
  int64_t *d_off = nullptr, *d_moff = nullptr;
  uint16_t* d_code = nullptr;
  int16_t* d_rank = nullptr;
  uint64_t* d_mains = nullptr;
  double *d_raw = nullptr, *d_pairs = nullptr;
  uint8_t* d_keep = nullptr;
  int32_t* d_kcnt = nullptr;
  uint16_t* d_seg = nullptr;
  unsigned long long* d_bcnt = nullptr;
  int rc = DGV_OK;
  auto cleanup = [&]() {
    hipFree(d_cps); hipFree(d_cnt); hipFree(d_off); hipFree(d_moff); hipFree(d_code); hipFree(d_rank);
    hipFree(d_mains); hipFree(d_raw); hipFree(d_keep); hipFree(d_kcnt); hipFree(d_seg); hipFree(d_bcnt);
  };
#define AG_HIP(call)                                                                           \
  do {                                                                                         \
    hipError_t e_ = (call);                                                                    \
    if (e_ != hipSuccess) {                                                                    \
      cleanup();                                                                               \
      if (d_pairs) hipFree(d_pairs);                                                           \
      return set_error(ctx, e_ == hipErrorOutOfMemory ? DGV_ERR_NOMEM : DGV_ERR_HIP,           \
                       std::string("A-array generator: ") + #call + ": " + hipGetErrorString(e_)); \
    }                                                                                          \
  } while (0)
  const NodeGeo G{ctx->d_u, ctx->d_v, ctx->d_w, ctx->d_gwts};
  const CellDims dims{g.Mv, g.Mw, nc};
  hipStream_t st = ctx->stream;
  AG_HIP(hipMalloc(&d_cps, sizeof(int2) * ncp));
  AG_HIP(hipMemcpyAsync(d_cps, cps.data(), sizeof(int2) * ncp, hipMemcpyHostToDevice, st));
  AG_HIP(hipMalloc(&d_cnt, sizeof(uint2) * ncp));
  hipLaunchKernelGGL((k_count<SU, SV, SW>), dim3(loop_blocks(ncp)), dim3(64), 0, st, C, dims, ncp, d_cps, G, d_cnt);
  AG_HIP(hipGetLastError());
  std::vector<uint2> cnt(ncp);
  AG_HIP(hipMemcpyAsync(cnt.data(), d_cnt, sizeof(uint2) * ncp, hipMemcpyDeviceToHost, st));
  AG_HIP(hipStreamSynchronize(st));
  std::vector<int64_t> off(ncp + 1, 0), moff(ncp + 1, 0);
  for (int64_t i = 0; i < ncp; ++i) {
    off[i + 1] = off[i] + cnt[i].x;
    moff[i + 1] = moff[i] + cnt[i].y;
  }
  const int64_t np = off[ncp], nmain = moff[ncp];
  AG_HIP(hipMalloc(&d_off, sizeof(int64_t) * (ncp + 1)));
  AG_HIP(hipMalloc(&d_moff, sizeof(int64_t) * (ncp + 1)));
  AG_HIP(hipMemcpyAsync(d_off, off.data(), sizeof(int64_t) * (ncp + 1), hipMemcpyHostToDevice, st));
  AG_HIP(hipMemcpyAsync(d_moff, moff.data(), sizeof(int64_t) * (ncp + 1), hipMemcpyHostToDevice, st));
  AG_HIP(hipMalloc(&d_code, sizeof(uint16_t) * std::max<int64_t>(np, 1)));
  AG_HIP(hipMalloc(&d_rank, sizeof(int16_t) * D * D * ncp));
  AG_HIP(hipMalloc(&d_mains, sizeof(uint64_t) * std::max<int64_t>(nmain, 1)));
  hipLaunchKernelGGL((k_list<SU, SV, SW>), dim3(loop_blocks(ncp)), dim3(64), 0, st, C, dims, ncp, d_cps, G, d_off, d_moff,
                     d_code, d_rank, d_mains);
  AG_HIP(hipGetLastError());
  AG_HIP(hipMalloc(&d_raw, sizeof(double) * (D + 1) * std::max<int64_t>(np, 1)));
  AG_HIP(hipMalloc(&d_keep, std::max<int64_t>(np, 1)));
  const PairsOut O{d_off, d_rank, min_sens, d_raw, d_keep};
  // integrate in slices so that each launch stays short
  const int64_t slice = 1 << 22;
  for (int64_t b = 0; b < nmain; b += slice) {
    const int64_t n = std::min(slice, nmain - b);
    const Mains M{d_cps, d_mains + b};
    hipLaunchKernelGGL((k_integrate<SU, SV, SW>), dim3((unsigned)((n + 127) / 128)), dim3(128), 0, st, C, dims, n, M, G, O);
    if (C.moment_mode == 0)
      hipLaunchKernelGGL((k_integrate_marked<SU, SV, SW>), dim3((unsigned)((n + kMarkedRun - 1) / kMarkedRun)), dim3(64), 0,
                         st, C, dims, n, M, G, O);
    AG_HIP(hipGetLastError());
  }
  // compaction
  AG_HIP(hipMalloc(&d_kcnt, sizeof(int32_t) * ncp));
  AG_HIP(hipMalloc(&d_seg, sizeof(uint16_t) * (D + 1) * ncp));
  AG_HIP(hipMalloc(&d_bcnt, sizeof(unsigned long long) * D));
  hipLaunchKernelGGL(k_kept<D>, dim3(loop_blocks(ncp)), dim3(64), 0, st, ncp, d_off, d_code, d_keep, d_kcnt, d_seg);
  AG_HIP(hipGetLastError());
  std::vector<int32_t> kcnt(ncp);
  std::vector<uint16_t> seg((size_t)ncp * (D + 1));
  AG_HIP(hipMemcpyAsync(kcnt.data(), d_kcnt, sizeof(int32_t) * ncp, hipMemcpyDeviceToHost, st));
  AG_HIP(hipMemcpyAsync(seg.data(), d_seg, sizeof(uint16_t) * (D + 1) * ncp, hipMemcpyDeviceToHost, st));
  AG_HIP(hipStreamSynchronize(st));
  std::vector<int64_t>& koff = moff;
  for (int64_t i = 0; i < ncp; ++i) koff[i + 1] = koff[i] + kcnt[i];
  const int64_t nk = koff[ncp];
  AG_HIP(hipMemcpyAsync(d_moff, koff.data(), sizeof(int64_t) * (ncp + 1), hipMemcpyHostToDevice, st));
  AG_HIP(hipMalloc(&d_pairs, sizeof(double) * (D + 1) * (nk + kPairPad)));
  AG_HIP(hipMemsetAsync(d_pairs + (D + 1) * nk, 0, sizeof(double) * (D + 1) * kPairPad, st));
  AG_HIP(hipMemsetAsync(d_bcnt, 0, sizeof(unsigned long long) * D, st));
  hipLaunchKernelGGL(k_compact<D>, dim3((unsigned)std::min<int64_t>(ncp, 4096)), dim3(256), 0, st, ncp, d_off, d_moff,
                     d_keep, d_raw, d_pairs, d_bcnt);
  AG_HIP(hipGetLastError());
  std::vector<unsigned long long> bcnt(D);
  AG_HIP(hipMemcpyAsync(bcnt.data(), d_bcnt, sizeof(unsigned long long) * D, hipMemcpyDeviceToHost, st));
  AG_HIP(hipStreamSynchronize(st));
  cleanup();
  // blocks (one per cell pair with kept pairs) and groups
  free_plan(ctx);
  free_pairblock(ctx);
  PairBlock& pb = ctx->pb;
  pb.D = D;
  pb.npairs = nk;
  pb.d_pairs = d_pairs;
  int64_t pbeg = 0;
  const int cc[3] = {g.ccu, g.ccv, g.ccw};
  std::map<std::array<int, 6>, std::vector<int32_t>> groups;
  for (int64_t cp = 0; cp < ncp; ++cp) {
    if (kcnt[cp] == 0) continue;
    BlockHdr h;
    std::memset(&h, 0, sizeof(h));
    h.pbeg = pbeg;
    const int X = cps[cp].x, Y = cps[cp].y;
    const int xc[3] = {(int)(X / ((int64_t)g.Mv * g.Mw)), (int)((X / g.Mw) % g.Mv), (int)(X % g.Mw)};
    const int yc[3] = {(int)(Y / ((int64_t)g.Mv * g.Mw)), (int)((Y / g.Mw) % g.Mv), (int)(Y % g.Mw)};
    int lo[3], ext[3];
    const int M[3] = {g.Mu, g.Mv, g.Mw};
    for (int d = 0; d < 3; ++d) {
      h.a[d] = (int8_t)(xc[d] - cc[d]);
      h.b[d] = (int8_t)(yc[d] - cc[d]);
      lo[d] = std::max(0, std::max(-(int)h.a[d], -(int)h.b[d]));
      ext[d] = std::min(M[d], std::min(M[d] - h.a[d], M[d] - h.b[d])) - lo[d];
    }
    h.npairs = (int16_t)kcnt[cp];
    for (int p = 0; p <= D; ++p) h.seg[p] = seg[(size_t)cp * (D + 1) + p];
    groups[{lo[0], lo[1], lo[2], ext[0], ext[1], ext[2]}].push_back((int32_t)pb.blocks.size());
    pb.blocks.push_back(h);
    pbeg += kcnt[cp];
  }
  for (auto& kv : groups) {
    Group Gr;
    for (int d = 0; d < 3; ++d) { Gr.lo[d] = kv.first[d]; Gr.ext[d] = kv.first[3 + d]; }
    Gr.ncells = Gr.ext[0] * Gr.ext[1] * Gr.ext[2];
    Gr.bbeg = (int32_t)pb.group_blocks.size();
    Gr.npairs = 0;
    for (int32_t b : kv.second) { pb.group_blocks.push_back(b); Gr.npairs += pb.blocks[b].npairs; }
    Gr.bend = (int32_t)pb.group_blocks.size();
    pb.groups.push_back(Gr);
  }
  pb.nrec_basis.assign(D, 0);
  for (int l = 0; l < D; ++l) pb.nrec_basis[l] = (int64_t)bcnt[l];
  pb.nrec_ref = std::accumulate(pb.nrec_basis.begin(), pb.nrec_basis.end(), (int64_t)0);
  DGV_HIP(ctx, hipMalloc(&pb.d_blocks, sizeof(BlockHdr) * std::max<size_t>(pb.blocks.size(), 1)));
  DGV_HIP(ctx, hipMemcpy(pb.d_blocks, pb.blocks.data(), sizeof(BlockHdr) * pb.blocks.size(), hipMemcpyHostToDevice));
  DGV_HIP(ctx, hipMalloc(&pb.d_group_blocks, sizeof(int32_t) * std::max<size_t>(pb.group_blocks.size(), 1)));
  DGV_HIP(ctx, hipMemcpy(pb.d_group_blocks, pb.group_blocks.data(), sizeof(int32_t) * pb.group_blocks.size(),
                         hipMemcpyHostToDevice));
  DGV_HIP(ctx, hipMalloc(&pb.d_groups, sizeof(Group) * std::max<size_t>(pb.groups.size(), 1)));
  DGV_HIP(ctx, hipMemcpy(pb.d_groups, pb.groups.data(), sizeof(Group) * pb.groups.size(), hipMemcpyHostToDevice));
  ctx->has_a = true;
  rc = build_quads(ctx);
  if (rc) return rc;
  rc = build_plan(ctx, ctx->tile);
#undef AG_HIP
  return rc;
}

int generate_pairblock(dgv_ctx* ctx, const dgv_agen_params& p) {
  AgenConsts C;
  std::string err;
  int rc = make_consts(ctx->g, p, C, err);
  if (rc) return set_error(ctx, rc, err);
  if (p.min_sens < 0) return set_error(ctx, DGV_ERR_ARG, "min_sens must be >= 0");
  DGV_HIP(ctx, hipSetDevice(ctx->device));
  const Grid& g = ctx->g;
  if (g.su == 3 && g.sv == 3 && g.sw == 3) return generate_t<3, 3, 3>(ctx, C, p.min_sens);
  if (g.su == 2 && g.sv == 2 && g.sw == 2) return generate_t<2, 2, 2>(ctx, C, p.min_sens);
  if (g.su == 1 && g.sv == 1 && g.sw == 1) return generate_t<1, 1, 1>(ctx, C, p.min_sens);
  return set_error(ctx, DGV_ERR_UNSUPPORTED, "A-array generator supports 1, 2 or 3 nodes per cell per dimension");
}

}  // namespace dgv

extern "C" int dgv_agen_pair(const dgv_grid_desc* grid, int64_t i2, int64_t i3, const dgv_agen_params* params,
                             double* raw, double* A) {
  using namespace dgv;
  if (!grid || !raw) { set_global_error("null argument"); return DGV_ERR_ARG; }
  Grid g;
  std::string err;
  int rc = build_grid(*grid, g, err);
  if (rc) { set_global_error(err); return rc; }
  dgv_agen_params p;
  p.Trad = 100.0; p.min_sens = 0.0; p.nquad = 0; p.moment_mode = 0;
  if (params) p = *params;
  AgenConsts C;
  rc = make_consts(g, p, C, err);
  if (rc) { set_global_error(err); return rc; }
  if (i2 < 1 || i3 < 1 || i2 > g.N || i3 > g.N) { set_global_error("node id out of range"); return DGV_ERR_INDEX; }
  const double x[3] = {g.u[i2 - 1], g.v[i2 - 1], g.w[i2 - 1]};
  const double y[3] = {g.u[i3 - 1], g.v[i3 - 1], g.w[i3 - 1]};
  double dsph = 0;
  rc = pair_raw_host(C, x, y, raw, &dsph);
  if (rc == -2) { set_global_error("unsupported nodes per cell"); return DGV_ERR_UNSUPPORTED; }
  const int D = g.D;
  if (rc == -1) {  // fails the prefilter: no record
    for (int l = 0; l < D; ++l) { raw[l] = 0.0; if (A) A[l] = 0.0; }
    return 1;
  }
  if (A)
    for (int l = 0; l < D; ++l) {
      double a = 0.0;
      if (std::fabs(raw[l]) > p.min_sens) {
        a = raw[l] * g.gwts[i3 - 1];
        a = a * g.gwts[i2 - 1];
        a = a * (dsph / 8.0);
      }
      A[l] = a;
    }
  return DGV_OK;
}
