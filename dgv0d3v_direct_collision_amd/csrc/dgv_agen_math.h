// dgv_agen_math.h -- per-pair values of the collision information operator A
// (host and device code).
//
// For a node pair (xi, xi1) and the Lagrange basis phi_l of the canonical cell K,
// SetA_DGV (dgvtools_mod.f90:377-681) computes
//   Atemp_l = int_0^pi int_0^2pi [phi_l(xi') + phi_l(xi1') - phi_l(xi) - phi_l(xi1)]
//             d eps  sin chi d chi,
//   A_l     = Atemp_l * w(xi1) * w(xi) * |g| / 8          (lines 654-659),
// with xi' = c + r k, xi1' = c - r k, c = (xi+xi1)/2, r = |xi-xi1|/2, k the unit
// vector of the angles (chi, eps) about g (EvalPhiPostCollIntegrand, lines
// 938-975).  The reference integrates with nested adaptive Simpson rules.
//
// Here the same integral is evaluated semi-analytically.  The measure
// sin chi d chi d eps is the surface measure of the unit sphere, so the gain
// term equals 2 * S_l with S_l = int_{S^2} phi_l(c + r k) dk, and the loss term
// is 4 pi (phi_l(xi) + phi_l(xi1)).  S_l is computed with the polar axis along w:
//   S_l = int sin(th) d th L_k(w^(th)) int_{arcs(th)} L_i(u^(eps)) L_j(v^(eps)) d eps,
// w = c_w + r cos(th), rho = r sin(th), u = c_u + rho cos eps, v = c_v + rho sin eps.
//  * The inner integral runs over the arcs of the circle of radius rho that lie
//    in [u0,u1]x[v0,v1]; the integrand is a polynomial in (cos eps, sin eps), so
//    it is integrated exactly with antiderivatives of cos^k sin^n.
//  * The outer integral is split at every polar angle where the arc structure
//    changes (circle tangent to a face line, circle through a corner, the
//    w-faces).  Inside a piece the integrand is analytic in th; at its ends it
//    has at worst square-root behaviour, which the substitution
//    th = ta + (tb-ta)(1-cos s)/2 removes, so Gauss-Legendre in s converges
//    exponentially.
//  * Inside a piece the arcs have the same ends throughout -- crossings of the same
//    face lines, in the same order -- so which crossings bound an arc inside the cell
//    is found once per piece.  A point of the outer integral then
//    takes each crossing's angle (one inverse function), its cosine and sine (one of
//    them the crossing's coordinate over rho, the other a square root; with up to two
//    nodes per dimension those of the angle), and adds its
//    antiderivatives with the sign of its end.
//  * The basis functions enter at the end: a point adds to the moments
//      W_kni = int w~^i sin(th) d th int_arcs u~^k v~^n d eps
//    of the distances u~, v~, w~ from the cell's centre (the inner ones from those of
//    cos and sin by u~ = a + rho cos eps), and S_l is a fixed combination of them.
#pragma once
#include <cmath>

#ifndef DGV_HD
#define DGV_HD __host__ __device__
#endif

namespace dgv {

constexpr int kAgenMaxS = 4;
constexpr int kAgenMaxQ = 48;

// Everything the per-pair evaluation needs, precomputed on the host.
struct AgenConsts {
  int su, sv, sw;
  double u0, u1, v0, v1, w0, w1;       // canonical cell
  double kap[3][kAgenMaxS];            // Gauss nodes on [-1,1] per dimension
  double mono[3][kAgenMaxS][kAgenMaxS];// L_i = sum_m mono[i][m] x^m, x the distance from the cell's centre
  double monol[2][kAgenMaxS][kAgenMaxS]; // the same in the local coordinate on [-1,1], u and v (grazing spheres)
  int nq;                              // Gauss points per smooth piece
  double qx[kAgenMaxQ], qw[kAgenMaxQ]; // Gauss-Legendre on [0, pi] in s: 1 - cos s, weight times sin s
  double qs[kAgenMaxQ], qv[kAgenMaxQ]; // the points s and weights themselves (grazing spheres)
  double Trad;
  int moment_mode;
};

// Lagrange basis function i on nodes kap[0..n-1] (lagrbasfun, dgvtools_mod.f90:31-56).
DGV_HD inline double lagr(int i, double x, const double* kap, int n) {
  double y = 1.0;
  for (int j = 0; j < n; ++j)
    if (j != i) y = y * (kap[j] - x) / (kap[j] - kap[i]);
  return y;
}

// Value of the canonical basis functions at a point (the restored
// EvalLagrBasisFunByNdsDGblzmEZ: zero outside the closed cell).
DGV_HD inline double basis_at(const AgenConsts& C, int iu, int iv, int iw, double u, double v, double w) {
  if (u < C.u0 || C.u1 < u || v < C.v0 || C.v1 < v || w < C.w0 || C.w1 < w) return 0.0;
  const double un = (u - (C.u1 + C.u0) / 2.0) / (C.u1 - C.u0) * 2.0;
  const double vn = (v - (C.v1 + C.v0) / 2.0) / (C.v1 - C.v0) * 2.0;
  const double wn = (w - (C.w1 + C.w0) / 2.0) / (C.w1 - C.w0) * 2.0;
  return lagr(iu, un, C.kap[0], C.su) * lagr(iv, vn, C.kap[1], C.sv) * lagr(iw, wn, C.kap[2], C.sw);
}

// Antiderivatives of cos^k sin^n for k, n < kAgenMaxS, by the reduction formulas
//   F_{k,n} = -s^{n-1} c^{k+1}/(k+n) + (n-1)/(k+n) F_{k,n-2}     (n >= 2)
//   F_{k,n} =  c^{k-1} s^{n+1}/(k+n) + (k-1)/(k+n) F_{k-2,n}     (k >= 2, n < 2):
// F_{k,n} = g_{k,n}(c, s) + t_{k,n} theta, t the mean of cos^k sin^n over the circle.
template <int ku, int kv>
DGV_HD inline void antideriv(double c, double s, double (&g)[ku][kv]) {   // g
  double cp[ku + 1], sp[kv + 1];
  cp[0] = 1.0;
  sp[0] = 1.0;
#pragma unroll
  for (int i = 1; i <= ku; ++i) cp[i] = cp[i - 1] * c;
#pragma unroll
  for (int i = 1; i <= kv; ++i) sp[i] = sp[i - 1] * s;
#pragma unroll
  for (int n = 0; n < kv; ++n)
#pragma unroll
    for (int k = 0; k < ku; ++k) {
      if (n >= 2) g[k][n] = -sp[n - 1] * cp[k + 1] * (1.0 / (k + n)) + ((double)(n - 1) / (k + n)) * g[k][n - 2];
      else if (k >= 2) g[k][n] = cp[k - 1] * sp[n + 1] * (1.0 / (k + n)) + ((double)(k - 1) / (k + n)) * g[k - 2][n];
      else g[k][n] = k == 0 ? (n == 0 ? 0.0 : -c) : (n == 0 ? s : s * s * 0.5);
    }
}

DGV_HD inline void sort_small(double* a, int n) {
  for (int i = 1; i < n; ++i) {
    const double x = a[i];
    int j = i - 1;
    while (j >= 0 && a[j] > x) { a[j + 1] = a[j]; --j; }
    a[j + 1] = x;
  }
}

// The arcs of the circle (cu + rho cos e, cv + rho sin e) inside [u0,u1]x[v0,v1], by their
// ends.  Line x (u = u0, u = u1, v = v0, v = v1) is crossed at two angles, a and 2 pi - a
// (u lines, a = acos(du / rho)) or a (+ 2 pi if negative) and pi - a (v lines, a = asin(dv / rho)).
// With the signs s1, s2 of the two crossings (1 where an arc ends, -1 where one begins,
// 0 where neither or both), diff = s1 - s2, sum = s1 + s2.  The angles are multiples of
// pi / 2 less or plus asin(d / rho): quarter counts those multiples, with their signs.
struct ArcEnds {
  double diff[4], sum[4], quarter;
  bool any;
};
DGV_HD inline ArcEnds arc_ends(const AgenConsts& C, double cu, double cv, const double du[2], const double dv[2],
                               double rho) {
  const double pi = 3.141592653589793238462643383279502884, twopi = 6.283185307179586476925286766559;
  double ang[9];
  int id[9], na = 0;   // crossing 2 x + i: the i-th of line x
  auto put = [&](double a, int x) {   // kept sorted
    int j = na++;
    while (j > 0 && ang[j - 1] > a) { ang[j] = ang[j - 1]; id[j] = id[j - 1]; --j; }
    ang[j] = a;
    id[j] = x;
  };
  for (int e = 0; e < 2; ++e) {
    const double X = du[e] / rho;
    if (X > -1.0 && X < 1.0) {
      const double a = acos(X);
      put(a, 2 * e);
      put(twopi - a, 2 * e + 1);
    }
    const double Y = dv[e] / rho;
    if (Y > -1.0 && Y < 1.0) {
      const double a = asin(Y);
      put(a < 0 ? a + twopi : a, 4 + 2 * e);
      put(pi - a, 5 + 2 * e);
    }
  }
  // distance of the circle's point at angle e to the nearest face line, negative outside
  auto margin = [&](double e) {
    const double x = cu + rho * cos(e), y = cv + rho * sin(e);
    return fmin(fmin(x - C.u0, C.u1 - x), fmin(y - C.v0, C.v1 - y));
  };
  // an arc may touch a line from within or without to rounding (where the sphere does):
  // of two points not both near the place, the one further from the lines decides
  auto inside = [&](double a, double b) {
    const double m = margin(a + 0.29 * (b - a)), n = margin(a + 0.63 * (b - a));
    return (fabs(m) > fabs(n) ? m : n) >= 0.0;
  };
  int beg = 0, end = 0, quarter = 0;
  if (na == 0) {
    quarter = inside(0.0, twopi) ? 4 : 0;   // the whole circle or none of it
  } else {
    ang[na] = ang[0] + twopi;
    id[na] = id[0];
    for (int i = 0; i < na; ++i) {
      const double a = ang[i], b = ang[i + 1];
      if (!(b > a) || !inside(a, b)) continue;
      beg |= 1 << id[i];
      end |= 1 << id[i + 1];
      if (i + 1 == na) quarter = 4;   // past 2 pi
    }
  }
  ArcEnds A;
  A.any = quarter != 0 || beg != end;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int s1 = ((end >> (2 * x)) & 1) - ((beg >> (2 * x)) & 1), s2 = ((end >> (2 * x + 1)) & 1) - ((beg >> (2 * x + 1)) & 1);
    A.diff[x] = s1 - s2;
    A.sum[x] = s1 + s2;
    quarter += x < 2 ? s1 + 3 * s2 : (dv[x & 1] < 0.0 ? 4 * s1 : 0) + 2 * s2;
  }
  A.quarter = quarter;
  return A;
}

// I[k][n] = integral of cos^k sin^n over the arcs with these ends at radius rho.  The
// second crossing of a line mirrors the first, s -> -s (u lines) or c -> -c (v lines), under
// which g_{k,n} is odd for even n (even k) and even else: one evaluation serves both.
// A far sphere's arcs are short and its circle's centre far away: to_local multiplies errors
// that theta and g do not share by the distance.  Hence the low part of pi / 2, and up to
// two nodes per dimension, where little else is lost, the cosine and sine of the rounded angle
// in place of the crossing's coordinate and a square root.  Against extended precision
// (random pairs, relative L2; the search at every point first, then without and with
// both): 2 nodes, 6 / 9 / 13 cells 3.3 4.0 2.8e-16 / 2.9 4.9 2.7e-16 / 4.4 8.9 4.3e-16; 3 nodes, 6 cells 3.9
// 3.2e-15 and with the low part alone 2.4e-15.
template <int ku, int kv>
DGV_HD inline void arc_moments(const ArcEnds& A, const double du[2], const double dv[2], double rho,
                               double (&I)[ku][kv]) {
  const double halfpi = 1.570796326794896619231321691639751442;
  double th = A.quarter * halfpi, g[ku][kv];
#pragma unroll
  for (int k = 0; k < ku; ++k)
#pragma unroll
    for (int n = 0; n < kv; ++n) I[k][n] = 0.0;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const double diff = A.diff[x], sum = A.sum[x];
    if (diff == 0.0 && sum == 0.0) continue;
    double X = fmin(1.0, fmax(-1.0, (x < 2 ? du[x & 1] : dv[x & 1]) / rho)), Z;
    const double a = asin(X);
    th += x < 2 ? -diff * a : diff * a;
    if constexpr (ku <= 2 && kv <= 2) {
      Z = cos(a);
      X = sin(a);
    } else {
      Z = sqrt((1.0 - X) * (1.0 + X));
    }
    antideriv<ku, kv>(x < 2 ? X : Z, x < 2 ? Z : X, g);
#pragma unroll
    for (int k = 0; k < ku; ++k)
#pragma unroll
      for (int n = 0; n < kv; ++n) I[k][n] += ((x < 2 ? n : k) & 1 ? sum : diff) * g[k][n];
  }
  th += A.quarter * 6.123233995736766035868820147291983e-17;   // pi / 2 less its double
#pragma unroll
  for (int k = 0; k < ku; k += 2)
#pragma unroll
    for (int n = 0; n < kv; n += 2) I[k][n] += (k == 0 ? (n == 0 ? 1.0 : 0.5) : (n == 0 ? 0.5 : 0.125)) * th;
}

// Moments of cos^k sin^n -> moments of (au + rho cos)^k (av + rho sin)^n, one dimension
// after the other, by (a + rho x) m_k = a m_k + rho m_{k+1} from the highest power down.
template <int ku, int kv>
DGV_HD inline void to_local(double au, double av, double rho, double (&I)[ku][kv]) {
#pragma unroll
  for (int p = 0; p + 1 < ku; ++p)
#pragma unroll
    for (int k = ku - 1; k > p; --k)
#pragma unroll
      for (int n = 0; n < kv; ++n) I[k][n] = au * I[k - 1][n] + rho * I[k][n];
#pragma unroll
  for (int p = 0; p + 1 < kv; ++p)
#pragma unroll
    for (int n = kv - 1; n > p; --n)
#pragma unroll
      for (int k = 0; k < ku; ++k) I[k][n] = av * I[k][n - 1] + rho * I[k][n];
}

// The outer integral's pieces for a sphere: ascending ends bp[0 .. n) in theta, n returned
// (0: the sphere misses the cell's w range)
DGV_HD inline int sphere_pieces(const AgenConsts& C, const double cen[3], double r, double (&bp)[20]) {
  const double pi = 3.141592653589793238462643383279502884;
  // polar angle theta about the w axis: w = c_w + r cos(theta), rho = r sin(theta)
  // is analytic in theta (no branch points at the poles)
  const double ca = (C.w1 - cen[2]) / r, cb = (C.w0 - cen[2]) / r;
  const double th_lo = ca >= 1.0 ? 0.0 : (ca <= -1.0 ? pi : acos(ca));
  const double th_hi = cb >= 1.0 ? 0.0 : (cb <= -1.0 ? pi : acos(cb));
  if (!(th_hi > th_lo)) return 0;
  // breakpoints: tangency to the four face lines and passage through the four
  // corners of the cell's u-v rectangle, at rho = d, i.e. theta = asin(d/r)
  // and pi - asin(d/r)
  int nb = 0;
  bp[nb++] = th_lo;
  bp[nb++] = th_hi;
  const double du[2] = {C.u0 - cen[0], C.u1 - cen[0]}, dv[2] = {C.v0 - cen[1], C.v1 - cen[1]};
  auto add = [&](double d) {
    if (d < r) {
      const double t = asin(d / r);
      if (t > th_lo && t < th_hi) bp[nb++] = t;
      if (pi - t > th_lo && pi - t < th_hi) bp[nb++] = pi - t;
    }
  };
  for (int e = 0; e < 2; ++e) { add(fabs(du[e])); add(fabs(dv[e])); }
  for (int e = 0; e < 2; ++e)
    for (int f = 0; f < 2; ++f) add(sqrt(du[e] * du[e] + dv[f] * dv[f]));
  sort_small(bp, nb);
  return nb;
}

// Whether the sphere touches the cell or all but contains it, or lies within it, to
// rounding: these are integrated point by point (grazing_point)
DGV_HD inline bool grazing(const AgenConsts& C, const double cen[3], double r) {
  const double lo[3] = {C.u0, C.v0, C.w0}, hi[3] = {C.u1, C.v1, C.w1};
  double near2 = 0.0, far2 = 0.0, depth = r + r;   // depth: distance of the centre to the nearest face, from within
  for (int d = 0; d < 3; ++d) {
    const double a = lo[d] - cen[d], b = cen[d] - hi[d], n = fmax(0.0, fmax(a, b)), f = fmax(fabs(a), fabs(b));
    near2 += n * n;
    far2 += f * f;
    depth = fmin(depth, fmin(-a, -b));
  }
  const double far = sqrt(far2), tol = 1e-10 * (r + far);
  return fabs(r - sqrt(near2)) <= tol || fabs(r - far) <= tol || r <= depth + tol;
}

// S[l] = int_{S^2} phi_l(c + r k) dk for the su*sv*sw canonical basis functions; the sphere
// is not a grazing one.  False, and no S, if a piece is a sliver: where the radius equals the
// distance of a face line or a corner to rounding, two breakpoints lie about 2e-8 apart and
// which of the sliver's arcs are inside is a matter of the last bits.  Left to the search at
// every point too, so that the values stay what that search gives (1e-8 of a raw value).
template <int su, int sv, int sw>
DGV_HD inline bool sphere_integrals(const AgenConsts& C, const double cen[3], double r, double* S) {
  constexpr int D = su * sv * sw;
#pragma unroll
  for (int l = 0; l < D; ++l) S[l] = 0.0;
  const double pi = 3.141592653589793238462643383279502884;
  double bp[20];
  const int nb = sphere_pieces(C, cen, r, bp);
  if (nb == 0) return true;
  for (int p = 0; p + 1 < nb; ++p)
    if (bp[p + 1] - bp[p] > 1e-11 && bp[p + 1] - bp[p] < 1e-6) return false;
  const double du[2] = {C.u0 - cen[0], C.u1 - cen[0]}, dv[2] = {C.v0 - cen[1], C.v1 - cen[1]};
  const double mu = 0.5 * (C.u1 + C.u0), mv = 0.5 * (C.v1 + C.v0), mw = 0.5 * (C.w1 + C.w0);
  const double au = cen[0] - mu, av = cen[1] - mv, aw = cen[2] - mw;
  double W[su][sv][sw];   // [k][n][i]
#pragma unroll
  for (int k = 0; k < su; ++k)
#pragma unroll
    for (int n = 0; n < sv; ++n)
#pragma unroll
      for (int i = 0; i < sw; ++i) W[k][n][i] = 0.0;
  for (int p = 0; p + 1 < nb; ++p) {
    const double ta = bp[p], tb = bp[p + 1];
    if (!(tb > ta)) continue;
    const double half = 0.5 * (tb - ta);
    // a point well inside the piece, away from the equator: there rho = r, and a sphere
    // that just reaches a corner or a line has its crossings coincide
    const double tl = ta + 0.7 * half, tr = ta + 1.3 * half;
    const ArcEnds A = arc_ends(C, cen[0], cen[1], du, dv, r * sin(fabs(tl - 0.5 * pi) > fabs(tr - 0.5 * pi) ? tl : tr));
    if (!A.any) continue;
    for (int q = 0; q < C.nq; ++q) {
      const double th = ta + half * C.qx[q];
      const double sth = sin(th), cth = cos(th);
      const double wt = C.qw[q] * half * sth;   // dt = sin(theta) dtheta
      const double rho = r * sth;
      if (!(rho > 0.0)) continue;
      double I[su][sv];
      arc_moments<su, sv>(A, du, dv, rho, I);
      const double wn = aw + r * cth;
      double pw[sw];
      pw[0] = wt;
#pragma unroll
      for (int i = 1; i < sw; ++i) pw[i] = pw[i - 1] * wn;
      to_local<su, sv>(au, av, rho, I);
#pragma unroll
      for (int k = 0; k < su; ++k)
#pragma unroll
        for (int n = 0; n < sv; ++n)
#pragma unroll
          for (int i = 0; i < sw; ++i) W[k][n][i] += pw[i] * I[k][n];
    }
  }
  // the basis functions of the moments, one dimension after the other
#pragma unroll
  for (int k = 0; k < su; ++k)
#pragma unroll
    for (int n = 0; n < sv; ++n) {
      double t[sw];
#pragma unroll
      for (int j = 0; j < sw; ++j) {
        t[j] = 0.0;
#pragma unroll
        for (int i = 0; i < sw; ++i) t[j] += C.mono[2][j][i] * W[k][n][i];
      }
#pragma unroll
      for (int j = 0; j < sw; ++j) W[k][n][j] = t[j];
    }
#pragma unroll
  for (int i = 0; i < su; ++i)
#pragma unroll
    for (int j = 0; j < sv; ++j)
#pragma unroll
      for (int l = 0; l < sw; ++l) {
        double E = 0.0;
#pragma unroll
        for (int k = 0; k < su; ++k) {
          double row = 0.0;
#pragma unroll
          for (int n = 0; n < sv; ++n) row += C.mono[1][j][n] * W[k][n][l];
          E += C.mono[0][i][k] * row;
        }
        S[(i * sv + j) * sw + l] = E;
      }
  return true;
}

// ---- Grazing spheres -------------------------------------------------------------------
//
// A record exists where a value exceeds min_sens, which may be 0.  For a sphere that
// touches the cell to rounding that is decided by single points whose arcs are a few
// units in the last place long; for one within the cell, or with a value that is zero but
// for rounding (near_cutoff), by how the last bits fall; and slivers (sphere_integrals) by
// them too.  These spheres keep the search
// for the arcs at every point, with the basis functions expanded there, so that the
// set of records does not depend on how the others are integrated.  They are few (1 in
// 500, up to 4 in 100 where cells and nodes are alike in all dimensions) and eight
// times as costly per point.
DGV_HD inline bool near_cutoff(double raw, double min_sens) { return fabs(fabs(raw) - min_sens) <= 1e-12; }

// F_{k,n}(theta) itself, by the formulas above
DGV_HD inline void antideriv_at(double th, double c, double s, int ku, int kv, double F[kAgenMaxS][kAgenMaxS]) {
  double cp[kAgenMaxS + 2], sp[kAgenMaxS + 2];
  cp[0] = 1.0;
  sp[0] = 1.0;
  for (int i = 1; i < kAgenMaxS + 2; ++i) { cp[i] = cp[i - 1] * c; sp[i] = sp[i - 1] * s; }
  for (int n = 0; n < kv; ++n)
    for (int k = 0; k < ku; ++k) {
      double v;
      if (n >= 2) {
        v = -sp[n - 1] * cp[k + 1] / (k + n) + (double)(n - 1) / (k + n) * F[k][n - 2];
      } else if (k >= 2) {
        v = cp[k - 1] * sp[n + 1] / (k + n) + (double)(k - 1) / (k + n) * F[k - 2][n];
      } else if (k == 0 && n == 0) {
        v = th;
      } else if (k == 1 && n == 0) {
        v = s;
      } else if (k == 0 && n == 1) {
        v = -c;
      } else {  // k == 1, n == 1
        v = s * s / 2.0;
      }
      F[k][n] = v;
    }
}

// I[k][n] = integral of cos^k sin^n over the arcs of the circle
// (cu + rho cos e, cv + rho sin e) lying inside [u0,u1]x[v0,v1].
template <int SU, int SV>
DGV_HD inline void arc_moments_at(const AgenConsts& C, double cu, double cv, double rho,
                               double I[kAgenMaxS][kAgenMaxS]) {
  constexpr int ku = SU, kv = SV;
  for (int k = 0; k < ku; ++k)
    for (int n = 0; n < kv; ++n) I[k][n] = 0.0;
  const double twopi = 6.283185307179586476925286766559;
  double ang[9];
  int na = 0;
  const double du[2] = {C.u0 - cu, C.u1 - cu}, dv[2] = {C.v0 - cv, C.v1 - cv};
  for (int e = 0; e < 2; ++e) {
    const double X = du[e] / rho;
    if (X > -1.0 && X < 1.0) {
      const double a = acos(X);
      ang[na++] = a;
      ang[na++] = twopi - a;
    }
    const double Y = dv[e] / rho;
    if (Y > -1.0 && Y < 1.0) {
      double a = asin(Y);
      if (a < 0) a += twopi;
      ang[na++] = a;
      double b = 3.141592653589793238462643383279502884 - asin(Y);
      ang[na++] = b;
    }
  }
  auto inside = [&](double e) {
    const double x = cu + rho * cos(e), y = cv + rho * sin(e);
    return x >= C.u0 && x <= C.u1 && y >= C.v0 && y <= C.v1;
  };
  double Fa[kAgenMaxS][kAgenMaxS], Fb[kAgenMaxS][kAgenMaxS];
  if (na == 0) {
    if (!inside(0.0)) return;
    antideriv_at(0.0, 1.0, 0.0, ku, kv, Fa);
    antideriv_at(twopi, 1.0, 0.0, ku, kv, Fb);
    for (int k = 0; k < ku; ++k)
      for (int n = 0; n < kv; ++n) I[k][n] = Fb[k][n] - Fa[k][n];
    return;
  }
  sort_small(ang, na);
  ang[na] = ang[0] + twopi;
  for (int i = 0; i < na; ++i) {
    const double a = ang[i], b = ang[i + 1];
    if (!(b > a)) continue;
    if (!inside(0.5 * (a + b))) continue;
    antideriv_at(a, cos(a), sin(a), ku, kv, Fa);
    antideriv_at(b, cos(b), sin(b), ku, kv, Fb);
    for (int k = 0; k < ku; ++k)
      for (int n = 0; n < kv; ++n) I[k][n] += Fb[k][n] - Fa[k][n];
  }
}

// Coefficients c[i][k] of L_i(alpha + beta x) = sum_k c[i][k] x^k.
template <int s>
DGV_HD inline void shifted_coeffs(const double mono[kAgenMaxS][kAgenMaxS], double alpha, double beta,
                                  double c[kAgenMaxS][kAgenMaxS]) {
  // binomial expansion of (alpha + beta x)^m
  double ap[kAgenMaxS], bp[kAgenMaxS];
  ap[0] = 1.0;
  bp[0] = 1.0;
  for (int m = 1; m < s; ++m) { ap[m] = ap[m - 1] * alpha; bp[m] = bp[m - 1] * beta; }
  for (int i = 0; i < s; ++i)
    for (int k = 0; k < s; ++k) {
      double acc = 0.0;
      for (int m = k; m < s; ++m) {
        double binom = 1.0;
        for (int t = 0; t < k; ++t) binom = binom * (m - t) / (t + 1);
        acc += mono[i][m] * binom * ap[m - k];
      }
      c[i][k] = acc * bp[k];
    }
}

// Point q of the piece [ta, tb]: it adds f[su sv + k] * f[i sv + j] to S_(i, j, k), in the
// order of the points.  False: it adds nothing.
template <int su, int sv, int sw>
DGV_HD inline bool grazing_point(const AgenConsts& C, const double cen[3], double r, double ta, double tb, int q,
                                 double* f) {
  const double hu = 0.5 * (C.u1 - C.u0), hv = 0.5 * (C.v1 - C.v0), hw = 0.5 * (C.w1 - C.w0);
  const double mu = 0.5 * (C.u1 + C.u0), mv = 0.5 * (C.v1 + C.v0), mw = 0.5 * (C.w1 + C.w0);
  const double au = (cen[0] - mu) / hu, av = (cen[1] - mv) / hv;
  double I[kAgenMaxS][kAgenMaxS], cU[kAgenMaxS][kAgenMaxS], cV[kAgenMaxS][kAgenMaxS];
  const double half = 0.5 * (tb - ta);
  const double sq = C.qs[q];
  const double th = ta + half * (1.0 - cos(sq));
  const double sth = sin(th);
  const double wt = C.qv[q] * half * sin(sq) * sth;   // dt = sin(theta) dtheta
  const double rho = r * sth;
  if (!(rho > 0.0)) return false;
  arc_moments_at<su, sv>(C, cen[0], cen[1], rho, I);
  shifted_coeffs<su>(C.monol[0], au, rho / hu, cU);
  shifted_coeffs<sv>(C.monol[1], av, rho / hv, cV);
  const double wn = (cen[2] + r * cos(th) - mw) / hw;
  for (int k = 0; k < sw; ++k) f[su * sv + k] = wt * lagr(k, wn, C.kap[2], sw);
  for (int i = 0; i < su; ++i)
    for (int j = 0; j < sv; ++j) {
      double E = 0.0;
      for (int k = 0; k < su; ++k) {
        double row = 0.0;
        for (int n = 0; n < sv; ++n) row += cV[j][n] * I[k][n];
        E += cU[i][k] * row;
      }
      f[i * sv + j] = E;
    }
  return true;
}

template <int su, int sv, int sw>
DGV_HD inline void grazing_integrals(const AgenConsts& C, const double cen[3], double r, double* S) {
  for (int l = 0; l < su * sv * sw; ++l) S[l] = 0.0;
  double bp[20], f[su * sv + sw];
  const int nb = sphere_pieces(C, cen, r, bp);
  for (int p = 0; p + 1 < nb; ++p)
    for (int q = 0; bp[p + 1] > bp[p] && q < C.nq; ++q)
      if (grazing_point<su, sv, sw>(C, cen, r, bp[p], bp[p + 1], q, f))
        for (int l = 0; l < su * sv * sw; ++l) S[l] += f[su * sv + l % sw] * f[l / sw];
}

// Raw values Atemp_l (before min_sens and the weights) of one pair from its sphere
// integrals S_l: the gain 2 S_l less the loss 4 pi (phi_l(xi) + phi_l(xi1)).
template <int SU, int SV, int SW>
DGV_HD inline void raw_from_sphere(const AgenConsts& C, const double x[3], const double y[3], const double* S,
                                   double* raw) {
  const double fourpi = 12.566370614359172953850573533118;
  for (int iu = 0; iu < SU; ++iu)
    for (int iv = 0; iv < SV; ++iv)
      for (int iw = 0; iw < SW; ++iw) {
        const int l = (iu * SV + iv) * SW + iw;
        const double loss = basis_at(C, iu, iv, iw, x[0], x[1], x[2]) + basis_at(C, iu, iv, iw, y[0], y[1], y[2]);
        raw[l] = 2.0 * S[l] - fourpi * loss;
      }
}

// The same for the moment test functions psi = 1,u,v,w,|u|^2 over the whole sphere
// (dgvtools_mod.f90:267-274): closed forms of int psi(c + r k) dk; the value is
// every basis function's.
DGV_HD inline double raw_moment(int mode, const double x[3], const double y[3], double r) {
  const double fourpi = 12.566370614359172953850573533118;
  const double cen[3] = {0.5 * (x[0] + y[0]), 0.5 * (x[1] + y[1]), 0.5 * (x[2] + y[2])};
  double S, px, py;
  switch (mode) {
    case 1: S = fourpi; px = 1.0; py = 1.0; break;
    case 2: S = fourpi * cen[0]; px = x[0]; py = y[0]; break;
    case 3: S = fourpi * cen[1]; px = x[1]; py = y[1]; break;
    case 4: S = fourpi * cen[2]; px = x[2]; py = y[2]; break;
    default:
      S = fourpi * (cen[0] * cen[0] + cen[1] * cen[1] + cen[2] * cen[2] + r * r);
      px = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
      py = y[0] * y[0] + y[1] * y[1] + y[2] * y[2];
      break;
  }
  return 2.0 * S - fourpi * (px + py);
}

// |xi - xi1| of a pair, or -1 if it fails SetA_DGV's prefilter
// (dgvtools_mod.f90:527-530).  Exchanging one component of the two nodes changes
// no bit of it, nor of the pair's midpoint.
DGV_HD inline double pair_distance(const AgenConsts& C, const double x[3], const double y[3]) {
  const double d0 = x[0] - y[0], d1 = x[1] - y[1], d2 = x[2] - y[2];
  const double dsph = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
  const double s0 = x[0] + y[0] - C.u0 - C.u1, s1 = x[1] + y[1] - C.v0 - C.v1, s2 = x[2] + y[2] - C.w0 - C.w1;
  const double dist2 = sqrt(s0 * s0 + s1 * s1 + s2 * s2);
  const double e0 = C.u1 - C.u0, e1 = C.v1 - C.v0, e2 = C.w1 - C.w0;
  const double dphi = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
  if ((dist2 > dsph + dphi) || (dist2 + dphi < dsph) || (dsph > C.Trad)) return -1.0;
  return dsph;
}

// Raw values Atemp_l of one pair; -1 if the pair fails the prefilter.
template <int SU, int SV, int SW>
DGV_HD inline int pair_raw(const AgenConsts& C, const double x[3], const double y[3], double* raw, double* dsph_out) {
  constexpr int D = SU * SV * SW;
  const double dsph = pair_distance(C, x, y);
  *dsph_out = dsph;
  if (dsph < 0.0) return -1;
  if (C.moment_mode != 0) {
    const double v = raw_moment(C.moment_mode, x, y, 0.5 * dsph);
    for (int l = 0; l < D; ++l) raw[l] = v;
    return 0;
  }
  const double cen[3] = {0.5 * (x[0] + y[0]), 0.5 * (x[1] + y[1]), 0.5 * (x[2] + y[2])};
  double S[D];
  const double r = 0.5 * dsph;
  bool pointwise = grazing(C, cen, r);
  if (!pointwise) pointwise = !sphere_integrals<SU, SV, SW>(C, cen, r, S);
  if (!pointwise) {
    raw_from_sphere<SU, SV, SW>(C, x, y, S, raw);
    bool hit = false, near = false;
    for (int l = 0; l < D; ++l) {
      hit = hit || S[l] != 0.0;
      near = near || near_cutoff(raw[l], 0.0);
    }
    pointwise = hit && near;
  }
  if (pointwise) {
    grazing_integrals<SU, SV, SW>(C, cen, r, S);
    raw_from_sphere<SU, SV, SW>(C, x, y, S, raw);
  }
  return 0;
}

}  // namespace dgv
