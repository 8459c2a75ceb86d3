// exact_math.hpp — binary64 triangle-pair kernels for the MI355X engine.
//
// These are the per-pair computations of the reference's bfSolver
// (delta/contact/detection/bf.cpp:217-1178) and penaltySolver
// (penalty.cpp:278-431, 434-581), re-expressed for a SIMT wavefront:
//   * the seven-region point-triangle case analysis is folded into a "kind"
//     code and a single division, so a wave does not diverge over regions;
//   * the nine segment-segment solves are branch-free selects;
//   * every arithmetic operation is the reference's own, in its order, and the
//     translation unit is compiled with -ffp-contract=off, so results are
//     bit-identical to the reference built without FMA.
// The header is also compiled for the host (DH_HD empty) so the same code can
// be checked against the CPU restatement without a GPU.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DH_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#define DH_HD inline
#endif

namespace dh {

template <typename T>
struct V3 {
  T x, y, z;
};

template <typename T>
DH_HD V3<T> sub(const V3<T>& a, const V3<T>& b) {
  return {a.x - b.x, a.y - b.y, a.z - b.z};
}

// ((a.x*b.x + a.y*b.y) + a.z*b.z), the reference's DOT macro (algo.h:167)
template <typename T>
DH_HD T dot(const V3<T>& a, const V3<T>& b) {
  return a.x * b.x + a.y * b.y + a.z * b.z;
}

template <typename T>
DH_HD T dsqrt(T v) {
  using std::sqrt;
  return sqrt(v);
}

// Clamped segment-segment parameters (bf.cpp:589-663).  Returns sc, tc.
template <typename T>
DH_HD void segseg(T a, T b, T c, T d, T e, T& sc, T& tc) {
  const T small_num = T(1E-30);
  const T D = a * c - b * b;
  const bool par = D < small_num;
  T sN = b * e - c * d;
  T tN = a * e - b * d;
  T sD = D, tD = D;
  // infinite-line solution clamped to the s-range
  const bool s_lo = !par && (sN < T(0));
  const bool s_hi = !par && !(sN < T(0)) && (sN > sD);
  if (par) {
    sN = T(0);
    sD = T(1);
    tN = e;
    tD = c;
  }
  if (s_lo) {
    sN = T(0);
    tN = e;
    tD = c;
  }
  if (s_hi) {
    sN = sD;
    tN = e + b;
    tD = c;
  }
  // clamp t and recompute s on the visible edge (selects, no branches)
  const bool tlo = tN < T(0);
  const bool thi = !tlo && (tN > tD);
  const T v = tlo ? -d : (-d + b);
  const bool lo = v < T(0);
  const bool hi = !lo && (v > a);
  const T nsN = lo ? T(0) : (hi ? sD : v);
  const T nsD = (lo || hi) ? sD : a;
  const bool clamp = tlo || thi;
  sN = clamp ? nsN : sN;
  sD = clamp ? nsD : sD;
  tN = tlo ? T(0) : (thi ? tD : tN);
  using std::fabs;
  const T qs = sN / sD;
  const T qt = tN / tD;
  sc = (fabs(sN) < small_num) ? T(0) : qs;
  tc = (fabs(tN) < small_num) ? T(0) : qt;
}

// Point-triangle squared distance (bf.cpp:922-1091).  The eight outcomes of
// the region analysis: F (s=t=0), S1 (s=1), T1 (t=1), SE (t=0, s=-d/a),
// TE (s=0, t=-e/c), IN (interior), D2 (s+t=1, s=numer/denom), D6 (s+t=1,
// t=numer/denom).

template <typename T>
DH_HD T pt_tri(T a, T b, T c, T d, T e, T f, T& s_out, T& t_out) {
  const T det = a * c - b * b;
  const T s0 = b * e - c * d;
  const T t0 = b * d - a * e;
  // region of (s0, t0) (Eberly's numbering) and the resulting case, as
  // booleans so that the wave selects instead of branching
  const bool c_st = (s0 + t0) <= det;
  const bool sneg = s0 < T(0), tneg = t0 < T(0);
  const bool r0 = c_st && !sneg && !tneg;
  const bool r4 = c_st && sneg && tneg;
  const bool r3 = c_st && sneg && !tneg;
  const bool r5 = c_st && !sneg && tneg;
  const bool r2 = !c_st && sneg;
  const bool r6 = !c_st && !sneg && tneg;
  const bool r1 = !c_st && !sneg && !tneg;
  const T tmp0 = sneg ? (b + d) : (b + e);  // region 2 : region 6
  const T tmp1 = sneg ? (c + e) : (a + d);
  const bool gt = tmp1 > tmp0;
  const T denom = a - T(2) * b + c;
  const T numer26 = tmp1 - tmp0;
  const T numer1 = c + e - b - d;
  const bool nge = numer26 >= denom, t1le = tmp1 <= T(0);
  const bool n1le = numer1 <= T(0), n1ge = numer1 >= denom;
  const bool e_pos = e >= T(0), e_big = -e >= c;
  const bool d_pos = d >= T(0), d_big = -d >= a, d_neg = d < T(0);
  const bool useE = r3 || (r4 && !d_neg) || (r2 && !gt && !t1le);  // s = 0 edge
  const bool useD = r5 || (r6 && !gt && !t1le);                    // t = 0 edge
  const bool bIN = r0;
  const bool bT1 = (useE && !e_pos && e_big) || (r2 && !gt && t1le) || (r6 && gt && nge) ||
                   (r1 && n1le);
  const bool bTE = useE && !e_pos && !e_big;
  const bool bS1 = (useD && !d_pos && d_big) || (r4 && d_neg && d_big) || (r2 && gt && nge) ||
                   (r6 && !gt && t1le) || (r1 && !n1le && n1ge);
  const bool bSE = (useD && !d_pos && !d_big) || (r4 && d_neg && !d_big);
  const bool bD2 = (r2 && gt && !nge) || (r1 && !n1le && !n1ge);
  const bool bD6 = r6 && gt && !nge;
  // one division: 1/det, -d/a, -e/c or numer/denom
  const T num = bIN ? T(1) : bSE ? -d : bTE ? -e : (r1 ? numer1 : numer26);
  const T den = bIN ? det : bSE ? a : bTE ? c : denom;
  const T q = num / den;
  const T s = bIN ? s0 * q : (bD2 || bSE) ? q : bD6 ? T(1) - q : bS1 ? T(1) : T(0);
  const T t = bIN ? t0 * q : bD2 ? T(1) - q : (bD6 || bTE) ? q : bT1 ? T(1) : T(0);
  const T quad = s * (a * s + b * t + T(2) * d) + t * (b * s + c * t + T(2) * e) + f;
  T sqr = (bIN || bD2 || bD6) ? quad
        : bSE ? d * s + f
        : bTE ? e * t + f
        : bS1 ? a + T(2) * d + f
        : bT1 ? c + T(2) * e + f : f;
  sqr = (sqr <= T(0)) ? T(0) : sqr;
  s_out = s;
  t_out = t;
  return sqr;
}

template <typename T>
struct Tri {
  V3<T> v[3];
};

// t.v[i] for a run-time i in 0..2, as selects
template <typename T>
DH_HD V3<T> pick3(const Tri<T>& t, int i) {
  const bool i1 = (i == 1), i2 = (i == 2);
  const T x0 = t.v[0].x, x1 = t.v[1].x, x2 = t.v[2].x;
  const T y0 = t.v[0].y, y1 = t.v[1].y, y2 = t.v[2].y;
  const T z0 = t.v[0].z, z1 = t.v[1].z, z2 = t.v[2].z;
  return {i2 ? x2 : (i1 ? x1 : x0), i2 ? y2 : (i1 ? y1 : y0), i2 ? z2 : (i1 ? z1 : z0)};
}

template <typename T>
DH_HD V3<T> sel3(bool c, const V3<T>& a, const V3<T>& b) {
  return {c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z};
}

// One segment-segment feature of bfSolver (bf.cpp:409-713), folded into the
// running minimum (strict <, first index wins).
template <typename T>
DH_HD void edge_edge(T& ssmin, T& ttc, T& ssc, int& ssid, const V3<T>& ha, const V3<T>& oa,
                     const V3<T>& hb, const V3<T>& ob, int j) {
  const V3<T> u = sub(ha, oa);
  const V3<T> v = sub(hb, ob);
  const V3<T> w = sub(oa, ob);
  const T a = dot(u, u), b = dot(u, v), c = dot(v, v), d = dot(u, w), e = dot(v, w);
  T sc, tc;
  segseg(a, b, c, d, e, sc, tc);
  const V3<T> dP = {w.x + (sc * u.x) - (tc * v.x), w.y + (sc * u.y) - (tc * v.y),
                    w.z + (sc * u.z) - (tc * v.z)};
  const T dist = dsqrt(dP.x * dP.x + dP.y * dP.y + dP.z * dP.z);
  const bool better = dist < ssmin;
  ssmin = better ? dist : ssmin;
  ttc = better ? tc : ttc;
  ssc = better ? sc : ssc;
  ssid = better ? j : ssid;
}

// One vertex-face feature (bf.cpp:875-1100): point pt against face f0 f1 f2.
template <typename T>
DH_HD void vertex_face(T& ptmin, T& ss, T& tt, int& id, const V3<T>& f0, const V3<T>& f1,
                       const V3<T>& f2, const V3<T>& pt, int j) {
  const V3<T> e0 = sub(f1, f0);
  const V3<T> e1 = sub(f2, f0);
  const V3<T> dd = sub(f0, pt);
  T s, t;
  const T sqr = pt_tri(dot(e0, e0), dot(e0, e1), dot(e1, e1), dot(e0, dd), dot(e1, dd),
                       dot(dd, dd), s, t);
  const T dist = dsqrt(sqr);
  const bool better = dist < ptmin;
  ptmin = better ? dist : ptmin;
  ss = better ? s : ss;
  tt = better ? t : tt;
  id = better ? j : id;
}

// The least edge-edge distance of a triangle pair (feature ssid, parameters
// ssc on A's edge and ttc on B's) and the least vertex-face distance (feature
// id, face parameters ss and tt).
template <typename T>
struct BfBest {
  T ssmin, ttc, ssc, ptmin, ss, tt;
  int ssid, id;
};

// The features of bfSolver for any input.
template <typename T>
DH_HD void bf_features(const Tri<T>& A, const Tri<T>& B, BfBest<T>& best) {
  T ssmin = T(1E+30), ttc = T(0), ssc = T(0);
  int ssid = 0;
  // Edge k of a triangle runs from its origin v[(k+1)%3] towards v[k].  The
  // features are visited in the reference's order by rotating the vertex
  // triples; the loops are kept rolled so that only one feature is live at a
  // time (register pressure decides the occupancy of this kernel).
  V3<T> a0 = A.v[0], a1 = A.v[1], a2 = A.v[2];
#pragma unroll 1
  for (int k = 0; k < 3; ++k) {
    V3<T> b0 = B.v[0], b1 = B.v[1], b2 = B.v[2];
#pragma unroll 1
    for (int m = 0; m < 3; ++m) {
      edge_edge(ssmin, ttc, ssc, ssid, a0, a1, b0, b1, 3 * k + m);
      const V3<T> tb = b0;
      b0 = b1;
      b1 = b2;
      b2 = tb;
    }
    const V3<T> ta = a0;
    a0 = a1;
    a1 = a2;
    a2 = ta;
  }
  T ptmin = T(1E30), ss = T(0), tt = T(0);
  int id = 0;
  // j = 0..2: vertex j of B against face A; j = 3..5: vertex j-3 of A against B
  {
    V3<T> p0 = B.v[0], p1 = B.v[1], p2 = B.v[2];
#pragma unroll 1
    for (int j = 0; j < 3; ++j) {
      vertex_face(ptmin, ss, tt, id, A.v[0], A.v[1], A.v[2], p0, j);
      const V3<T> tp = p0;
      p0 = p1;
      p1 = p2;
      p2 = tp;
    }
  }
  {
    V3<T> p0 = A.v[0], p1 = A.v[1], p2 = A.v[2];
#pragma unroll 1
    for (int j = 3; j < 6; ++j) {
      vertex_face(ptmin, ss, tt, id, B.v[0], B.v[1], B.v[2], p0, j);
      const V3<T> tp = p0;
      p0 = p1;
      p1 = p2;
      p2 = tp;
    }
  }
  best = {ssmin, ttc, ssc, ptmin, ss, tt, ssid, id};
}

// ---- the same features with fewer instructions, for regular pairs
//
// One pair per lane is bound by the instructions it issues, and the general
// form above spends most of its own on selects, on moving the rotating
// vertices and on the scaling that a division and a square root need for
// extreme exponents.  bf_features_regular unrolls the features (edges, their
// squared lengths and the faces' terms are formed once), clamps the
// parameters instead of selecting among the clamped cases, and divides and
// takes roots without scaling.  Every value that reaches a result is the same
// operation on the same operands, so the results are the same bit for bit.
// Regular means that no intermediate value leaves the range in which that
// holds: squared edge lengths (and a face's third one, as the face's formula
// has it) of at least 1e-30, so that a clamped parameter's numerator and
// denominator are not taken for zero, and of less than 2^180, so that nothing
// overflows (a feature further away than the 1e30 that the minima start from
// is not taken, whatever its value), no point over the inside of a face
// whose determinant is in (0, 1e-60), and no feature's distance in (0, 2^-350).
// Coordinates that are NaN are regular: as in the general form, the distance
// of each feature that they are part of is NaN, which is never the least.
// MI355X, 2^24 pairs: 2,807 to 2,185 vector instructions per wave of 64 pairs,
// 1.39 to 1.17 ms.  A wave leaves as soon as one of its lanes has too
// short or too long an edge: with two such pairs in 100, 2^20 pairs took 148
// us where the others went on, 102 by the general form alone.

// a / b, correctly rounded, for 2^-400 < |a|, |b| < 2^400 (other operands: any
// value): the reciprocal by two Newton steps, then Markstein's final step (the
// quotient's residual, exact in a fused multiply-add, times the reciprocal),
// which rounds correctly where the reciprocal is good to half a unit or so
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990).  The GPU tests compare it with the host's division.
DH_HD double div_regular(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(b);
  y = fma(fma(-b, y, 1.0), y, y);
  y = fma(fma(-b, y, 1.0), y, y);
  const double q = a * y;
  return fma(fma(-b, q, a), y, q);
#else
  return a / b;
#endif
}

// div_regular in two parts, for several quotients by one b.
DH_HD double recip_regular(double b) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(b);
  y = fma(fma(-b, y, 1.0), y, y);
  return fma(fma(-b, y, 1.0), y, y);
#else
  return 1.0 / b;
#endif
}

DH_HD double quotient_regular(double a, double b, double y) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double q = a * y;
  return fma(fma(-b, q, a), y, q);
#else
  (void)y;
  return a / b;
#endif
}

// The smaller of e and a's binary exponent (0 for a = 0).
DH_HD int least_exponent(int e, double a) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int x = __builtin_amdgcn_frexp_exp(a);
#else
  int x = 0;
  std::frexp(a, &x);
#endif
  return x < e ? x : e;
}

// The square root at which a squared distance is too small for sqrt_regular.
constexpr double kSqrtLeast = 0x1p-349;

// sqrt(x), correctly rounded, for x >= 2^-700 and x = 0, by Goldschmidt's
// iteration and two residual corrections (Markstein, as above).  Between 0 and
// 2^-700 the value is positive and below kSqrtLeast: the estimate y of
// 1 / sqrt(2^-700) gives g = x * y in (0, 2^-350), and every correction adds a
// factor of 1 to 1.5.
DH_HD double sqrt_regular(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double y = __builtin_amdgcn_rsq(fmax(x, 0x1p-700));
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
#else
  return std::sqrt(x);
#endif
}

// q in [0, 1] (the clamp of an instruction's result).
DH_HD double clamp01(double q) {
#if defined(__HIP_DEVICE_COMPILE__)
  return fmin(fmax(q, 0.0), 1.0);
#else
  return q > 0.0 ? (q < 1.0 ? q : 1.0) : 0.0;
#endif
}

// segseg and the distance for edges u (squared length a) and v (c) of a
// regular pair, w from v's origin to u's.  The s-range's clamps are the
// clamp of sN / D; only parallel edges that keep their t need a zero of
// their own.
DH_HD double edge_edge_regular(const V3<double>& u, double a, const V3<double>& v, double c,
                               const V3<double>& w, double& sc, double& tc) {
  using std::fabs;
  const double small_num = 1E-30;
  const double b = dot(u, v), d = dot(u, w), e = dot(v, w);
  const double D = a * c - b * b;
  const double sN = b * e - c * d;
  const bool par = D < small_num;
  const bool s_hi = !par && sN > D;
  const bool edge = par || sN < 0.0 || s_hi;
  const double eb = e + b, t0 = a * e - b * d, bd = b - d, nd = -d;
  const double te = s_hi ? eb : e;
  const double tN = edge ? te : t0;
  const double tD = edge ? c : D;
  const bool tlo = tN < 0.0, clamp = tlo || tN > tD;
  const double x = tlo ? nd : bd;
  const double num = clamp ? x : sN, den = clamp ? a : D;
  const double qs = clamp01(div_regular(num, den));
  const double qt = clamp01(div_regular(tN, tD));
  sc = (fabs(num) < small_num || (par && !clamp)) ? 0.0 : qs;
  tc = (fabs(tN) < small_num) ? 0.0 : qt;
  const V3<double> dP = {w.x + (sc * u.x) - (tc * v.x), w.y + (sc * u.y) - (tc * v.y),
                         w.z + (sc * u.z) - (tc * v.z)};
  return sqrt_regular(dP.x * dP.x + dP.y * dP.y + dP.z * dP.z);
}

// The terms of a face that its three points share.
struct FaceTerms {
  V3<double> o, e0, e1;
  double a, b, c, det, denom;
  bool inside;  // 1 / det does not overflow, or is the infinity that leaves NaN
  DH_HD explicit FaceTerms(const Tri<double>& t)
      : o(t.v[0]), e0(sub(t.v[1], t.v[0])), e1(sub(t.v[2], t.v[0])), a(dot(e0, e0)),
        b(dot(e0, e1)), c(dot(e1, e1)), det(a * c - b * b), denom(a - 2.0 * b + c),
        inside(det >= 1E-60 || det == 0.0) {}
};

// pt_tri and the distance for a regular face: the face parameters are
// (s0, t0) / det inside, and on the boundary one clamped quotient: along
// t = 0, along s = 0, or along s + t = 1.  pt_tri's sums for the three
// corners are its quadratic form at (0, 0), (1, 0) and (0, 1) term by term,
// so only the two edges t = 0 and s = 0 have a form of their own.  `ok` is
// cleared over the inside of a face that is nearly, but not quite, a line.
DH_HD double vertex_face_regular(const FaceTerms& f, const V3<double>& pt, double& s, double& t,
                                 bool& ok) {
  const V3<double> dd = sub(f.o, pt);
  const double d = dot(f.e0, dd), e = dot(f.e1, dd), ff = dot(dd, dd);
  const double a = f.a, b = f.b, c = f.c;
  const double s0 = b * e - c * d, t0 = b * d - a * e;
  const bool in = (s0 + t0) <= f.det, sneg = s0 < 0.0, tneg = t0 < 0.0, dneg = d < 0.0;
  const double bd = b + d, be = b + e, ce = c + e, ad = a + d;
  const bool gt2 = ce > bd, gt6 = ad > be;
  const bool r0 = in && !sneg && !tneg;
  const bool r1 = !in && !sneg && !tneg, r2 = !in && sneg, r6 = !in && !sneg && tneg;
  const bool useE = (in && sneg && !(tneg && dneg)) || (r2 && !gt2);
  const bool useD = (in && tneg && (!sneg || dneg)) || (r6 && !gt6);
  const bool hyp6 = r6 && gt6;
  const double h1 = ce - b - d, h2 = ce - bd, h6 = ad - be, ne = -e, nd = -d;
  double num = r2 ? h2 : h6, den = f.denom;
  num = r1 ? h1 : num;
  num = useD ? nd : num;
  den = useD ? a : den;
  num = useE ? ne : num;
  den = useE ? c : den;
  num = r0 ? 1.0 : num;
  den = r0 ? f.det : den;
  const double q = num / den;
  const double p = clamp01(q), p1 = 1.0 - p;
  const double si = s0 * q, ti = t0 * q;
  s = hyp6 ? p1 : p;
  t = hyp6 ? p : p1;
  t = useD ? 0.0 : t;
  s = useE ? 0.0 : s;
  t = useE ? p : t;
  s = r0 ? si : s;
  t = r0 ? ti : t;
  const double quad = s * (a * s + b * t + 2.0 * d) + t * (b * s + c * t + 2.0 * e) + ff;
  const double line = (useE ? e : d) * p + ff;
  const double sqr = ((useE || useD) && num < den) ? line : quad;
  ok &= !r0 || f.inside;
  return fma(sqr, 0.0, sqrt_regular(fmax(sqr, 0.0)));  // NaN stays, which fmax drops
}

// Forgets what the compiler has derived from a triangle's first vertex, so
// that it forms the faces' terms again after the edges instead of keeping
// them in registers meanwhile.
DH_HD void forget_derived(Tri<double>& t) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(t.v[0].x), "+v"(t.v[0].y), "+v"(t.v[0].z));
#endif
}

DH_HD void feature_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// Whether `ok` holds for every lane of the wave (on the host: for this pair).
DH_HD bool whole_wave(bool ok) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __all(ok);
#else
  return ok;
#endif
}

// The features of a regular pair; false (and `best` to be ignored) for others.
DH_HD bool bf_features_regular(Tri<double> A, Tri<double> B, BfBest<double>& best) {
  bool ok = true;
  double least = 1E300, most = 0.0;  // fmin and fmax skip NaN
  double ssmin = 1E+30, ssc = 0.0, ttc = 0.0, ptmin = 1E+30, ss = 0.0, tt = 0.0;
  int ssid = 0, id = 0;
  V3<double> v[3];
  double c[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    v[m] = sub(B.v[m], B.v[m == 2 ? 0 : m + 1]);
    c[m] = dot(v[m], v[m]);
    const V3<double> u = sub(A.v[m], A.v[m == 2 ? 0 : m + 1]);
    const double a = fma(u.x, u.x, fma(u.y, u.y, u.z * u.z));  // dot(u, u) but for rounding
    least = fmin(least, fmin(a, c[m]));
    most = fmax(most, fmax(a, c[m]));
  }
  if (!whole_wave(least >= 1.0001E-30 && most < 0x1p179)) return false;
  // A's vertices rotate through a loop that stays rolled (three turns put
  // them back), B's edges are unrolled
#pragma unroll 1
  for (int k = 0; k < 9; k += 3) {
    const V3<double> u = sub(A.v[0], A.v[1]);
    const double a = dot(u, u);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      feature_fence();
      const V3<double> w = sub(A.v[1], B.v[m == 2 ? 0 : m + 1]);
      double sc, tc;
      const double dist = edge_edge_regular(u, a, v[m], c[m], w, sc, tc);
      const bool better = dist < ssmin;
      ssmin = better ? dist : ssmin;
      ssc = better ? sc : ssc;
      ttc = better ? tc : ttc;
      ssid = better ? k + m : ssid;
    }
    const V3<double> t = A.v[0];
    A.v[0] = A.v[1];
    A.v[1] = A.v[2];
    A.v[2] = t;
  }
  forget_derived(A);
  forget_derived(B);
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const FaceTerms face(f ? B : A);
    least = fmin(least, face.denom);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      feature_fence();
      double s, t;
      const double dist = vertex_face_regular(face, f ? A.v[j] : B.v[j], s, t, ok);
      const bool better = dist < ptmin;
      ptmin = better ? dist : ptmin;
      ss = better ? s : ss;
      tt = better ? t : tt;
      id = better ? 3 * f + j : id;
    }
  }
  best = {ssmin, ttc, ssc, ptmin, ss, tt, ssid, id};
  // a distance that sqrt_regular did not round is the least of its kind
  ok &= (ssmin >= kSqrtLeast || ssmin == 0.0) && (ptmin >= kSqrtLeast || ptmin == 0.0);
  return ok && least >= 1E-30;
}

// The closest points of the better feature; true when it is the edge-edge one
// (ptmin > ssmin, bf.cpp:1102).  With kZoltan the output stage is that of
// zoltan/bf.cpp, whose switch cases 1 fall through into cases 2
// (zoltan/bf.cpp:527-559, 907-925): edge-edge feature 1 takes its Q from B's
// edge 2->0 with feature 1's parameter, vertex-face feature 1 reports B's
// vertex 2.
template <typename T, bool kZoltan = false>
DH_HD bool bf_points(const Tri<T>& A, const Tri<T>& B, const BfBest<T>& best, V3<T>& P, V3<T>& Q) {
  const int ssid = best.ssid, id = best.id;
  const T ssc = best.ssc, ttc = best.ttc, ss = best.ss, tt = best.tt;
  if (best.ptmin > best.ssmin) {
    const int k = ssid / 3, m = (kZoltan && ssid == 1) ? 2 : ssid - 3 * (ssid / 3);
    // register selects instead of dynamic indexing (keeps Tri out of scratch)
    const V3<T> ha = pick3(A, k), oa = pick3(A, k == 2 ? 0 : k + 1);
    const V3<T> hb = pick3(B, m), ob = pick3(B, m == 2 ? 0 : m + 1);
    const V3<T> u = sub(ha, oa), v = sub(hb, ob);
    P = {oa.x + (u.x * ssc), oa.y + (u.y * ssc), oa.z + (u.z * ssc)};
    Q = {ob.x + (v.x * ttc), ob.y + (v.y * ttc), ob.z + (v.z * ttc)};
    return true;
  }
  const bool onA = id < 3;
  const V3<T> f0 = sel3(onA, A.v[0], B.v[0]);
  const V3<T> f1 = sel3(onA, A.v[1], B.v[1]);
  const V3<T> f2 = sel3(onA, A.v[2], B.v[2]);
  const V3<T> onf = {f0.x + ((f2.x - f0.x) * tt) + ((f1.x - f0.x) * ss),
                     f0.y + ((f2.y - f0.y) * tt) + ((f1.y - f0.y) * ss),
                     f0.z + ((f2.z - f0.z) * tt) + ((f1.z - f0.z) * ss)};
  const V3<T> vtx = sel3(onA, pick3(B, (kZoltan && id == 1) ? 2 : id), pick3(A, id - 3));
  P = sel3(onA, onf, vtx);
  Q = sel3(onA, vtx, onf);
  return false;
}

// bfSolver: closest points P on A and Q on B, and the least features of both
// kinds.  Returns true when the edge-edge result is kept.
template <bool kZoltan = false>
DH_HD bool bf_solver_ids(const Tri<double>& A, const Tri<double>& B, V3<double>& P, V3<double>& Q,
                         int& ssid_out, int& id_out) {
  BfBest<double> best;
  if (!bf_features_regular(A, B, best)) bf_features(A, B, best);
  ssid_out = best.ssid;
  id_out = best.id;
  return bf_points<double, kZoltan>(A, B, best, P, Q);
}

DH_HD bool bf_solver_ids(const Tri<float>& A, const Tri<float>& B, V3<float>& P, V3<float>& Q,
                         int& ssid_out, int& id_out) {
  BfBest<float> best;
  bf_features(A, B, best);
  ssid_out = best.ssid;
  id_out = best.id;
  return bf_points(A, B, best, P, Q);
}

template <typename T>
DH_HD bool bf_solver(const Tri<T>& A, const Tri<T>& B, V3<T>& P, V3<T>& Q) {
  int ssid, id;
  return bf_solver_ids(A, B, P, Q, ssid, id);
}

// The same by the general path alone, for the detection without the survivor
// queue: its few survivors per item wait for loads and barriers rather than
// for instructions, while the particles of a run that has left all bounds (so
// far out that their triangles round to lines and points) pair with every
// other.
DH_HD bool bf_solver_general(const Tri<double>& A, const Tri<double>& B, V3<double>& P,
                             V3<double>& Q) {
  BfBest<double> best;
  bf_features(A, B, best);
  return bf_points(A, B, best, P, Q);
}

// |Q-P| in the caller's order (bf.cpp:117, contactpoint.cpp:157-159).
template <typename T>
DH_HD T pq_dist(const V3<T>& P, const V3<T>& Q) {
  return dsqrt(((Q.x - P.x) * (Q.x - P.x)) + ((Q.y - P.y) * (Q.y - P.y)) +
               ((Q.z - P.z) * (Q.z - P.z)));
}

// True when one triangle's plane separates the other triangle from it by
// more than the contact margin (no contact, bf.cpp:125): with n = (A1 - A0) x
// (A2 - A0), all of B on one side of A's plane at heights |n.(B_k - A0)| /
// |n| above the margin (or the same with A and B exchanged).  A lies in its
// plane, so the smallest height bounds the distance from below.  Rounding:
// the heights' numerators are within 2^-49.3 |u||v||r| of exact (u, v A's
// edges, r the vertex offsets) and |n| within 2^-49.8 |u||v|; the test
// lowers the heights by 2^-46 |u|_1 |v|_1 |r|_1 and raises |n| by 2^-48
// |u|_1 |v|_1, against the box test's threshold margin (1 + 2^-20) + mag
// 2^-40, beyond which bfSolver's binary64 distance exceeds the margin.
// Two faces of near-touching convex particles are separated by their planes
// almost always when they are apart, so this removes most of the pairs the
// box test leaves at the cost of two cross products.
DH_HD bool plane_side_apart(const Tri<double>& A, const Tri<double>& B, double thr) {
  using std::fabs;
  const V3<double> u = sub(A.v[1], A.v[0]), v = sub(A.v[2], A.v[0]);
  const V3<double> n = {u.y * v.z - u.z * v.y, u.z * v.x - u.x * v.z, u.x * v.y - u.y * v.x};
  const double uv = (fabs(u.x) + fabs(u.y) + fabs(u.z)) * (fabs(v.x) + fabs(v.y) + fabs(v.z));
  double lo = 1e308, hi = -1e308, R = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const V3<double> r = sub(B.v[k], A.v[0]);
    const double h = dot(n, r);
    lo = fmin(lo, h);
    hi = fmax(hi, h);
    R = fmax(R, fabs(r.x) + fabs(r.y) + fabs(r.z));
  }
  const double E = 0x1p-46 * uv * R;
  const double nn = std::sqrt(dot(n, n)) + 0x1p-48 * uv;
  const double h = lo > 0.0 ? lo : -hi;  // the least height, when all on one side
  return h - E > thr * nn;
}

// The separating axes of the nine edge pairs: n = ea x eb for an edge ea of
// A and eb of B.  Every vertex is projected onto n (relative to A's first
// vertex); when B's projections lie beyond A's by a gap g, every point of B
// is at least g / |n| from every point of A.  n is used as computed (any
// axis bounds the distance), so only the projections round: each is within
// E = 2^-46 |ea|_1 |eb|_1 R of exact (R the largest relative vertex
// distance, as in plane_side_apart), and |n| is bounded above as there.
// True when some axis separates A and B by more than thr.
DH_HD bool edge_axes_apart(const Tri<double>& A, const Tri<double>& B, double thr) {
  using std::fabs;
  V3<double> ra[3], rb[3];
  double R = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    ra[k] = sub(A.v[k], A.v[0]);
    rb[k] = sub(B.v[k], A.v[0]);
    R = fmax(R, fmax(fabs(ra[k].x) + fabs(ra[k].y) + fabs(ra[k].z),
                     fabs(rb[k].x) + fabs(rb[k].y) + fabs(rb[k].z)));
  }
  // unrolled: a variable index into A.v or B.v would put both triangles
  // in scratch memory
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const V3<double> ea = sub(A.v[k == 2 ? 0 : k + 1], A.v[k]);
    const double la = fabs(ea.x) + fabs(ea.y) + fabs(ea.z);
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      const V3<double> eb = sub(B.v[m == 2 ? 0 : m + 1], B.v[m]);
      const V3<double> n = {ea.y * eb.z - ea.z * eb.y, ea.z * eb.x - ea.x * eb.z,
                            ea.x * eb.y - ea.y * eb.x};
      const double uv = la * (fabs(eb.x) + fabs(eb.y) + fabs(eb.z));
      double loA = 1e308, hiA = -1e308, loB = 1e308, hiB = -1e308;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const double ha = dot(n, ra[i]), hb = dot(n, rb[i]);
        loA = fmin(loA, ha);
        hiA = fmax(hiA, ha);
        loB = fmin(loB, hb);
        hiB = fmax(hiB, hb);
      }
      const double E = 0x1p-46 * uv * R;
      const double nn = std::sqrt(dot(n, n)) + 0x1p-48 * uv;
      const double gap = fmax(loB - hiA, loA - hiB);
      if (gap - 2.0 * E > thr * nn) return true;
    }
  }
  return false;
}

// The margin with its rounding band for the axes of A and B.
DH_HD double axis_reach(const Tri<double>& A, const Tri<double>& B, double margin) {
  using std::fabs;
  double mag = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    mag = fmax(mag, fmax(fmax(fabs(A.v[k].x), fabs(A.v[k].y)),
                         fmax(fmax(fabs(A.v[k].z), fabs(B.v[k].x)),
                              fmax(fabs(B.v[k].y), fabs(B.v[k].z)))));
  return margin * (1.0 + 0x1p-20) + mag * 0x1p-40;
}

DH_HD bool plane_apart(const Tri<double>& A, const Tri<double>& B, double margin) {
  const double thr = axis_reach(A, B, margin);
  return plane_side_apart(A, B, thr) || plane_side_apart(B, A, thr);
}

// Screen before bfSolver in binary64: true when A and B are provably farther
// apart than the contact margin (no contact, bf.cpp:125).  bfSolver in
// binary32 (coordinates relative to A's first vertex) gives a direction n =
// Q32 - P32; every point of A and B projects onto n, and the gap between the
// two projections divided by |n| bounds the distance from below whatever n
// is.  (The binary32 points themselves may be far from the closest pair: a
// small triangle against a large one, such as a floor, cancels most of the
// bits of the point-face quadratic form, so their distance is no bound.)
// Rounding: the vertices relative to A's first one are rounded once to
// binary32 (within 2^-24 of their length), the projections add 3 ulp, so
// each projection is within 2^-21 |n| S of exact, S the largest relative
// vertex length; the bound is lowered by 2^-19 |n| S and compared, like the
// box test, against margin (1 + 2^-20) + mag 2^-40 (mag the largest
// coordinate magnitude), beyond which bfSolver's binary64 distance exceeds
// the margin as well.
DH_HD bool screened_far(const Tri<double>& A, const Tri<double>& B, double margin) {
  using std::fabs;
  const V3<double> o = A.v[0];
  Tri<float> a32, b32;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    a32.v[k] = {static_cast<float>(A.v[k].x - o.x), static_cast<float>(A.v[k].y - o.y),
                static_cast<float>(A.v[k].z - o.z)};
    b32.v[k] = {static_cast<float>(B.v[k].x - o.x), static_cast<float>(B.v[k].y - o.y),
                static_cast<float>(B.v[k].z - o.z)};
  }
  V3<float> p32, q32;
  bf_solver(a32, b32, p32, q32);
  const V3<float> n = {q32.x - p32.x, q32.y - p32.y, q32.z - p32.z};
  float amax = -3.0e38f, bmin = 3.0e38f, S = 0.f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const V3<float> a = a32.v[k], b = b32.v[k];
    amax = fmaxf(amax, n.x * a.x + n.y * a.y + n.z * a.z);
    bmin = fminf(bmin, n.x * b.x + n.y * b.y + n.z * b.z);
    S = fmaxf(S, fmaxf(fabs(a.x) + fabs(a.y) + fabs(a.z), fabs(b.x) + fabs(b.y) + fabs(b.z)));
  }
  const double nn = std::sqrt(static_cast<double>(n.x) * n.x + static_cast<double>(n.y) * n.y +
                              static_cast<double>(n.z) * n.z);
  const double lower = (static_cast<double>(bmin) - static_cast<double>(amax) -
                        0x1p-19 * nn * static_cast<double>(S)) /
                       (nn * (1.0 + 0x1p-20));
  const double mag = fmax(fmax(fabs(o.x), fabs(o.y)), fabs(o.z)) + static_cast<double>(S);
  return nn > 0.0 && lower > margin * (1.0 + 0x1p-20) + mag * 0x1p-40;
}

// Penalty Newton solver state (penalty.cpp:278-357).
template <typename T>
struct Penalty {
  V3<T> A0, B0, BA, CA, ED, FD;
  T h[16];
  T r, reg0;

  DH_HD void setup(const Tri<T>& A, const Tri<T>& B) {
    A0 = A.v[0];
    B0 = B.v[0];
    BA = sub(A.v[1], A.v[0]);
    CA = sub(A.v[2], A.v[0]);
    ED = sub(B.v[1], B.v[0]);
    FD = sub(B.v[2], B.v[0]);
    h[0] = T(2.) * dot(BA, BA);
    h[1] = T(2.) * dot(CA, BA);
    h[2] = T(-2.) * dot(ED, BA);
    h[3] = T(-2.) * dot(FD, BA);
    h[4] = h[1];
    h[5] = T(2.) * dot(CA, CA);
    h[6] = T(-2.) * dot(ED, CA);
    h[7] = T(-2.) * dot(FD, CA);
    h[8] = h[2];
    h[9] = h[6];
    h[10] = T(2.) * dot(ED, ED);
    h[11] = T(2.) * dot(FD, ED);
    h[12] = h[3];
    h[13] = h[7];
    h[14] = h[11];
    h[15] = T(2.) * dot(FD, FD);
    const T trace = h[0] + h[5] + h[10] + h[15];
    reg0 = trace * T(1E-2);
    r = dsqrt(T(0.0125) * trace) * T(1E5);
  }

  // One regularised Newton step from x (penalty.cpp:361-412).
  DH_HD void step(const T x[4], T reg, T dx[4]) const {
    const bool c0 = (-x[0] <= T(0)), c1 = (-x[1] <= T(0)), c2 = (x[0] + x[1] - T(1) <= T(0));
    const bool c3 = (-x[2] <= T(0)), c4 = (-x[3] <= T(0)), c5 = (x[2] + x[3] - T(1) <= T(0));
    T dh[8], mx[6];
    dh[0] = c0 ? T(0) : T(-1);
    mx[0] = c0 ? T(0) : -x[0];
    dh[2] = c1 ? T(0) : T(-1);
    mx[1] = c1 ? T(0) : -x[1];
    dh[1] = dh[3] = c2 ? T(0) : T(1);
    mx[2] = c2 ? T(0) : x[0] + x[1] - T(1);
    dh[4] = c3 ? T(0) : T(-1);
    mx[3] = c3 ? T(0) : -x[2];
    dh[6] = c4 ? T(0) : T(-1);
    mx[4] = c4 ? T(0) : -x[3];
    dh[5] = dh[7] = c5 ? T(0) : T(1);
    mx[5] = c5 ? T(0) : x[2] + x[3] - T(1);
    const V3<T> sxy = {(A0.x + (BA.x * x[0]) + (CA.x * x[1])) - (B0.x + (ED.x * x[2]) + (FD.x * x[3])),
                       (A0.y + (BA.y * x[0]) + (CA.y * x[1])) - (B0.y + (ED.y * x[2]) + (FD.y * x[3])),
                       (A0.z + (BA.z * x[0]) + (CA.z * x[1])) - (B0.z + (ED.z * x[2]) + (FD.z * x[3]))};
    T a[16], b[4];
    b[0] = T(2) * dot(sxy, BA) + r * (dh[0] * mx[0] + dh[1] * mx[2]);
    a[0] = h[0] + r * (dh[0] * dh[0] + dh[1] * dh[1]) + reg;
    a[4] = h[4] + r * (dh[3] * dh[1]);
    const T tmp1 = (h[1] + r * (dh[1] * dh[3])) / a[0];
    a[13] = h[13] - h[12] * tmp1;
    a[9] = h[9] - h[8] * tmp1;
    a[5] = (h[5] + r * (dh[2] * dh[2] + dh[3] * dh[3]) + reg) - a[4] * tmp1;
    b[1] = (T(2) * dot(sxy, CA) + r * (dh[2] * mx[1] + dh[3] * mx[2])) - b[0] * tmp1;
    const T tmp2 = h[2] / a[0];
    const T tmp3 = h[3] / a[0];
    const T tmp4 = ((h[6]) - a[4] * tmp2) / a[5];
    a[14] = ((h[14] + r * (dh[7] * dh[5])) - h[12] * tmp2) - a[13] * tmp4;
    a[10] = ((h[10] + r * (dh[4] * dh[4] + dh[5] * dh[5]) + reg) - h[8] * tmp2) - a[9] * tmp4;
    b[2] = ((T(-2) * dot(sxy, ED) + r * (dh[4] * mx[3] + dh[5] * mx[5])) - b[0] * tmp2) - b[1] * tmp4;
    const T tmp5 = (h[7] - a[4] * tmp3) / a[5];
    const T tmp6 = (((h[11] + r * (dh[5] * dh[7])) - h[8] * tmp3) - a[9] * tmp5) / a[10];
    dx[3] = ((((T(-2) * dot(sxy, FD) + r * (dh[6] * mx[4] + dh[7] * mx[5])) - b[2] * tmp6) -
              b[0] * tmp3) - b[1] * tmp5) /
            ((((h[15] + r * (dh[6] * dh[6] + dh[7] * dh[7]) + reg) - h[12] * tmp3) - a[13] * tmp5) -
             a[14] * tmp6);
    dx[2] = (b[2] - (a[14] * dx[3])) / a[10];
    dx[1] = (b[1] - (a[9] * dx[2] + a[13] * dx[3])) / a[5];
    dx[0] = (b[0] - (a[4] * dx[1] + h[8] * dx[2] + h[12] * dx[3])) / a[0];
  }

  // Whether step_regular may be tried: edges of some 2^-20 to 2^20 (the sum of
  // their squares), a first vertex within 2^30.
  DH_HD bool regular() const {
    const double trace = h[0] + h[5] + h[10] + h[15];
    return trace >= 0x1p-40 && trace <= 0x1p40 && fabs(A0.x) <= 0x1p30 && fabs(A0.y) <= 0x1p30 &&
           fabs(A0.z) <= 0x1p30 && fabs(B0.x) <= 0x1p30 && fabs(B0.y) <= 0x1p30 &&
           fabs(B0.z) <= 0x1p30;
  }

  // step() on a regular pair: the same sums, with the penalty terms selected
  // instead of multiplied by 0, 1 or -1, and one reciprocal per pivot for its
  // quotients (238 vector instructions a step for 333 in the assembly; a pair's
  // four steps and the rest are 1,201 per wave of 64; the penalty over 363 pairs
  // of 80 x 80 triangles 153 -> 130 us).  The quotients are correctly rounded, as
  // division is, where no pivot is below 2^-10 of the trace, every non-zero
  // numerator is at least 2^-600 (`low` is the least binary exponent seen) and
  // the new x stays within 2^20, which with regular() keeps everything finite;
  // else the caller takes the general path.  The fused
  // doublings round once, as the sums after an exact product do.  (The sign of a zero quotient may
  // differ from division's; no sum here ends in a zero whose sign shows.)
  DH_HD bool step_regular(const double x[4], double reg, double dx[4], int& low) const {
    const bool c0 = x[0] >= 0.0, c1 = x[1] >= 0.0, c3 = x[2] >= 0.0, c4 = x[3] >= 0.0;
    const double over0 = x[0] + x[1] - 1.0, over1 = x[2] + x[3] - 1.0;
    const bool c2 = over0 <= 0.0, c5 = over1 <= 0.0;
    const double r0 = c0 ? 0.0 : r, r1 = c1 ? 0.0 : r, r2 = c2 ? 0.0 : r;
    const double r3 = c3 ? 0.0 : r, r4 = c4 ? 0.0 : r, r5 = c5 ? 0.0 : r;
    const double m2 = c2 ? 0.0 : over0, m5 = c5 ? 0.0 : over1;
    const V3<double> sxy = {
        (A0.x + (BA.x * x[0]) + (CA.x * x[1])) - (B0.x + (ED.x * x[2]) + (FD.x * x[3])),
        (A0.y + (BA.y * x[0]) + (CA.y * x[1])) - (B0.y + (ED.y * x[2]) + (FD.y * x[3])),
        (A0.z + (BA.z * x[0]) + (CA.z * x[1])) - (B0.z + (ED.z * x[2]) + (FD.z * x[3]))};
    const double least = (h[0] + h[5] + h[10] + h[15]) * 0x1p-10;
    const double p0 = h[0] + (r0 + r2) + reg;
    const double y0 = recip_regular(p0);
    const double a4 = h[4] + r2;
    const double tmp1 = quotient_regular(a4, p0, y0);
    const double tmp2 = quotient_regular(h[2], p0, y0);
    const double tmp3 = quotient_regular(h[3], p0, y0);
    const double b0 = fma(2.0, dot(sxy, BA), r * ((c0 ? 0.0 : x[0]) + m2));
    const double b1 = fma(2.0, dot(sxy, CA), r * ((c1 ? 0.0 : x[1]) + m2)) - b0 * tmp1;
    const double a13 = h[13] - h[12] * tmp1;
    const double a9 = h[9] - h[8] * tmp1;
    const double p1 = (h[5] + (r1 + r2) + reg) - a4 * tmp1;
    const double y1 = recip_regular(p1);
    const double n4 = h[6] - a4 * tmp2, n5 = h[7] - a4 * tmp3;
    const double tmp4 = quotient_regular(n4, p1, y1);
    const double tmp5 = quotient_regular(n5, p1, y1);
    const double a14 = ((h[14] + r5) - h[12] * tmp2) - a13 * tmp4;
    const double p2 = ((h[10] + (r3 + r5) + reg) - h[8] * tmp2) - a9 * tmp4;
    const double y2 = recip_regular(p2);
    const double b2 =
        (fma(-2.0, dot(sxy, ED), r * ((c3 ? 0.0 : x[2]) + m5)) - b0 * tmp2) - b1 * tmp4;
    const double n6 = ((h[11] + r5) - h[8] * tmp3) - a9 * tmp5;
    const double tmp6 = quotient_regular(n6, p2, y2);
    const double d3 = ((fma(-2.0, dot(sxy, FD), r * ((c4 ? 0.0 : x[3]) + m5)) - b2 * tmp6) -
                       b0 * tmp3) - b1 * tmp5;
    const double p3 =
        (((h[15] + (r4 + r5) + reg) - h[12] * tmp3) - a13 * tmp5) - a14 * tmp6;
    dx[3] = quotient_regular(d3, p3, recip_regular(p3));
    const double d2 = b2 - (a14 * dx[3]);
    dx[2] = quotient_regular(d2, p2, y2);
    const double d1 = b1 - (a9 * dx[2] + a13 * dx[3]);
    dx[1] = quotient_regular(d1, p1, y1);
    const double d0 = b0 - (a4 * dx[1] + h[8] * dx[2] + h[12] * dx[3]);
    dx[0] = quotient_regular(d0, p0, y0);
    low = least_exponent(least_exponent(low, a4), n4);
    low = least_exponent(least_exponent(low, n5), n6);
    low = least_exponent(least_exponent(low, d0), d1);
    low = least_exponent(least_exponent(low, d2), d3);
    return p0 >= least && p1 >= least && p2 >= least && p3 >= least;
  }

  DH_HD void points(const T x[4], V3<T>& P, V3<T>& Q) const {
    P = {A0.x + (BA.x * x[0]) + (CA.x * x[1]), A0.y + (BA.y * x[0]) + (CA.y * x[1]),
         A0.z + (BA.z * x[0]) + (CA.z * x[1])};
    Q = {B0.x + (ED.x * x[2]) + (FD.x * x[3]), B0.y + (ED.y * x[2]) + (FD.y * x[3]),
         B0.z + (ED.z * x[2]) + (FD.z * x[3])};
  }
};

template <typename T>
DH_HD T dot4(const T a[4], const T b[4]) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3];
}

// penaltySolver(..., bool& failed): `iters` >= 1 fixed steps (4 in the
// reference), regularisation x1e4 after every step, `failed` from the last
// step.  By step_regular where it takes the pair.  A pair that regular() refuses
// (NaN, extreme sizes) sends its whole wave to step(), so that no wave pays for
// both (2 in 100 pairs with a NaN, 2^20 pairs: 78 us with both, 60 by step()
// alone); `regular` (may be null) says which way a pair went.
template <typename T>
DH_HD bool penalty_fixed(const Tri<T>& A, const Tri<T>& B, const T x0[4], int iters, T max_err,
                         V3<T>& P, V3<T>& Q, bool* regular = nullptr) {
  Penalty<T> pen;
  pen.setup(A, B);
  T x[4] = {x0[0], x0[1], x0[2], x0[3]}, dx[4];
  T reg = pen.reg0;
  bool ok = whole_wave(pen.regular());
  int low = least_exponent(least_exponent(0, pen.h[2]), pen.h[3]);
#pragma unroll 1
  for (int i = 0; ok && i < iters; ++i) {
    if (i > 0)
      for (int q = 0; q < 4; ++q) x[q] -= dx[q];
    ok = pen.step_regular(x, reg, dx, low) && ok;
    reg = T(1E4) * reg;
    for (int q = 0; q < 4; ++q) ok = fabs(x[q] - dx[q]) <= 0x1p20 && ok;
  }
  ok = ok && low >= -600;
  if (regular) *regular = ok;
  if (!ok) {
    for (int q = 0; q < 4; ++q) x[q] = x0[q];
    reg = pen.reg0;
#pragma unroll 1
    for (int i = 0; i < iters; ++i) {
      if (i > 0)
        for (int q = 0; q < 4; ++q) x[q] -= dx[q];
      pen.step(x, reg, dx);
      reg = T(1E4) * reg;
    }
  }
  const bool failed = dot4(dx, dx) / dot4(x, x) > max_err * max_err;
  for (int q = 0; q < 4; ++q) x[q] -= dx[q];
  pen.points(x, P, Q);
  return failed;
}

// penaltySolver(..., int& its) (penalty.cpp:434-581): <= 16 steps, early exit.
// Returns the iteration count written by the reference, or -1 when it leaves
// the caller's value untouched (no convergence).
template <typename T>
DH_HD int penalty_adaptive(const Tri<T>& A, const Tri<T>& B, T max_err, V3<T>& P, V3<T>& Q) {
  Penalty<T> pen;
  pen.setup(A, B);
  T x[4] = {T(0.33), T(0.33), T(0.33), T(0.33)};
  T reg = pen.reg0;
  int its = -1;
  for (int i = 0; i < 16; ++i) {
    T dx[4];
    reg = i < 3 ? reg : T(1E5) * reg;
    pen.step(x, reg, dx);
    const T err = dot4(dx, dx) / dot4(x, x);
    if (err < max_err * max_err) {
      its = i;
      break;
    }
    x[0] = x[0] - dx[0];
    x[1] = x[1] - dx[1];
    x[2] = x[2] - dx[2];
    x[3] = x[3] - dx[3];
  }
  pen.points(x, P, Q);
  return its;
}

}  // namespace dh
