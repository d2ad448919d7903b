// Screening nodes of the FP64 unit in point-folded form.
//
// At a loop node only the protons change: p1T = p1T(tree) - k, p2T = p2T(tree) + k,
// and the central pair X = p3 + p4 stays. In light-cone components (p+- = E +- p_z)
// momentum conservation reads
//   p1+ = sqrt(s) - X+ - delta2,  p2- = sqrt(s) - X- - delta1,
//   delta1 = p1- = b5 / p1+,      delta2 = p2+ = b6 / p2-,     b = m^2 + pT^2,
// which is the solution that SolvePz (MKinematics.h:33-229) has in closed form. The
// deltas are of order pT^2 / sqrt(s) ~ 1e-4 GeV, so two steps of this iteration from
// the tree point's values are exact to FP64 rounding, without a square root or a
// division. Everything else is linear in the deltas and k:
//   t1     = (X+ + delta2 - d_a)(d_a - delta1) - |p1T|^2,      d_a = E - |p_z| of the beam
//   2p1.p3 = p1+ p3- + delta1 p3+ - 2 p1T.p3T,  and its mirror images.
// No quantity of order E^2 is squared and subtracted, so the rounding is that of the
// result, where the component form carries E^2 eps ~ 1e-8 GeV^2 (s_ij), 1e-12 (t).
// d_a is formed from the beam's rounded components (f_cb), the mass shell that the
// tree amplitude sees: m^2 / (E + |p_z|) differs by up to 1e-8 of itself and would
// move every node's t by the same 1e-11 GeV^2.
//
// launch_screen takes this form only for runs whose bound on delta / p+ keeps the
// dropped third order below FP64 rounding (fold_process).
#pragma once

#include "gra_device.h"

// ---------------------------------------------------------------------------
// Elementary functions on FP64 hardware seeds. Arguments are moderate and positive
// where they have to be (invariants of 1e-4 .. 1e9 GeV^2, exponents below 100, phases
// of a few revolutions), so the library's special cases are left out.
// ---------------------------------------------------------------------------
// 1 / x: one Newton step from the seed (relative error 2^-24 or better), then a
// residual correction
__device__ __forceinline__ double rcp64(double x) {
  const double r0 = __builtin_amdgcn_rcp(x);
  const double r1 = __builtin_fma(__builtin_fma(-x, r0, 1.0), r0, r0);
  return __builtin_fma(__builtin_fma(-x, r1, 1.0), r1, r1);
}
// 1 / sqrt(x), x > 0 (two Newton steps)
__device__ __forceinline__ double rsq64(double x) {
  double r = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  r = __builtin_fma(r, __builtin_fma(-hx * r, r, 0.5), r);
  return __builtin_fma(r, __builtin_fma(-hx * r, r, 0.5), r);
}
// x = 2^e m with m in [sqrt(1/2), sqrt(2)), x normal and positive
__device__ __forceinline__ double split64(double x, double& e) {
  const int hi = __double2hiint(x);
  const int n = (hi - 0x3FE6A09E) >> 20;
  e = (double)n;
  return __hiloint2double(hi - (n << 20), __double2loint(x));
}
// log2 of m from f = m - 1 and r = 1 / (m + 1) (to 2^-45 or better): with s = f r,
// log2 m = (2 / ln 2)(s + s^3 / 3 + ...), s^2 <= 0.0295; polynomial in s^2 of degree 7
// through the Chebyshev nodes (relative error 1.4e-17)
__device__ __forceinline__ double log2_tail(double f, double r, double e) {
  double s = f * r;
  s = __builtin_fma(__builtin_fma(-s, f + 2.0, f), r, s);
  const double z = s * s;
  double p = 0.2136589569431927;
  p = __builtin_fma(p, z, 0.2209130842311768);
  p = __builtin_fma(p, z, 0.262334352504183);
  p = __builtin_fma(p, z, 0.32059853491395984);
  p = __builtin_fma(p, z, 0.4121985858409005);
  p = __builtin_fma(p, z, 0.5770780163455203);
  p = __builtin_fma(p, z, 0.9617966939259898);
  p = __builtin_fma(p, z, 2.8853900817779268);
  return __builtin_fma(s, p, e);
}
// log2 of two and of four numbers: the reciprocals of the m + 1 (1.7 .. 2.4) share one
// seed, which runs at a quarter of the FMA rate
__device__ __forceinline__ void log2_two64(double x0, double x1, double& l0, double& l1) {
  double e0, e1;
  const double f0 = split64(x0, e0) - 1.0, f1 = split64(x1, e1) - 1.0;
  const double g0 = f0 + 2.0, g1 = f1 + 2.0, g = g0 * g1;
  double r = __builtin_amdgcn_rcp(g);
  r = __builtin_fma(__builtin_fma(-g, r, 1.0), r, r);
  l0 = log2_tail(f0, r * g1, e0);
  l1 = log2_tail(f1, r * g0, e1);
}
__device__ __forceinline__ void log2_four64(double x0, double x1, double x2, double x3, double& l0,
                                            double& l1, double& l2, double& l3) {
  double e0, e1, e2, e3;
  const double f0 = split64(x0, e0) - 1.0, f1 = split64(x1, e1) - 1.0;
  const double f2 = split64(x2, e2) - 1.0, f3 = split64(x3, e3) - 1.0;
  const double g0 = f0 + 2.0, g1 = f1 + 2.0, g2 = f2 + 2.0, g3 = f3 + 2.0;
  const double g01 = g0 * g1, g23 = g2 * g3, g = g01 * g23;
  double r = __builtin_amdgcn_rcp(g);
  r = __builtin_fma(__builtin_fma(-g, r, 1.0), r, r);
  const double r01 = r * g23, r23 = r * g01;
  l0 = log2_tail(f0, r01 * g1, e0);
  l1 = log2_tail(f1, r01 * g0, e1);
  l2 = log2_tail(f2, r23 * g3, e2);
  l3 = log2_tail(f3, r23 * g2, e3);
}
// 2^x: x = n + r, |r| <= 1/2, and the polynomial of degree 11 through the Chebyshev
// nodes (relative error 2.0e-17)
__device__ __forceinline__ double exp2_64(double x) {
  const double n = __builtin_rint(x);
  const double r = x - n;
  double p = 4.4558179083360645e-10;
  p = __builtin_fma(p, r, 7.074194297288521e-09);
  p = __builtin_fma(p, r, 1.0178057087733941e-07);
  p = __builtin_fma(p, r, 1.3215432535912375e-06);
  p = __builtin_fma(p, r, 1.5252733841556773e-05);
  p = __builtin_fma(p, r, 0.00015403530463724353);
  p = __builtin_fma(p, r, 0.001333355814640647);
  p = __builtin_fma(p, r, 0.009618129107587256);
  p = __builtin_fma(p, r, 0.055504108664821625);
  p = __builtin_fma(p, r, 0.24022650695910158);
  p = __builtin_fma(p, r, 0.6931471805599453);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_ldexp(p, (int)n);
}
// cos and sin of q pi / 2 + th, |th| <= pi / 4, q a whole number: polynomials in th^2
// through the Chebyshev nodes (relative errors 7e-18 and 1.3e-17)
__device__ __forceinline__ void sincos_quarter64(double q, double th, double& sn, double& cs) {
  const double z = th * th;
  double c = -1.1353379638297575e-11;
  c = __builtin_fma(c, z, 2.0875582380663952e-09);
  c = __builtin_fma(c, z, -2.7557313097790086e-07);
  c = __builtin_fma(c, z, 2.4801587283881152e-05);
  c = __builtin_fma(c, z, -0.0013888888888861095);
  c = __builtin_fma(c, z, 0.04166666666666645);
  c = __builtin_fma(c, z, -0.5);
  c = __builtin_fma(c, z, 1.0);
  double s = 1.5894736651849094e-10;
  s = __builtin_fma(s, z, -2.5050716974102745e-08);
  s = __builtin_fma(s, z, 2.755731337640013e-06);
  s = __builtin_fma(s, z, -0.000198412698286503);
  s = __builtin_fma(s, z, 0.008333333333320363);
  s = __builtin_fma(s, z, -0.16666666666666616);
  s = __builtin_fma(s * z, th, th);
  const int k = (int)q;
  const double a = (k & 1) ? s : c, b = (k & 1) ? c : s;
  cs = ((k + 1) & 2) ? -a : a;
  sn = (k & 2) ? -b : b;
}
// cos and sin of 2 pi x: x less its nearest quarter
__device__ __forceinline__ void sincos_rev64(double x, double& sn, double& cs) {
  const double q = __builtin_rint(4.0 * x);
  sincos_quarter64(q, __builtin_fma(-0.25, q, x) * 6.2831853071795865, sn, cs);
}

// Record of a screened point for the folded nodes, written by k_tree
struct FoldRec {
  double p1x, p1y, p2x, p2y;  // tree proton pT
  double m1, m2;              // proton masses from pfinal_orig[].M()
  dv4 dt[2];                  // central momenta
  double wfac;                // W / |M|^2 at the tree point
  double h0re, h0im;          // tree amplitude
  uint32_t pt, pad;
};

// Constants of one point's nodes
struct FoldPt {
  double q1x, q1y, q2x, q2y;  // -2 p1T, +2 p2T
  double i1, i2, del1, del2;  // 1 / p1+, 1 / p2-, and the deltas at the tree
  double a5, a6, m1sq, m2sq;  // pT^2 at the tree, proton masses squared
  double w1, w2;              // X+ - d_a, X- - d_b
  double p3m, p4m, p3p, p4p;  // E -+ p_z of the central pair
  double p3x, p3y, p4x, p4y;  // 2 pT of the central pair
  double S13, S24, S14, S23, T3, T4;  // s_ij, t^ - m^2 - t1, u^ - m^2 - t1 less their node terms
};

__device__ __forceinline__ void fold_point(const RunParams& P, const FoldRec& r, FoldPt& F) {
#pragma clang fp contract(fast)
  const dv4 p3 = r.dt[0], p4 = r.dt[1];
  F.p3m = p3.e - p3.z;
  F.p4m = p4.e - p4.z;
  F.p3p = p3.e + p3.z;
  F.p4p = p4.e + p4.z;
  const double Xp = F.p3p + F.p4p, Xm = F.p3m + F.p4m;
  F.m1sq = r.m1 * r.m1;
  F.m2sq = r.m2 * r.m2;
  F.a5 = r.p1x * r.p1x + r.p1y * r.p1y;
  F.a6 = r.p2x * r.p2x + r.p2y * r.p2y;
  const double b5 = F.m1sq + F.a5, b6 = F.m2sq + F.a6;
  const double rp = P.beamsum.e - Xp, rm = P.beamsum.e - Xm;
  double P1 = rp, P2 = rm;
#pragma unroll
  for (int k = 0; k < 3; ++k) {  // converges by delta / p+ per step
    const double d1 = b5 / P1, d2 = b6 / P2;
    P1 = rp - d2;
    P2 = rm - d1;
  }
  F.i1 = 1.0 / P1;
  F.i2 = 1.0 / P2;
  F.del1 = b5 * F.i1;
  F.del2 = b6 * F.i2;
  F.q1x = -2.0 * r.p1x;
  F.q1y = -2.0 * r.p1y;
  F.q2x = 2.0 * r.p2x;
  F.q2y = 2.0 * r.p2y;
  F.w1 = Xp - P.f_cb1;
  F.w2 = Xm - P.f_cb2;
  F.p3x = 2.0 * p3.x;
  F.p3y = 2.0 * p3.y;
  F.p4x = 2.0 * p4.x;
  F.p4y = 2.0 * p4.y;
  const double m3 = m2of(p3), m4 = m2of(p4);
  const double k13 = r.p1x * F.p3x + r.p1y * F.p3y, k14 = r.p1x * F.p4x + r.p1y * F.p4y;
  const double k23 = r.p2x * F.p3x + r.p2y * F.p3y, k24 = r.p2x * F.p4x + r.p2y * F.p4y;
  F.S13 = F.m1sq + m3 + rp * F.p3m - k13;
  F.S14 = F.m1sq + m4 + rp * F.p4m - k14;
  F.S23 = F.m2sq + m3 + rm * F.p3p - k23;
  F.S24 = F.m2sq + m4 + rm * F.p4p - k24;
  F.T3 = m3 - P.m_prop2 - F.w1 * F.p3m - P.f_cb1 * F.p3p - k13;
  F.T4 = m4 - P.m_prop2 - F.w1 * F.p4m - P.f_cb1 * F.p4p - k14;
}

// Kinematics of one node
struct FoldKin {
  double del1, del2, a5, a6;
  double t1, t2, s13, s24, s14, s23, th, tu;
  double dz, dq;  // of q1 = p_a - p1: z component, and z component + d_a - energy
};
__device__ __forceinline__ void fold_kin(const RunParams& P, const FoldPt& F, double kx, double ky,
                                         FoldKin& K) {
#pragma clang fp contract(fast)
  const double k2 = kx * kx + ky * ky;
  K.a5 = F.a5 + __builtin_fma(F.q1x, kx, __builtin_fma(F.q1y, ky, k2));
  K.a6 = F.a6 + __builtin_fma(F.q2x, kx, __builtin_fma(F.q2y, ky, k2));
  // delta1 = b5 / (p1+(tree) - (delta2 - delta2(tree))) = b5 i1 (1 + e + e^2 ...)
  const double d1 = (F.m1sq + K.a5) * F.i1, d2 = (F.m2sq + K.a6) * F.i2;
  double e1 = (d2 - F.del2) * F.i1, e2 = (d1 - F.del1) * F.i2;
  const double f1 = __builtin_fma(d1, e1, d1), f2 = __builtin_fma(d2, e2, d2);
  e1 = (f2 - F.del2) * F.i1;
  e2 = (f1 - F.del1) * F.i2;
  K.del1 = __builtin_fma(d1, __builtin_fma(e1, e1, e1), d1);
  K.del2 = __builtin_fma(d2, __builtin_fma(e2, e2, e2), d2);
  K.t1 = __builtin_fma(F.w1 + K.del2, P.f_cb1 - K.del1, -K.a5);
  K.t2 = __builtin_fma(F.w2 + K.del1, P.f_cb2 - K.del2, -K.a6);
  const double k3 = __builtin_fma(kx, F.p3x, ky * F.p3y), k4 = __builtin_fma(kx, F.p4x, ky * F.p4y);
  const double L3 = __builtin_fma(K.del1, F.p3p, __builtin_fma(-K.del2, F.p3m, k3));
  const double L4 = __builtin_fma(K.del1, F.p4p, __builtin_fma(-K.del2, F.p4m, k4));
  K.s13 = F.S13 + L3;
  K.s14 = F.S14 + L4;
  K.s23 = F.S23 - L3;  // (p1 + p2).p3 does not depend on the node
  K.s24 = F.S24 - L4;
  K.th = K.t1 + (F.T3 + L3);
  K.tu = K.t1 + (F.T4 + L4);
  K.dz = 0.5 * ((F.w1 + K.del1) + (K.del2 - P.f_cb1));
  K.dq = K.del1;
}

// t1, t2, t^, u^ and q1 of a node from the momentum components, in the reference's operation
// order. The component form rounds them at the 1e-12 GeV^2 level (E eps times an energy
// transfer), the tree amplitude with them, and a screened weight that nearly cancels
// against its tree amplitude shows it at 1e-10. Only nodes near the tree point matter:
// the loop's weight sits at small k, and further out the roundings differ from node to
// node and average. So the nodes below kFoldRefKt (13% of the Simpson grid), which
// come first in the node table, take this form and weights keep the reference's rounding
// to 3e-11; the others take it at 1e-10.
__device__ __forceinline__ void fold_kin_components(const RunParams& P, const FoldRec& r,
                                                    double kx, double ky, FoldKin& K) {
  const double p1x = r.p1x - kx, p1y = r.p1y - ky, p2x = r.p2x + kx, p2y = r.p2y + ky;
  const double pt1 = msq(p1x * p1x + p1y * p1y), pt2 = msq(p2x * p2x + p2y * p2y);
  const dv4 X = v4add(r.dt[0], r.dt[1]);
  const double p1z = solvepz(r.m1, r.m2, pt1, pt2, X.z, X.e, P);
  const double p2z = -(X.z + p1z);
  const dv4 q1 = v4sub(P.pbeam1, v4m(p1x, p1y, p1z, msq(r.m1 * r.m1 + pt1 * pt1 + p1z * p1z)));
  const dv4 q2 = v4sub(P.pbeam2, v4m(p2x, p2y, p2z, msq(r.m2 * r.m2 + pt2 * pt2 + p2z * p2z)));
  K.t1 = m2of(q1);
  K.t2 = m2of(q2);
  K.th = m2of(v4sub(q1, r.dt[0])) - P.m_prop2;
  K.tu = m2of(v4sub(q1, r.dt[1])) - P.m_prop2;
  K.dz = q1.z;
  K.dq = (q1.z + P.f_cb1) - q1.e;
}

// (1 - t / fc1)(1 - t / fc2), the inverse of form::S3F
__device__ __forceinline__ double inv_s3f(const RunParams& P, double t) {
#pragma clang fp contract(fast)
  return __builtin_fma(__builtin_fma(P.f_fpq, t, -P.f_fsq), t, 1.0);
}
// The continuum's modulus at a node without couplings and proton form factors:
//   ff(t^)^2 / t^' (s13/s0)^a1 (s24/s0)^a2 + the u term,  t^' = t^ - m^2,
// with ff = 1 / (1 - t^' / b_POW), as numerator and denominator
__device__ __forceinline__ void fold_regge(const RunParams& P, const FoldKin& K, double a1,
                                           double a2, double& num, double& den) {
#pragma clang fp contract(fast)
  const double off = P.f_ls0 * (a1 + a2);
  double l13, l24, l14, l23;
  log2_four64(K.s13, K.s24, K.s14, K.s23, l13, l24, l14, l23);
  const double et = exp2_64(__builtin_fma(a1, l13, __builtin_fma(a2, l24, -off)));
  const double eu = exp2_64(__builtin_fma(a1, l14, __builtin_fma(a2, l23, -off)));
  const double gt = __builtin_fma(-K.th, P.f_ibp, 1.0), gu = __builtin_fma(-K.tu, P.f_ibp, 1.0);
  const double Dt = gt * gt * K.th, Du = gu * gu * K.tu;
  num = __builtin_fma(et, Du, eu * Dt);
  den = Dt * Du;
}
