// The resonance sum of PP[RES(+CON)] (res_sum, gra_res.h) on point-folded FP64 nodes.
//
// The central system X = p3 + p4 does not move in the loop, so at every node of a point
// its mass, each resonance's Breit-Wigner and form factor, the decay angles and their
// spin traces, and the quantisation axis of the spin density are the same: they become
// one complex coefficient per resonance, formed once per point (lane r of the point's
// lanes forms that of resonance r). A node is left with the exchange factors of t and
// s_i = (X + p_i)^2, the photon fluxes, and the production traces.
//
// Traces. For a diagonal spin density the contraction Tr[f rho_rot f^dagger] of
// spin_trace is sum_a rho_aa |d^J_{lambda a}(theta)|^2, theta the angle between the
// momentum and the quantisation axis: a polynomial in its sin^2 and cos^2, with
// coefficients that are the same at every point (FoldResTab). Neither angles nor Wigner
// matrices are formed, and resonances with one density share their trace. (With
// off-diagonal elements the trace also follows the azimuth about the axis, which is
// rounding noise where both proton pT vanish: fold_process leaves those runs on the
// reference-order nodes.)
#pragma once

#include "gra_fold.h"
#include "gra_res.h"

// sum_a rho_aa |d_{lambda a}|^2 from u2 = sin^2, w2 = cos^2, for J = 2, lambda = 0
__device__ __forceinline__ double trace2(const double* __restrict__ c, double u2, double w2) {
#pragma clang fp contract(fast)
  const double C = 1.5 * w2 - 0.5;
  return u2 * (c[0] * u2 + c[1] * w2) + c[2] * (C * C);
}
// and for J = 1, summed over the rows lambda = +-1 with weight a and lambda = 0 with b
__device__ __forceinline__ double trace1(const double* __restrict__ c, double a, double b,
                                         double u2, double w2) {
#pragma clang fp contract(fast)
  return c[0] * (0.5 * a * (1.0 + w2) + 0.5 * b * u2) + c[1] * (a * u2 + b * w2);
}
__device__ __forceinline__ double sqrt_pos64(double x) {
  const double v = fmax(x, 1e-300);
  return x > 0.0 ? v * rsq64(v) : 0.0;
}

// Constants of one point's resonance nodes: the three components of q1 = p_a - p1 in
// the axis frame of the X rest frame, each linear in (kx, ky, dz = p_az - p1z, delta1),
// and s1 - s13 - s14, s2 - s23 - s24
struct FoldResPt {
  double v0[3], vx[3], vy[3], vz[3], vd[3];
  double S1, S2;
};
// Quantisation axis (spin::GetRhoRotation; FoldResTab excludes Gottfried-Jackson, whose
// axis moves with the node) and the frame's transverse vectors
struct AxisFrame {
  double t[3], p[3], n[3];
};
__device__ __forceinline__ void axis_frame(const RunParams& P, const dv4& X, double M,
                                           AxisFrame& A) {
  double nx = 0.0, ny = 0.0, nz = 1.0;
  if (P.spin_frame == GRA_FRAME_HX) {
    nx = X.x;
    ny = X.y;
    nz = X.z;
  } else if (P.spin_frame == GRA_FRAME_CS) {
    const dv4 b1 = boost_rest(X, M, P.pbeam1), b2 = boost_rest(X, M, P.pbeam2);
    const double n1 = sqrt(p3mod2(b1)), n2 = sqrt(p3mod2(b2));
    nx = b1.x / n1 - b2.x / n2;
    ny = b1.y / n1 - b2.y / n2;
    nz = b1.z / n1 - b2.z / n2;
  }
  const double nT = sqrt(nx * nx + ny * ny), nn = sqrt(nx * nx + ny * ny + nz * nz);
  const double ct = nn > 0.0 ? nz / nn : 1.0, st = nn > 0.0 ? nT / nn : 0.0;
  const double cp = nT > 0.0 ? nx / nT : 1.0, sp = nT > 0.0 ? ny / nT : 0.0;
  A.t[0] = ct * cp;
  A.t[1] = ct * sp;
  A.t[2] = -st;
  A.p[0] = -sp;
  A.p[1] = cp;
  A.p[2] = 0.0;
  A.n[0] = st * cp;
  A.n[1] = st * sp;
  A.n[2] = ct;
}
// sin^2 and cos^2 of the angle between p (in the X rest frame) and the axis
__device__ __forceinline__ void axis_angle(const AxisFrame& A, dv4 p, double& u2, double& w2) {
  const double a = A.t[0] * p.x + A.t[1] * p.y + A.t[2] * p.z;
  const double b = A.p[0] * p.x + A.p[1] * p.y + A.p[2] * p.z;
  const double c = A.n[0] * p.x + A.n[1] * p.y + A.n[2] * p.z;
  const double r2 = a * a + b * b + c * c;
  u2 = r2 > 0.0 ? (a * a + b * b) / r2 : 0.0;
  w2 = r2 > 0.0 ? c * c / r2 : 1.0;
}

// The node-independent factor of resonance r: Breit-Wigner, form factor, production
// coupling and decay amplitude, times 2 (1/m^2)^omega for a Pomeron-Pomeron resonance;
// with a production trace also its sqrt(2J + 1)
__device__ __forceinline__ cxd fold_res_coef(const RunParams& P, const FoldResTab& T, int r,
                                             const dv4& X, double m2, const AxisFrame& A,
                                             const dv4& d0, const dv4& d1) {
  const ResDev& R = P.res[r];
  const cxd bw = cbw(R, m2, mof(d0), mof(d1));
  double f = exp(-((m2 - R.M02) * (m2 - R.M02)) / R.gFF4) * R.gdec;
  cxd z = cmul(bw, cd(R.g_re, R.g_im));
  if (P.spin_dec) {
    if (R.J == 0) {
      z = cmul(z, cd(R.T_re, R.T_im));
    } else {
      double u2, w2;
      axis_angle(A, boost_rest(X, msq(m2), d0), u2, w2);
      const double tr = R.J == 1 ? trace1(T.c1[T.cls[r]], 0.0, 1.0, u2, w2)
                                 : trace2(T.c2[T.cls[r]], u2, w2);
      f *= sqrt(2.0 * R.J + 1.0) * msq(tr * (R.T_re * R.T_re + R.T_im * R.T_im));
    }
  }
  if (P.spin_gen && R.J > 0) f *= sqrt(2.0 * R.J + 1.0);
  if (!R.photo) f *= 2.0 * pow(1.0 / m2, P.omega);
  return cscale(z, f);
}

__device__ __forceinline__ void fold_res_point(const RunParams& P, const FoldRec& r,
                                               const FoldPt& F, const dv4& X, double m2,
                                               const AxisFrame& A, FoldResPt& R) {
#pragma clang fp contract(fast)
  const double M = sqrt(m2), i = 1.0 / (M * (X.e + M)), iM = 1.0 / M;
  // boost of q1 = (dz + d_a - delta1; -p1T + k, dz): q + X kappa
  const double kx = X.x * i, ky = X.y * i, kz = X.z * i - iM;
  const double k0 = -(kx * r.p1x + ky * r.p1y) - P.f_cb1 * iM;
  const double* e[3] = {A.t, A.p, A.n};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double eX = e[a][0] * X.x + e[a][1] * X.y + e[a][2] * X.z;
    R.v0[a] = eX * k0 - (e[a][0] * r.p1x + e[a][1] * r.p1y);
    R.vx[a] = eX * kx + e[a][0];
    R.vy[a] = eX * ky + e[a][1];
    R.vz[a] = eX * kz + e[a][2];
    R.vd[a] = eX * iM;
  }
  // s_i = m_i^2 + m_X^2 + 2 X.p_i, with 2 X.p1 = s13 + s14 - 2 m1^2 - m3^2 - m4^2
  const double m34 = m2of(r.dt[0]) + m2of(r.dt[1]);
  R.S1 = m2 - m34 - F.m1sq;
  R.S2 = m2 - m34 - F.m2sq;
}

// sqrt(coherent flux / x) of one photon (coh_flux, gra_res.h) with q = pT^2 + x^2 m_p^2:
//   flux / x = 16 pi alpha [(1 - x) pT^2 P1 / q^2 + x^2 G_M^2 / (4 q)] / x^2,
// the form factors' denominators collected under one reciprocal square root
__device__ __forceinline__ double fold_flux(const RunParams& P, double x, double t, double pt2) {
#pragma clang fp contract(fast)
  const double mp2 = P.tp_mp_ff * P.tp_mp_ff;
  const double tau = fabs(t) * P.f_i4mp2;
  const double d1 = 1.0 + tau * (10.98 + tau * (12.82 + tau * 21.97));
  const double d2 = 1.0 + tau * (10.97 + tau * (18.86 + tau * 6.55));
  const double n1 = 1.0 - 0.24 * tau, n2 = 2.792847337 * (1.0 + 0.12 * tau);
  const double x2 = x * x, q = pt2 + x2 * mp2;
  const double e = n1 * d2, m = n2 * d1;
  const double dd = d1 * d1, tp = 1.0 + tau;
  const double num = (1.0 - x) * pt2 * (e * e + tau * (m * m)) +
                     0.25 * x2 * q * tp * (n2 * n2) * dd;
  const double xq = x * q * (d1 * d2);
  const double den = xq * xq * tp;
  // sqrt(16 pi alpha) = 0.6056...
  return num > 0.0 ? 0.6056442417441775 * num * rsq64(fmax(num * den, 1e-300)) : 0.0;
}

// Resonance part of a node: Ze, the coefficient of the Pomeron-Pomeron factor
// 2^(a1 l1 + a2 l2), from the production traces of q1's angle to the axis (u2, w2).
// slots: the point's coefficient sums (re, im), st apart.
__device__ __forceinline__ void fold_res_node(const FoldResTab& T, const FoldResPt& R,
                                              const FoldKin& K, double kx, double ky,
                                              const double* slots, int st, cxd& Ze, double& u2,
                                              double& w2) {
#pragma clang fp contract(fast)
  double v[3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
    v[a] = __builtin_fma(
        R.vx[a], kx,
        __builtin_fma(R.vy[a], ky,
                      __builtin_fma(R.vz[a], K.dz, __builtin_fma(R.vd[a], K.dq, R.v0[a]))));
  const double vt = v[0] * v[0] + v[1] * v[1], vl = v[2] * v[2];
  const double ir = rcp64(vt + vl);
  u2 = vt * ir;
  w2 = vl * ir;
  Ze = cd(slots[0], slots[st]);
  for (int c = 0; c < T.n2; ++c) {
    const double s = sqrt_pos64(trace2(T.c2[T.prod2[c]], u2, w2));
    Ze.re = __builtin_fma(s, slots[(2 * c + 2) * st], Ze.re);
    Ze.im = __builtin_fma(s, slots[(2 * c + 3) * st], Ze.im);
  }
}
// Photon exchange on either side: sum_k sqrt(trace) B_k [gf2 e1 2^(x1 + beta_k t1) +
// gf1 e2 2^(x2 + beta_k t2)], e1, e2 the Regge phases of t1, t2 and x_i = a_i log2 s_i
__device__ __forceinline__ cxd fold_photo_node(const RunParams& P, const FoldResTab& T,
                                               const FoldPt& F, const FoldKin& K, double x1,
                                               double x2, cxd e1, cxd e2, double u2, double w2,
                                               const double* slots, int st) {
#pragma clang fp contract(fast)
  const double dz2 = 0.5 * ((F.w2 + K.del2) + (K.del1 - P.f_cb2));
  const double gf1 = fold_flux(P, K.dz * P.f_ibz, K.t1, K.a5);
  const double gf2 = fold_flux(P, dz2 * P.f_ibz, K.t2, K.a6);
  cxd A = cd(0.0, 0.0);
  double tr = 1.0;
  for (int k = 0; k < T.nph; ++k) {
    const int c = T.ph_cls[k];
    if (c >= 0 && (k == 0 || c != T.ph_cls[k - 1]))
      tr = sqrt_pos64(trace1(T.c1[c], 0.697 * 0.697, 0.169 * 0.169, u2, w2));
    const double g1 = tr * gf2 * exp2_64(__builtin_fma(T.beta[k], K.t1, x1));
    const double g2 = tr * gf1 * exp2_64(__builtin_fma(T.beta[k], K.t2, x2));
    const cxd G = cd(__builtin_fma(g1, e1.re, g2 * e2.re), __builtin_fma(g1, e1.im, g2 * e2.im));
    const int s = 2 * (1 + T.n2 + k);
    A = cadd(A, cmul(G, cd(slots[s * st], slots[(s + 1) * st])));
  }
  return A;
}

// ---------------------------------------------------------------------------
// The FP32-amplitude form (res_sum32 and regge_me4_32, gra_res.h) on folded kinematics:
// the same FP32 operations on the same FP64 scalars, with what the node does not change
// taken out of the loop. Per resonance and point: Breit-Wigner, form factor and decay
// amplitude (FoldRes32, formed by the resonance's lane); per node and spin: the rows
// g_a of the production trace, shared by the resonances of that spin; of the trace only
// the density's diagonal (fold_process), whose other terms add exact zeros.
// ---------------------------------------------------------------------------
struct FoldRes32 {
  cxf bw;     // times rff for a photoproduced resonance
  cxf decay;  // times the production coupling where there is no production trace
  float rff;
};
__device__ __forceinline__ FoldRes32 fold_res32_coef(const RunParams& P, int r, float m2, float mA,
                                                     float mB, float thd, float phd,
                                                     const RotD32& D) {
#pragma clang fp contract(fast)
  const ResDev& R = P.res[r];
  FoldRes32 z;
  z.bw = cbw32(R, m2, mA, mB);
  const float dm = m2 - (float)R.M02;
  z.rff = __expf(-(dm * dm) / (float)R.gFF4);
  z.decay = decay_amp32(P, R, thd, phd, D);
  if (R.photo) z.bw = rf_scale(z.bw, z.rff);
  if (!P.spin_gen || R.J == 0) z.decay = cfmul(cf((float)R.g_re, (float)R.g_im), z.decay);
  return z;
}

// g_a of the rows lambda_r (spin_trace32) for the diagonal entries a in mask
template <int J, int NROW>
__device__ __forceinline__ void fold_rows32(const int* lam, const float* T, float c, float s,
                                            float cd_, float sd, const RotD32& D, int mask,
                                            float* nrm) {
#pragma clang fp contract(fast)
  constexpr int n = 2 * J + 1;
  cxf ph_[n];
  ph_[J] = cf(1.f, 0.f);
#pragma unroll
  for (int k = 1; k <= J; ++k) {
    ph_[J + k] = cfmul(ph_[J + k - 1], cf(cd_, sd));
    ph_[J - k] = cf(ph_[J + k].re, -ph_[J + k].im);
  }
#pragma unroll
  for (int r = 0; r < NROW; ++r) {
    cxf f[n];
#pragma unroll
    for (int j = 0; j < n; ++j) f[j] = rf_scale(ph_[j], T[r] * wigner_d32(c, s, lam[r], j - J, J));
#pragma unroll
    for (int a = 0; a < n; ++a) {
      nrm[r * n + a] = 0.f;
      if (!(mask & (1 << a))) continue;  // wave-uniform
      cxf acc = cf(0.f, 0.f);
#pragma unroll
      for (int j = 0; j < n; ++j)
        acc = rf_add(acc, rf_scale(f[j], J == 1 ? D.d1[a][j] : D.d2[a][j]));
      nrm[r * n + a] = cfmul(acc, cf(acc.re, -acc.im)).re;
    }
  }
}
// The trace's terms in spin_trace32's order
template <int J, int NROW>
__device__ __forceinline__ float fold_trace32(const ResDev& R, const float* nrm) {
  constexpr int n = 2 * J + 1;
  float tr = 0.f;
#pragma unroll
  for (int r = 0; r < NROW; ++r)
#pragma unroll
    for (int a = 0; a < n; ++a) {
      const float term = (float)R.rho_re[a * n + a] * nrm[r * n + a];
      tr = tr + term;
    }
  return tr;
}

struct FoldRes32Pt {
  float m2, V;   // m_X^2 and its flux factor
  RotD32 D;
};
// MRegge::PhotoProp without its slope factor: eta e^{i ph t} and s^alpha
__device__ __forceinline__ cxf photo_eta32(const RunParams& P, float s, float t, float& pw) {
#pragma clang fp contract(fast)
  const float alpha = (float)P.regge_a0[0] + (float)P.regge_ap[0] * t;
  float sn, cs;
  __sincosf((float)((-GRA_PI / 2.0) * P.regge_ap[0]) * t, &sn, &cs);
  pw = rf_pow(s, alpha);
  return cfmul(cf((float)P.eta0_re[0], (float)P.eta0_im[0]), cf(cs, sn));
}

// The amplitude at a node: regge_me4_32 + res_sum32
__device__ __forceinline__ cxf fold_node32(const RunParams& P, const FoldResTab& T,
                                           const FoldRes32Pt& R32, const FoldRes32* coef, int st,
                                           const FoldKin& K, double s1d, double s2d, double dz2,
                                           dv4 q1b) {
#pragma clang fp contract(fast)
  const float s1 = (float)s1d, s2 = (float)s2d;
  const float t1 = (float)K.t1, t2 = (float)K.t2;
  const float FF_A = (float)P.gN_P * s3f32(P, t1), FF_B = (float)P.gN_P * s3f32(P, t2);
  const cxf pr12 = cfmul(regge_prop32(P, s1, t1), regge_prop32(P, s2, t2));
  const float cont = 2.f * FF_A * FF_B * R32.V;
  float n1[9], n2[5];
  if (P.spin_gen) {
    float thq, phq, s, c, sd, cd_;
    theta_phi32(q1b, thq, phq);
    __sincosf(0.5f * thq, &s, &c);
    __sincosf(phq - R32.D.phR, &sd, &cd_);
    if (T.mask1) {
      const int lam[3] = {1, 0, -1};
      const float T1[3] = {-0.697f, -0.169f, 0.697f};
      fold_rows32<1, 3>(lam, T1, c, s, cd_, sd, R32.D, T.mask1, n1);
    }
    if (T.mask2) {
      const int lam[1] = {0};
      const float T2[1] = {1.f};
      fold_rows32<2, 1>(lam, T2, c, s, cd_, sd, R32.D, T.mask2, n2);
    }
  }
  float gf1 = 0.f, gf2 = 0.f, pw1 = 0.f, pw2 = 0.f;
  cxf eta1 = cf(0.f, 0.f), eta2 = eta1;
  if (T.nph > 0) {
    const float x1 = (float)(K.dz * P.f_ibz), x2 = (float)(dz2 * P.f_ibz), mp = (float)P.tp_mp_ff;
    gf1 = sqrtf(fmaxf(coh_flux32(x1, t1, (float)sqrt_pos64(K.a5), mp) / x1, 0.f));
    gf2 = sqrtf(fmaxf(coh_flux32(x2, t2, (float)sqrt_pos64(K.a6), mp) / x2, 0.f));
    eta1 = photo_eta32(P, s1, t1, pw1);
    eta2 = photo_eta32(P, s2, t2, pw2);
  }
  cxf A = cf(0.f, 0.f);
  int c1 = -1, c2 = -1;  // the densities that sc1, sc2 = sqrt(2J + 1) sqrt(trace) belong to
  float sc1 = 0.f, sc2 = 0.f;
  for (int r = 0; r < P.nres; ++r) {
    const ResDev& R = P.res[r];
    const FoldRes32 z = coef[r * st];
    cxf spin = z.decay;
    if (P.spin_gen && R.J != 0) {
      const int c = T.cls[r];
      if (R.J == 1 && c != c1) {
        c1 = c;
        sc1 = sqrtf(2.f * R.J + 1.f) * sqrtf(fmaxf(fold_trace32<1, 3>(R, n1), 0.f));
      } else if (R.J == 2 && c != c2) {
        c2 = c;
        sc2 = sqrtf(2.f * R.J + 1.f) * sqrtf(fmaxf(fold_trace32<2, 1>(R, n2), 0.f));
      }
      spin = cfmul(rf_scale(cf((float)R.g_re, (float)R.g_im), R.J == 1 ? sc1 : sc2), z.decay);
    }
    if (R.photo) {
      const float B0 = (float)R.B0;
      const float F1 = (float)P.gN_P * __expf(0.5f * B0 * t1);
      const float F2 = (float)P.gN_P * __expf(0.5f * B0 * t2);
      const cxf A12 = rf_add(rf_scale(cfmul(z.bw, rf_scale(eta1, pw1 * F1)), gf2),
                             rf_scale(cfmul(z.bw, rf_scale(eta2, pw2 * F2)), gf1));
      A = rf_add(A, cfmul(A12, spin));
    } else {
      A = rf_add(A, rf_scale(cfmul(cfmul(pr12, z.bw), spin), cont * z.rff));
    }
  }
  if (P.process != GRA_PROC_RES) {
    Kin k;
    k.t1 = K.t1;
    k.t2 = K.t2;
    k.ss13 = K.s13;
    k.ss24 = K.s24;
    k.ss14 = K.s14;
    k.ss23 = K.s23;
    k.t_hat = K.th + P.m_prop2;
    k.u_hat = K.tu + P.m_prop2;
    A = rf_add(A, regge_me4_32(P, k));
  }
  return A;
}
