// Eikonal Fourier-Bessel tables (MEikonal::S3Density / S3Screening,
// src/MEikonal.cc:177-245), built with -ffp-contract=off: each term of a row's
// composite-Simpson sum is formed in the reference's operation order.
#include <hip/hip_runtime.h>

#include "gra_device.h"
#include "gra_fold.h"
#include "gra_kernels.h"
#include "gra_round15.h"

namespace {

using gra_hip::ElasticAmp;

// J0 by the rational / asymptotic fits of Abramowitz-Stegun 9.4 as tabulated by
// Clenshaw (NPL Math. Tables 5, 1962); the same approximation the reference
// evaluates (BESSJ0, libs/extmath.hpp:12-49).
__device__ __forceinline__ double bessj0(double X) {
  const double P1 = 1.0, P2 = -0.1098628627E-2, P3 = 0.2734510407E-4, P4 = -0.2073370639E-5,
               P5 = 0.2093887211E-6, Q1 = -0.1562499995E-1, Q2 = 0.1430488765E-3,
               Q3 = -0.6911147651E-5, Q4 = 0.7621095161E-6, Q5 = -0.9349451520E-7,
               R1 = 57568490574.0, R2 = -13362590354.0, R3 = 651619640.7, R4 = -11214424.18,
               R5 = 77392.33017, R6 = -184.9052456, S1 = 57568490411.0, S2 = 1029532985.0,
               S3 = 9494680.718, S4 = 59272.64853, S5 = 267.8532712, S6 = 1.0;
  if (X == 0.0) return 1.0;
  const double AX = fabs(X);
  if (AX < 8.0) {
    const double Y = X * X;
    const double FR = R1 + Y * (R2 + Y * (R3 + Y * (R4 + Y * (R5 + Y * R6))));
    const double FS = S1 + Y * (S2 + Y * (S3 + Y * (S4 + Y * (S5 + Y * S6))));
    return FR / FS;
  }
  // The fit's division, root and sincos as one reciprocal root and a reduction by
  // quarter turns (exact in the first step: the difference is a multiple of 2^-52 below 1)
  const double y = rsq64(AX);
  const double Z = 8.0 * (y * y);
  const double Y = Z * Z;
  const double XX = AX - 0.785398164;
  const double FP = __builtin_fma(Y, __builtin_fma(Y, __builtin_fma(Y, __builtin_fma(Y, P5, P4), P3), P2), P1);
  const double FQ = __builtin_fma(Y, __builtin_fma(Y, __builtin_fma(Y, __builtin_fma(Y, Q5, Q4), Q3), Q2), Q1);
  const double n = __builtin_rint(XX * 0.63661977236758138);
  const double th = __builtin_fma(-n, 6.123233995736766e-17, __builtin_fma(-n, 1.5707963267948966, XX));
  double sn, cs;
  sincos_quarter64(n, th, sn, cs);
  return 0.7978845605725179 * y * (FP * cs - Z * FQ * sn);  // sqrt(0.636619772 / AX) (..)
}

// The two integrands' factors at the quadrature nodes, a thread each; on the host these
// loops (pow, log, exp and sincos at 10001 nodes each) took 0.7 of 3.4 ms of a set-up, here
// 9 us.
//
// Each is multiplied by its node and by its weight 1, 2 or 4 in the composite Simpson sum
// (CSIntegral: h (f0 + 2 I_even + 4 I_odd + fN) / 3, include/Graniitti/MMath.h:378-394).
__device__ __forceinline__ double simpson_node(int q, int nf, double v) {
  return (q == 0 || q == nf) ? v : (q & 1) ? 4.0 * v : 2.0 * v;
}

// Density: pre_q = MEikonal::SingleAmpElastic(s, -kt_q^2), src/MEikonal.cc:139-154, with
// form::S3HPL, S3PomAlpha and ReggeEta (src/MForm.cc:382-426)
__global__ void k_density_pre(ElasticAmp A, int nf, double kmin, double kstep,
                              double* __restrict__ pre) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q > nf) return;
  const double kt = kmin + q * kstep, t = -(kt * kt);
  const double F = (1.0 / (1 - t / A.fc1)) * (1.0 / (1 - t / A.fc2));
  const double mpi2 = A.mpi * A.mpi, beta = (2.0 / 3.0) * A.gN;
  const double tau = 4.0 * mpi2 / fabs(t);
  const double sqrtau = msq(1 + tau);
  const double Fpi = 1.0 / (1.0 - t / A.fc3);
  const double hpl = (4.0 / tau) * (Fpi * Fpi) *
                     (2.0 * tau - pow(1.0 + tau, 1.5) * log((sqrtau + 1.0) / (sqrtau - 1.0)) +
                      log(1.0 / mpi2));
  const double pic = (beta * beta) * mpi2 / (32.0 * (GRA_PI * (GRA_PI * GRA_PI)));
  const double alpha = 1.0 + A.delta + A.slope * t - pic * hpl;
  double sn, cs;
  sincos(GRA_PI * alpha, &sn, &cs);
  const double a = ((A.gN * A.gN) * F) * F * pow(A.s, alpha);
  const double w = simpson_node(q, nf, kt);
  pre[2 * q] = -((1.0 + cs) / sn) * a * w;  // eta = -(1 + exp(-i pi alpha)) / sin(pi alpha)
  pre[2 * q + 1] = (sn / sn) * a * w;  // the factor is 1, or NaN at a pole of eta
}
// Screening: pre_q = i (1 - exp(i Omega(bt_q) / 2)), Omega between the density table's rows
// (x, re, im) as IArray1D::Interpolate1D takes it (src/MEikonal.cc:489-512)
__global__ void k_screening_pre(const double* __restrict__ T, int n_bt, double bmin, double bstep,
                                int nf, double step, double* __restrict__ pre) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q > nf) return;
  const double w = simpson_node(q, nf, bmin + q * step);
  double b = bmin + q * step;
  if (b < bmin) b = bmin;
  int i = (int)floor((b - bmin) / bstep);
  i = min(max(i, 0), n_bt - 1);
  const double* r = T + 3 * (size_t)i;
  const double dx = r[3] - r[0], f = b - r[0];
  const double re = r[1] + ((r[4] - r[1]) / dx) * f, im = r[2] + ((r[5] - r[2]) / dx) * f;
  const double e = exp(-im / 2.0);
  double sn, cs;
  sincos(re / 2.0, &sn, &cs);
  pre[2 * q] = e * sn * w;  // i (1 - e (cos + i sin))
  pre[2 * q + 1] = (1.0 - e * cs) * w;
}

// Two table rows per wave: lane l takes the quadrature nodes l, l + 64, ... (coalesced
// loads, and the same Bessel branch across the wave but at one boundary), whose parity is
// the lane's, and a butterfly adds the lanes' sums in a fixed order. With one thread per
// row 10001 rows were 40 blocks, each a serial chain of 10001 terms: 6.0 ms a table at 16%
// of the CUs. As waves they fill the chip, bound by the FP64 VALU: 0.52 ms with a division,
// a library root and sincos a term (207 instructions), 0.33 with bessj0's (150), 0.29 with
// the nodes' weights in pre and its loads shared by two rows (a set-up 1.35 -> 1.27 ms). Against
// 80-bit sums of the same fit the tables are off, relative to their largest value and for
// beams of 3.5 and 6.5 TeV, by 3.1e-15 and 2.9e-15 (density; 2.7e-15 and 3.6e-15 with the
// library functions) and 3.1e-15 and 0.9e-15 (screening; 5.2e-15 and 2.9e-15).
constexpr int kFbWaves = 4;  // of two rows each, per block
__global__ __launch_bounds__(64 * kFbWaves) void k_fb_table(int which, const double2* __restrict__ pre, int nf,
                                                  double qmin, double qstep, double xmin,
                                                  double xstep, int nrows, double factor,
                                                  const double* __restrict__ xs,
                                                  double* __restrict__ out) {
  const int i0 = 2 * (blockIdx.x * kFbWaves + (threadIdx.x >> 6));  // wave-uniform
  const int lane = threadIdx.x & 63;
  if (i0 >= nrows) return;
  double m[2], sr[2] = {0.0, 0.0}, si[2] = {0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = min(i0 + k, nrows - 1);  // an odd last row twice
    const double xv = xs ? xs[i] : xmin + i * xstep;
    m[k] = (which == 0) ? xv : msq(xv);
  }
  for (int q = lane; q <= nf; q += 64) {
    const double qv = qmin + q * qstep;
    const double2 p = pre[q];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double j0 = bessj0(m[k] * qv);
      sr[k] = __builtin_fma(p.x, j0, sr[k]);
      si[k] = __builtin_fma(p.y, j0, si[k]);
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      sr[k] += __shfl_xor(sr[k], o);
      si[k] += __shfl_xor(si[k], o);
    }
  // lanes 0 .. 2 and 32 .. 34 write a row each
  const int k = lane >> 5, i = i0 + k, c = lane & 31;
  if (i >= nrows) return;
  const double re = (((k ? sr[1] : sr[0]) * qstep) / 3.0) * factor;
  const double im = (((k ? si[1] : si[0]) * qstep) / 3.0) * factor;
  if (xs) {
    if (c < 2) out[2 * i + c] = c ? im : re;
  } else if (c < 3) {
    // a table row (x, re, im); values that need the text round trip stay as they are
    const double v = c == 0 ? xmin + i * xstep : c == 1 ? re : im;
    out[3 * i + c] = gra_hip::round15_exact(v) ? gra_hip::round15_arith(v) : v;
  }
}

}  // namespace

namespace gra_hip {

hipError_t launch_density_pre(const ElasticAmp& A, int nf, double kmin, double kstep, double* pre,
                              hipStream_t st) {
  hipLaunchKernelGGL(k_density_pre, dim3((nf + 256) / 256), dim3(256), 0, st, A, nf, kmin, kstep,
                     pre);
  return hipGetLastError();
}
hipError_t launch_screening_pre(const double* mbt, int n_bt, double bmin, double bstep, int nf,
                                double step, double* pre, hipStream_t st) {
  hipLaunchKernelGGL(k_screening_pre, dim3((nf + 256) / 256), dim3(256), 0, st, mbt, n_bt, bmin,
                     bstep, nf, step, pre);
  return hipGetLastError();
}
hipError_t launch_fb_table(int which, const double* pre, int nf, double qmin, double qstep,
                           double xmin, double xstep, int nrows, double factor, double* out,
                           hipStream_t st, const double* xs) {
  const int per = 2 * kFbWaves;
  hipLaunchKernelGGL(k_fb_table, dim3((nrows + per - 1) / per), dim3(64 * kFbWaves), 0, st, which,
                     (const double2*)pre, nf, qmin, qstep, xmin, xstep, nrows, factor, xs, out);
  return hipGetLastError();
}

}  // namespace gra_hip
