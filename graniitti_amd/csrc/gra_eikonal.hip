// Eikonal Fourier-Bessel tables (MEikonal::S3Density / S3Screening,
// src/MEikonal.cc:177-245), built with -ffp-contract=off: each term of a row's
// composite-Simpson sum is formed in the reference's operation order.
#include <hip/hip_runtime.h>

#include "gra_device.h"
#include "gra_kernels.h"

namespace {

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
  const double Z = 8.0 / AX;
  const double Y = Z * Z;
  const double XX = AX - 0.785398164;
  const double FP = P1 + Y * (P2 + Y * (P3 + Y * (P4 + Y * P5)));
  const double FQ = Q1 + Y * (Q2 + Y * (Q3 + Y * (Q4 + Y * Q5)));
  double sn, cs;
  sincos(XX, &sn, &cs);
  return sqrt(0.636619772 / AX) * (FP * cs - Z * FQ * sn);
}

// One wave per table row: lane l takes the quadrature nodes l, l + 64, ... (coalesced
// loads, and the same Bessel branch across the wave but at one boundary), whose parity is
// the lane's, and a butterfly adds the lanes' sums in a fixed order. With one thread per
// row 10001 rows were 40 blocks, each a serial chain of 10001 terms: 6.0 ms a table at 16%
// of the CUs. As waves they fill the chip, bound by the FP64 VALU (a division and a square
// root or a sincos per term): 0.47 ms.
constexpr int kFbWaves = 4;  // rows per block
__global__ __launch_bounds__(64 * kFbWaves) void k_fb_table(int which, const double* __restrict__ pre, int nf,
                                                  double qmin, double qstep, double xmin,
                                                  double xstep, int nrows, double factor,
                                                  const double* __restrict__ xs,
                                                  double* __restrict__ out) {
  const int i = blockIdx.x * kFbWaves + (threadIdx.x >> 6);  // wave-uniform
  const int lane = threadIdx.x & 63;
  if (i >= nrows) return;
  const double xv = xs ? xs[i] : xmin + i * xstep;
  const double m = (which == 0) ? xv : msq(xv);
  double fr = 0.0, fi = 0.0;  // this lane's interior nodes
  double er = 0.0, ei = 0.0;  // the end nodes f0 + fN (lanes 0 and nf mod 64)
  for (int q = lane; q <= nf; q += 64) {
    const double qv = qmin + q * qstep;
    const double j0 = bessj0(m * qv);
    const double tr = (pre[2 * q] * j0) * qv, ti = (pre[2 * q + 1] * j0) * qv;
    if (q == 0 || q == nf) {
      er += tr;
      ei += ti;
    } else {
      fr += tr;
      fi += ti;
    }
  }
  // CSIntegral: h (f0 + 2 I_even + 4 I_odd + fN) / 3, include/Graniitti/MMath.h:378-394
  const double w = (lane & 1) ? 4.0 : 2.0;
  double sr = er + w * fr, si = ei + w * fi;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    sr += __shfl_xor(sr, o);
    si += __shfl_xor(si, o);
  }
  if (lane != 0) return;
  out[2 * i] = ((sr * qstep) / 3.0) * factor;
  out[2 * i + 1] = ((si * qstep) / 3.0) * factor;
}

}  // namespace

namespace gra_hip {

hipError_t launch_fb_table(int which, const double* pre, int nf, double qmin, double qstep,
                           double xmin, double xstep, int nrows, double factor, double* out,
                           hipStream_t st, const double* xs) {
  hipLaunchKernelGGL(k_fb_table, dim3((nrows + kFbWaves - 1) / kFbWaves), dim3(64 * kFbWaves), 0, st,
                     which, pre, nf, qmin, qstep, xmin, xstep, nrows, factor, xs, out);
  return hipGetLastError();
}

}  // namespace gra_hip
