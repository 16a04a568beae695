// Device helpers shared by the kernels: Gauss-Legendre tables in constant memory, Bernstein
// bases and rational Bezier surface points.
#pragma once
#include <hip/hip_runtime.h>

#include "gauss_legendre_table.inc"

namespace bmi {

static __constant__ int c_gl_offset[52] = BMI_GL_OFFSET_INIT;
static __constant__ double c_gl_nodes[BMI_GL_TABLE_SIZE] = BMI_GL_NODES_INIT;
static __constant__ double c_gl_weights[BMI_GL_TABLE_SIZE] = BMI_GL_WEIGHTS_INIT;

template <int P>
struct Binom {
  static constexpr double c(int k) {
    double r = 1.0;
    for (int i = 1; i <= k; ++i) r = r * (P - k + i) / i;
    return r;
  }
};

// Bernstein basis of degree P at x (Spline/Bernstein.hpp:44-48)
template <int P>
__device__ __forceinline__ void bernstein_basis(double x, double* B) {
  if constexpr (P == 0) {
    B[0] = 1.0;
  } else {
    const double y = 1.0 - x;
    double xp[P + 1], yp[P + 1];
    xp[0] = 1.0, yp[0] = 1.0;
#pragma unroll
    for (int k = 1; k <= P; ++k) xp[k] = xp[k - 1] * x, yp[k] = yp[k - 1] * y;
#pragma unroll
    for (int k = 0; k <= P; ++k) B[k] = Binom<P>::c(k) * xp[k] * yp[P - k];
  }
}

// Bernstein basis and derivative of degree P (Bernstein.hpp:239-244)
template <int P>
__device__ __forceinline__ void bernstein_basis_der(double x, double* B, double* D) {
  if constexpr (P == 0) {
    B[0] = 1.0;
    D[0] = 0.0;
  } else {
    const double y = 1.0 - x;
    double xp[P + 1], yp[P + 1];
    xp[0] = 1.0, yp[0] = 1.0;
#pragma unroll
    for (int k = 1; k <= P; ++k) xp[k] = xp[k - 1] * x, yp[k] = yp[k - 1] * y;
#pragma unroll
    for (int k = 0; k <= P; ++k) B[k] = Binom<P>::c(k) * xp[k] * yp[P - k];
    double L[P];  // degree P-1 basis
#pragma unroll
    for (int k = 0; k < P; ++k) L[k] = Binom<P - 1>::c(k) * xp[k] * yp[P - 1 - k];
#pragma unroll
    for (int k = 0; k <= P; ++k) {
      const double lo = k >= 1 ? L[k - 1] : 0.0;
      const double hi = k <= P - 1 ? L[k] : 0.0;
      D[k] = P * (lo - hi);
    }
  }
}

// Rational Bezier patch with PD x PD homogeneous control points (cp[4*(i*PD+j)+k]):
// point and parameter derivatives by the quotient rule (Geometry/Patch.hpp:294-365).
// The contraction is done one direction at a time (x first, then y).
template <int PD>
__device__ __forceinline__ void surface_point(const double* __restrict__ cp, double s, double t, double X[3],
                                              double Ds[3], double Dt[3]) {
  double Bs[PD], Es[PD], Bt[PD], Et[PD];
  bernstein_basis_der<PD - 1>(s, Bs, Es);
  bernstein_basis_der<PD - 1>(t, Bt, Et);
  double v[4] = {0, 0, 0, 0}, vs[4] = {0, 0, 0, 0}, vt[4] = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < PD; ++j) {
    double r[4] = {0, 0, 0, 0}, rs[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < PD; ++i) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const double c = cp[4 * (i * PD + j) + k];
        r[k] += Bs[i] * c;
        rs[k] += Es[i] * c;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] += Bt[j] * r[k];
      vs[k] += Bt[j] * rs[k];
      vt[k] += Et[j] * r[k];
    }
  }
  const double bot = 1.0 / v[3];
  const double b2 = bot * bot;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    X[k] = v[k] * bot;
    Ds[k] = (vs[k] * v[3] - v[k] * vs[3]) * b2;
    Dt[k] = (vt[k] * v[3] - v[k] * vt[3]) * b2;
  }
}

// 1 / sqrt(s), s > 0: the hardware estimate (v_rsq_f64) refined by two steps of Newton's
// iteration for 1/sqrt, y <- y + y (1 - s y^2) / 2, each of which squares the relative error
// (the residual 1 - s y^2 formed with one rounding by an FMA); within a few ulps of the rounded
// quotient 1 / sqrt(s), for a third of the instructions of a square root and a division
__device__ __forceinline__ double rsqrt_newton(double s) {
  double y = __builtin_amdgcn_rsq(s);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double e = fma(-(s * y), y, 1.0);
    y = fma(0.5 * y, e, y);
  }
  return y;
}

// the same for every s >= 0: where the estimate is 0 or infinite (s infinite or 0) it is the result, of
// which the iteration would make a NaN
__device__ __forceinline__ double rsqrt_newton_any(double s) {
  const double y0 = __builtin_amdgcn_rsq(s);
  return __builtin_amdgcn_class(y0, 0x240) ? y0 : rsqrt_newton(s);  // +infinity, +0
}

// y = 1 / sqrt(s) as above and r = sqrt(s): s y corrected once by its residual, with the half of the iterate before
// (s y alone is off by up to two ulps, which a phase kappa r multiplies by its size)
__device__ __forceinline__ void rsqrt_sqrt_newton(double s, double& y, double& r) {
  const double y0 = __builtin_amdgcn_rsq(s);
  const double y1 = fma(0.5 * y0, fma(-(s * y0), y0, 1.0), y0), h = 0.5 * y1;
  y = __builtin_amdgcn_class(y0, 0x240) ? y0 : fma(h, fma(-(s * y1), y1, 1.0), y1);
  r = s * y;
  r = fma(h, fma(-r, r, s), r);
}

// a b + c with the constant c in scalar registers: from vector registers the compiler copies it first,
// into the accumulator of the two-operand form
__device__ __forceinline__ double fma_const(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// sine and cosine of the phases kappa r, |x| < SINCOS_NEAR: reduction to [-pi/4, pi/4] by subtracting
// n pi/2 in two parts (Cody and Waite, with fused multiply-adds) and the Taylor sums of both, whose first
// neglected terms are below 2.1e-18 there.  Absolute error within 3e-16 (checked against extended
// precision), a third of the library function's instructions.
constexpr double SINCOS_NEAR = 1048576.0;
__device__ __forceinline__ void sincos_near(double x, double* s, double* c) {
  // n = 2 x / pi rounded: adding 3 2^51 leaves the integer in the low bits
  const double t = fma(x, 0.63661977236758134308, 6755399441055744.0);
  const double n = t - 6755399441055744.0;
  double y = fma(-n, 1.57079632679489655800, x);  // pi / 2 rounded, and the rest
  y = fma(-n, 6.12323399573676603587e-17, y);
  const double z = y * y;
  double p = 1.0 / 355687428096000.0;  // 1 / 17!
  p = fma_const(p, z, -1.0 / 1307674368000.0);
  p = fma_const(p, z, 1.0 / 6227020800.0);
  p = fma_const(p, z, -1.0 / 39916800.0);
  p = fma_const(p, z, 1.0 / 362880.0);
  p = fma_const(p, z, -1.0 / 5040.0);
  p = fma_const(p, z, 1.0 / 120.0);
  p = fma_const(p, z, -1.0 / 6.0);
  const double sn = fma(y * z, p, y);
  double q = 1.0 / 20922789888000.0;  // 1 / 16!
  q = fma_const(q, z, -1.0 / 87178291200.0);
  q = fma_const(q, z, 1.0 / 479001600.0);
  q = fma_const(q, z, -1.0 / 3628800.0);
  q = fma_const(q, z, 1.0 / 40320.0);
  q = fma_const(q, z, -1.0 / 720.0);
  q = fma_const(q, z, 1.0 / 24.0);
  const double cs = fma(z * z, q, fma(-0.5, z, 1.0));
  const unsigned k = static_cast<unsigned>(__double2loint(t));  // quadrant k mod 4
  const double a = (k & 1) ? cs : sn, b = (k & 1) ? sn : cs;
  const unsigned sa = (k << 30) & 0x80000000u, sb = ((k + 1) << 30) & 0x80000000u;  // their signs
  *s = __hiloint2double(__double2hiint(a) ^ sa, __double2loint(a));
  *c = __hiloint2double(__double2hiint(b) ^ sb, __double2loint(b));
}

// the same for any x.  Beyond the reach of the reduction the library's function is kept out of line:
// inlined, its registers (a reduction by a long expansion of 2 / pi) would be those of every kernel
static __device__ __noinline__ double2 sincos_far(double x) {
  double s, c;
  sincos(x, &s, &c);
  return make_double2(s, c);
}
__device__ __forceinline__ void sincos_phase(double x, double* s, double* c) {
  if (!(fabs(x) < SINCOS_NEAR)) {
    const double2 v = sincos_far(x);
    *s = v.x, *c = v.y;
    return;
  }
  sincos_near(x, s, c);
}

}  // namespace bmi
