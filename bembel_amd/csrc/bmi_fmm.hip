// Interpolation-FMM kernels: coupling assembly and the H2 matrix-vector product.
//
// Restates H2Multipole::interpolateKernel (H2Matrix/H2Multipole.hpp:336-375), the forward and
// backward transformations (:380-469) and the leaf sweep of H2_time_dense_product_impl::run
// (H2Matrix/EigenHelper/H2DenseProduct.hpp:39-164).  Instead of one RHS column at a time and
// per-thread copies of the backward tree, every level is one launch over all clusters and
// right-hand sides; sums over leaves are owned by their row cluster (no atomics), so the
// result is deterministic.
//
// Vector layouts (S = 1 real or 2 complex doubles per scalar):
//   super vectors xs/ys: [component][element][local function] rows, one column per RHS
//   (column stride = nsuper), exactly the reference's super-space order.
//   multipole levels fw/bw: [cluster][rhs][row], row = comp*np2 + node.
#include <hip/hip_runtime.h>

#include <cstdlib>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "bmi_device.h"
#include "bmi_fmm.h"
#include "bmi_internal.h"

namespace bmi {

// ------------------------------------------------------------------ cluster node tables
// surface points of the Chebyshev nodes of every cluster of one level:
// out[(c*np2 + i)*CP_STRIDE] = x0 x1 x2 kappa ds0 ds1 ds2 dt0 dt1 dt2 (pad to 12)
template <int PD>
__global__ void k_cluster_points(const double* __restrict__ cp, int cp_stride, int level, int ncl,
                                 int np, const double* __restrict__ cheb, double* out) {
  const int np2 = np * np;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(ncl) * np2) return;
  const int c = static_cast<int>(gid / np2), i = static_cast<int>(gid % np2);
  const int patch = c >> (2 * level);
  const int m = c & ((1 << (2 * level)) - 1);
  int ix = 0, iy = 0;
  for (int l = level - 1; l >= 0; --l) {
    const int d = (m >> (2 * l)) & 3;
    ix = (ix << 1) | ((d == 1 || d == 2) ? 1 : 0);
    iy = (iy << 1) | (d >= 2 ? 1 : 0);
  }
  const double H = 1.0 / static_cast<double>(1 << level);
  const double u = cheb[i / np], v = cheb[i % np];
  double X[3], Ds[3], Dt[3];
  surface_point<PD>(cp + static_cast<int64_t>(patch) * cp_stride, ix * H + H * u, iy * H + H * v, X, Ds,
                    Dt);
  const double c0 = Ds[1] * Dt[2] - Ds[2] * Dt[1];
  const double c1 = Ds[2] * Dt[0] - Ds[0] * Dt[2];
  const double c2 = Ds[0] * Dt[1] - Ds[1] * Dt[0];
  double* o = out + gid * CP_STRIDE;
  o[0] = X[0], o[1] = X[1], o[2] = X[2];
  o[3] = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  o[4] = Ds[0], o[5] = Ds[1], o[6] = Ds[2];
  o[7] = Dt[0], o[8] = Dt[1], o[9] = Dt[2];
  o[10] = 0.0, o[11] = 0.0;
}

void launch_cluster_points(const bmi_space* s, int level, int np, const double* d_cheb, double* out,
                           hipStream_t st) {
  const int ncl = s->npatch << (2 * level);
  const int64_t total = static_cast<int64_t>(ncl) * np * np;
  const int blocks = static_cast<int>((total + 255) / 256);
  const int stride = 4 * s->pd * s->pd;
  if (s->pd == 5)
    hipLaunchKernelGGL(k_cluster_points<5>, dim3(blocks), dim3(256), 0, st, s->d_cp.ptr, stride, level,
                       ncl, np, d_cheb, out);
  else if (s->pd == 2)
    hipLaunchKernelGGL(k_cluster_points<2>, dim3(blocks), dim3(256), 0, st, s->d_cp.ptr, stride, level,
                       ncl, np, d_cheb, out);
  else
    throw Error(BMI_UNSUPPORTED, "patch degree not supported on the device");
  BMI_CHECK_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ coupling assembly
// F(i + (ii*nc+a)*np2, j + (jj*nc+b)*np2) of one admissible block, stored per component
// block (r = ii, c = jj) column-major with dimension cd = nc*np2
// (evaluateFMMInterpolation_impl: Laplace/SingleLayerOperator.hpp:87-110,
//  Helmholtz/SingleLayerOperator.hpp:87-110, Maxwell/SingleLayerOperator.hpp:90-120)
template <int KIND>
__global__ void k_coupling_assemble(const int4* __restrict__ leaves, int nleaves, int np2,
                                    const double* const* __restrict__ level_pts, double kre, double kim,
                                    double k2re, double k2im, double* out) {
  constexpr bool CPLX = KIND != BMI_LAPLACE_SL;
  constexpr int VD = KIND == BMI_MAXWELL_SL ? 2 : 1;
  constexpr int NC = KIND == BMI_MAXWELL_SL ? 2 : 1;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t per = static_cast<int64_t>(np2) * np2;
  if (gid >= per * nleaves) return;
  const int leaf = static_cast<int>(gid / per);
  const int q = static_cast<int>(gid % per);
  const int j = q / np2, i = q % np2;  // column-major: consecutive threads walk rows
  const int4 L = leaves[leaf];         // level, c1, c2, unused
  const double* pts = level_pts[L.x];
  const double* a = pts + (static_cast<int64_t>(L.y) * np2 + i) * CP_STRIDE;
  const double* b = pts + (static_cast<int64_t>(L.z) * np2 + j) * CP_STRIDE;
  const double d0 = a[0] - b[0], d1 = a[1] - b[1], d2 = a[2] - b[2];
  const double r = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
  const int cd = NC * np2;
  const int64_t blk = static_cast<int64_t>(cd) * cd;
  const int64_t base = static_cast<int64_t>(leaf) * VD * VD * blk;
  if constexpr (KIND == BMI_LAPLACE_SL) {
    out[base + static_cast<int64_t>(j) * cd + i] = (0.25 * M_1_PI) / r * a[3] * b[3];
  } else {
    double sn, cs;
    sincos_phase(kre * r, &sn, &cs);
    const double mag = (kim == 0.0 ? 1.0 : exp(kim * r)) * (0.25 * M_1_PI) / r;
    const double kr = mag * cs, ki = -mag * sn;
    if constexpr (KIND == BMI_HELMHOLTZ_SL) {
      const int64_t idx = base + static_cast<int64_t>(j) * cd + i;
      const double f = a[3] * b[3];
      out[2 * idx] = kr * f;
      out[2 * idx + 1] = ki * f;
    } else {
      // Maxwell: the kernel values alone, K(x_i, y_j) (np2 x np2 per leaf).  The reference's
      // interpolant per vector-component pair (r, c) is [[K t_r(x).t_c(y), 0], [0, -K/kappa^2]]
      // (t_0, t_1 the tangents d/ds, d/dt); the product applies the tangents and -1/kappa^2 per
      // cluster around one sweep over K (k_mx_prep, k_mx_finish), and bmi_h2_leaf_matrix expands a leaf
      const int64_t idx = static_cast<int64_t>(leaf) * per + static_cast<int64_t>(j) * np2 + i;
      out[2 * idx] = kr;
      out[2 * idx + 1] = ki;
      (void)k2re, (void)k2im;
    }
  }
}

void launch_coupling_assemble(int kind, const int4* d_leaves, int nleaves, int np2,
                              const double* const* d_level_pts, double kre, double kim, double* out,
                              hipStream_t st) {
  if (nleaves == 0) return;
  const int64_t total = static_cast<int64_t>(nleaves) * np2 * np2;
  const int blocks = static_cast<int>((total + 255) / 256);
  const double k2re = kre * kre - kim * kim, k2im = 2 * kre * kim;
  TimedScope ts("coupling_assemble", st);
  if (kind == BMI_LAPLACE_SL)
    hipLaunchKernelGGL(k_coupling_assemble<BMI_LAPLACE_SL>, dim3(blocks), dim3(256), 0, st, d_leaves,
                       nleaves, np2, d_level_pts, kre, kim, k2re, k2im, out);
  else if (kind == BMI_HELMHOLTZ_SL)
    hipLaunchKernelGGL(k_coupling_assemble<BMI_HELMHOLTZ_SL>, dim3(blocks), dim3(256), 0, st, d_leaves,
                       nleaves, np2, d_level_pts, kre, kim, k2re, k2im, out);
  else
    hipLaunchKernelGGL(k_coupling_assemble<BMI_MAXWELL_SL>, dim3(blocks), dim3(256), 0, st, d_leaves,
                       nleaves, np2, d_level_pts, kre, kim, k2re, k2im, out);
  BMI_CHECK_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ complex helpers
template <bool C>
struct Val;
template <>
struct Val<false> {
  double r;
  __device__ Val() : r(0) {}
  __device__ static Val load(const double* p, int64_t i) {
    Val v;
    v.r = p[i];
    return v;
  }
  __device__ void store(double* p, int64_t i) const { p[i] = r; }
  __device__ void fma_real(double a, const Val& x) { r += a * x.r; }
  __device__ void fma(const Val& a, const Val& x) { r += a.r * x.r; }
};
template <>
struct Val<true> {
  double r, i;
  __device__ Val() : r(0), i(0) {}
  __device__ static Val load(const double* p, int64_t k) {
    Val v;
    v.r = p[2 * k];
    v.i = p[2 * k + 1];
    return v;
  }
  __device__ void store(double* p, int64_t k) const {
    p[2 * k] = r;
    p[2 * k + 1] = i;
  }
  __device__ void fma_real(double a, const Val& x) {
    r += a * x.r;
    i += a * x.i;
  }
  __device__ void fma(const Val& a, const Val& x) {
    r += a.r * x.r - a.i * x.i;
    i += a.r * x.i + a.i * x.r;
  }
};

// ------------------------------------------------------------------ sparse T, T^T
// y[row, k] = alpha * sum_j A[row, j] (x[j, k] + x2[j, k]) + beta * y[row, k]   (x2 optional)
template <bool C>
__global__ void k_spmv(int nrows, int nrhs, const int* __restrict__ rp, const int* __restrict__ ci,
                       const double* __restrict__ v, const double* __restrict__ x, const double* __restrict__ x2,
                       int64_t ldx, double* y, int64_t ldy, double ar, double ai, double br, double bi, int use_beta) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(nrows) * nrhs) return;
  const int row = static_cast<int>(gid % nrows), k = static_cast<int>(gid / nrows);
  Val<C> acc;
  const double* xk = x + (C ? 2 : 1) * static_cast<int64_t>(k) * ldx;
  if (x2) {
    const double* x2k = x2 + (C ? 2 : 1) * static_cast<int64_t>(k) * ldx;
    for (int p = rp[row]; p < rp[row + 1]; ++p) {
      Val<C> a = Val<C>::load(xk, ci[p]);
      a.fma_real(1.0, Val<C>::load(x2k, ci[p]));
      acc.fma_real(v[p], a);
    }
  } else {
    for (int p = rp[row]; p < rp[row + 1]; ++p) acc.fma_real(v[p], Val<C>::load(xk, ci[p]));
  }
  double* yk = y + (C ? 2 : 1) * static_cast<int64_t>(k) * ldy;
  if constexpr (C) {
    double r = ar * acc.r - ai * acc.i, im = ar * acc.i + ai * acc.r;
    if (use_beta) {
      const double yr = yk[2 * row], yi = yk[2 * row + 1];
      r += br * yr - bi * yi;
      im += br * yi + bi * yr;
    }
    yk[2 * row] = r;
    yk[2 * row + 1] = im;
  } else {
    double r = ar * acc.r;
    if (use_beta) r += br * yk[row];
    yk[row] = r;
  }
}

// long rows (T^T: about (P+1)^4 entries per row): LPR lanes share a row and are summed by
// cross-lane shuffles
template <bool C, int LPR>
__global__ void k_spmv_sub(int nrows, int nrhs, const int* __restrict__ rp, const int* __restrict__ ci,
                           const double* __restrict__ v, const double* __restrict__ x, const double* __restrict__ x2,
                           int64_t ldx, double* y, int64_t ldy, double ar, double ai, double br, double bi,
                           int use_beta) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t rk = gid / LPR;
  const int l = static_cast<int>(gid % LPR);
  const bool valid = rk < static_cast<int64_t>(nrows) * nrhs;
  const int row = valid ? static_cast<int>(rk % nrows) : 0, k = valid ? static_cast<int>(rk / nrows) : 0;
  Val<C> acc;
  if (valid) {
    const double* xk = x + (C ? 2 : 1) * static_cast<int64_t>(k) * ldx;
    const double* x2k = x2 ? x2 + (C ? 2 : 1) * static_cast<int64_t>(k) * ldx : nullptr;
    for (int p = rp[row] + l; p < rp[row + 1]; p += LPR) {
      Val<C> a = Val<C>::load(xk, ci[p]);
      if (x2k) a.fma_real(1.0, Val<C>::load(x2k, ci[p]));
      acc.fma_real(v[p], a);
    }
  }
#pragma unroll
  for (int m = LPR / 2; m > 0; m >>= 1) {
    acc.r += __shfl_xor(acc.r, m, 64);
    if constexpr (C) acc.i += __shfl_xor(acc.i, m, 64);
  }
  if (!valid || l != 0) return;
  double* yk = y + (C ? 2 : 1) * static_cast<int64_t>(k) * ldy;
  if constexpr (C) {
    double r = ar * acc.r - ai * acc.i, im = ar * acc.i + ai * acc.r;
    if (use_beta) {
      const double yr = yk[2 * row], yi = yk[2 * row + 1];
      r += br * yr - bi * yi;
      im += br * yi + bi * yr;
    }
    yk[2 * row] = r;
    yk[2 * row + 1] = im;
  } else {
    double r = ar * acc.r;
    if (use_beta) r += br * yk[row];
    yk[row] = r;
  }
}

// ------------------------------------------------------------------ Maxwell far field
// The Maxwell coupling leaf (level, t, s) is K_ts (np2 x np2 kernel values at the Chebyshev nodes
// of clusters t and s), and its component block (r, c) in the reference is
//   [[K_ts o (t_r(x_i) . t_c(y_j)), 0], [0, -K_ts / kappa^2]]
// over (value moments, derivative moments) (Maxwell/SingleLayerOperator.hpp:90-120,
// H2Matrix.hpp:213-232).  Summed over c, the local expansions of component r are
//   value rows:      t_r(x_i) . sum_s K_ts u_s,   u_s(j) = sum_c t_c(y_j) fw_c[s](j)      (3-vectors)
//   derivative rows: -1/kappa^2 sum_s K_ts v_s,   v_s(j) = sum_c fw_c[s](np2 + j)
// so one sweep reads each K_ts once and multiplies it with four columns (u's three components
// and v), instead of four component blocks of (2 np2)^2 entries.
//
// tan: per cluster entry e (level offset + cluster) and node j, 6 doubles (t_0, t_1); Z: per entry
// 4 nrhs columns of np2 complex values, first (u_x, u_y) of every right-hand side, then (u_z, v): the
// sums of either half have the shape of one component's expansions (2 np2 = cd values) and overwrite the
// consumed moments.
__global__ void k_mx_prep(int64_t ne, int nrhs, int np2, int cd, const double* __restrict__ fw0,
                          const double* __restrict__ fw1, const double* __restrict__ tan, double* __restrict__ Z) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= ne * nrhs * np2) return;
  const int j = static_cast<int>(gid % np2);
  const int64_t ek = gid / np2;  // e * nrhs + k
  const int64_t e = ek / nrhs;
  const int64_t f = ek * cd;
  const double a0r = fw0[2 * (f + j)], a0i = fw0[2 * (f + j) + 1];
  const double a1r = fw1[2 * (f + j)], a1i = fw1[2 * (f + j) + 1];
  const double* t = tan + (e * np2 + j) * 6;
  double* z = Z + 2 * ((e * 4 * nrhs + 2 * (ek - e * nrhs)) * np2 + j);
  const int64_t half = static_cast<int64_t>(4) * nrhs * np2;  // doubles from (u_x, u_y) to (u_z, v)
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    double* zx = z + (x == 2 ? half : 2 * x * np2);
    zx[0] = t[x] * a0r + t[3 + x] * a1r;
    zx[1] = t[x] * a0i + t[3 + x] * a1i;
  }
  double* zv = z + half + 2 * np2;
  zv[0] = fw0[2 * (f + np2 + j)] + fw1[2 * (f + np2 + j)];
  zv[1] = fw0[2 * (f + np2 + j) + 1] + fw1[2 * (f + np2 + j) + 1];
}

// Both components' local expansions from the four columns of sums, in place: a thread owns node i of
// an entry and right-hand side.
__global__ void k_mx_finish(int64_t ne, int nrhs, int np2, int cd, const double* __restrict__ tan, double* w0,
                            double* w1, double qre, double qim) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= ne * nrhs * np2) return;
  const int i = static_cast<int>(gid % np2);
  const int64_t ek = gid / np2;  // e * nrhs + k
  const double* t = tan + (ek / nrhs * np2 + i) * 6;
  double2* a = reinterpret_cast<double2*>(w0) + ek * cd + i;
  double2* b = reinterpret_cast<double2*>(w1) + ek * cd + i;
  const double2 s[3] = {a[0], a[np2], b[0]};
  const double2 v = b[np2];
  double r0 = 0, i0 = 0, r1 = 0, i1 = 0;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    r0 += t[x] * s[x].x, i0 += t[x] * s[x].y;
    r1 += t[3 + x] * s[x].x, i1 += t[3 + x] * s[x].y;
  }
  const double2 d = make_double2(qre * v.x - qim * v.y, qre * v.y + qim * v.x);
  a[0] = make_double2(r0, i0), a[np2] = d;
  b[0] = make_double2(r1, i1), b[np2] = d;
}

// ------------------------------------------------------------------ wave-per-cluster sweeps
// The two HBM-bound sweeps of the matvec stream every stored leaf exactly once.  One 64-lane
// wave owns one row cluster (near field) or one target cluster (coupling): lane i owns row i,
// issues all DD (CD) column loads of a block before its first multiply-add, so each wave keeps a
// whole block in flight, and reads the source segment of the input, which is wave-uniform, via
// scalar loads.  One column; with BF16 copies of the coarsest coupling blocks RT right-hand sides share each
// block load.

// near field: ys[c*DD + i] = sum_blocks F (DD x DD) xs[c2*DD + ..].  UB blocks are loaded per iteration
// (their products are still added in block order, so every UB gives the same bits).
struct LeafArgs {
  int ncl;
  const int* rp;
  const int* src;
  const void* F;  // double, or float for the reduced-precision copy
  int64_t fstride;
  const double* xs;
  double* ys;
};

// wave-uniform double from lane l of v
__device__ __forceinline__ double lane_double(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

template <bool C, int DD, int UB, typename FT = double>
__device__ __forceinline__ void leaf_wave(int c, const LeafArgs& a) {
  constexpr int S = C ? 2 : 1;
  static_assert(DD <= 64, "leaf rows exceed a wave");
  const int lane = threadIdx.x & 63;
  const int i = lane < DD ? lane : 0;  // spare lanes shadow row 0 and store nothing
  const int p0 = a.rp[c], p1 = a.rp[c + 1];
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  const double* __restrict__ xs = a.xs;
  double ar = 0.0, ai = 0.0;
  // the source clusters of 64 entries at a time, one per lane: the block loop reads them with
  // lane reads instead of a dependent load per block
  for (int q0 = p0; q0 < p1; q0 += 64) {
    const int srcv = q0 + lane < p1 ? a.src[q0 + lane] : 0;
    const int q1 = p1 - q0 < 64 ? p1 : q0 + 64;
    for (int p = q0; p < q1; p += UB) {
      const int nb = q1 - p < UB ? q1 - p : UB;
      FT fr[UB][DD], fi[UB][C ? DD : 1];
      // the source vectors: one coalesced load per lane (lane j: entry j), issued before the
      // blocks and handed to every lane with lane reads.  Read straight from global memory, each
      // entry would be a load of one address by the whole wave, and these wait on each other
      double xr0[UB], xi0[UB];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (UB > 1 && u >= nb) break;
        const double* x = xs + S * (static_cast<int64_t>(__builtin_amdgcn_readlane(srcv, p + u - q0)) * DD + i);
        if constexpr (C) {
          const double2 v = *reinterpret_cast<const double2*>(x);
          xr0[u] = v.x, xi0[u] = v.y;
        } else {
          xr0[u] = x[0];
        }
      }
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (UB > 1 && u >= nb) break;
        const FT* f = F + S * (static_cast<int64_t>(p + u) * a.fstride);
#pragma unroll
        for (int j = 0; j < DD; ++j) {
          if constexpr (C && std::is_same<FT, double>::value) {
            const double2 v = *reinterpret_cast<const double2*>(f + 2 * (j * DD + i));
            fr[u][j] = v.x, fi[u][j] = v.y;
          } else if constexpr (C) {
            const float2 v = *reinterpret_cast<const float2*>(f + 2 * (j * DD + i));
            fr[u][j] = v.x, fi[u][j] = v.y;
          } else {
            fr[u][j] = f[j * DD + i];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (UB > 1 && u >= nb) break;
#pragma unroll
        for (int j = 0; j < DD; ++j) {
          const double f_r = static_cast<double>(fr[u][j]);
          const double xr = lane_double(xr0[u], j);
          if constexpr (C) {
            const double f_i = static_cast<double>(fi[u][j]);
            const double xi = lane_double(xi0[u], j);
            ar += f_r * xr - f_i * xi;
            ai += f_r * xi + f_i * xr;
          } else {
            ar += f_r * xr;
          }
        }
      }
    }
  }
  if (lane < DD) {
    double* y = a.ys + S * (static_cast<int64_t>(c) * DD + lane);
    y[0] = ar;
    if constexpr (C) y[1] = ai;
  }
}

template <bool C, int DD, int UB>
__global__ __launch_bounds__(256) void k_leaf_w(LeafArgs a) {
  const int c = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6));
  if (c >= a.ncl) return;
  leaf_wave<C, DD, UB>(c, a);
}

// coupling: bw[t][k][i] (+)= sum over blocks (t, s) of F (CD x CD) fw[s][k][:], all levels in one
// launch.  A wave owns one target; its 64 lanes form G = 64/CDP groups that take every G-th block
// and are summed with cross-lane shuffles at the end.
struct CplArgs {
  int ntgt, nrhs;
  const int2* tgt;
  const int* rp;
  const int* src;
  const void* F;
  int64_t fstride, fcomp;
  const int64_t* lvl_off;
  const double* fw;
  double* bw;
  int accumulate;
  const unsigned short* Fc;  // BF16 copies of the first ncoarse blocks (coarsest levels), or null
  int ncoarse;
  int ld;  // column stride of F blocks (cd, or cd padded to whole 16-byte row vectors for FP32)
  // symmetric sweeps: block index of each list entry, the partial vectors B^T x_t and the slot of
  // each entry's partial (its position in the gather order)
  const int* blk;
  double* part;
  const int* slot;
};

__device__ __forceinline__ double bf16_to_double(unsigned short b) {
  return static_cast<double>(__uint_as_float(static_cast<unsigned>(b) << 16));
}

template <bool C, typename FT, int CD, int RT, int UB>
__device__ __forceinline__ void coupling_wave(int t, const CplArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int CDP = CD <= 16 ? 16 : (CD <= 32 ? 32 : 64);
  constexpr int G = 64 / CDP;
  const int lane = threadIdx.x & 63;
  const int g = lane / CDP, li = lane % CDP;
  const int i = li < CD ? li : 0;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x] * a.nrhs;
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  const double* __restrict__ fw = a.fw;
  for (int k0 = 0; k0 < a.nrhs; k0 += RT) {
    double ar[RT], ai[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) ar[r] = 0.0, ai[r] = 0.0;
    for (int p = p0 + g; p < p1; p += G * UB) {
      double fr[UB][CD], fi[UB][C ? CD : 1];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (p + G * u >= p1) break;
        const int64_t fo = S * (static_cast<int64_t>(p + G * u) * a.fstride + a.fcomp);
        if (std::is_same<FT, float>::value && p + G * u < a.ncoarse) {
          const unsigned short* f = a.Fc + fo;
#pragma unroll
          for (int j = 0; j < CD; ++j) {
            fr[u][j] = bf16_to_double(f[S * (j * CD + i)]);
            if constexpr (C) fi[u][j] = bf16_to_double(f[S * (j * CD + i) + 1]);
          }
        } else {
          const FT* f = F + fo;
          const int ld = std::is_same<FT, double>::value ? CD : a.ld;  // FP64 blocks are unpadded
#pragma unroll
          for (int j = 0; j < CD; ++j) {
            fr[u][j] = static_cast<double>(f[S * (j * ld + i)]);
            if constexpr (C) fi[u][j] = static_cast<double>(f[S * (j * ld + i) + 1]);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        if (p + G * u >= p1) break;
        const int s2 = a.src[p + G * u];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const int k = k0 + r;
          if (k >= a.nrhs) break;
          const double* x = fw + S * (off + (static_cast<int64_t>(s2) * a.nrhs + k) * CD);
#pragma unroll
          for (int j = 0; j < CD; ++j) {
            if constexpr (C) {
              const double xr = x[2 * j], xi = x[2 * j + 1];
              ar[r] += fr[u][j] * xr - fi[u][j] * xi;
              ai[r] += fr[u][j] * xi + fi[u][j] * xr;
            } else {
              ar[r] += fr[u][j] * x[j];
            }
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
      for (int m = CDP; m < 64; m <<= 1) {
        ar[r] += __shfl_xor(ar[r], m, 64);
        if constexpr (C) ai[r] += __shfl_xor(ai[r], m, 64);
      }
    }
    if (g == 0 && li < CD) {
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const int k = k0 + r;
        if (k >= a.nrhs) break;
        double* y = a.bw + S * (off + (static_cast<int64_t>(T.y) * a.nrhs + k) * CD + li);
        if (a.accumulate) {
          ar[r] += y[0];
          if constexpr (C) ai[r] += y[1];
        }
        y[0] = ar[r];
        if constexpr (C) y[1] = ai[r];
      }
    }
  }
}

template <bool C, typename FT, int CD, int RT, int UB>
__global__ __launch_bounds__(256) void k_coupling_w(CplArgs a) {
  const int t = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6));
  if (t >= a.ntgt) return;
  coupling_wave<C, FT, CD, RT, UB>(t, a);
}

// Real FP64 blocks, one RHS: each lane loads two adjacent rows of a column (16 bytes, as the
// complex kernels do) instead of one, so a load instruction moves up to 1 KiB.  Near field: the
// DD/2 lanes of a group cover a column, the NG = 64/(DD/2) groups split the columns of the same
// block (x of a column is read per lane, broadcast within the group); coupling: a group of CD/2
// lanes owns a block, NG groups take every NG-th block.  Group sums are combined with shuffles.
// vector of RPL consecutive rows of one column as one 16-byte load
template <bool C, typename FT>
struct RowVec {
  static constexpr int RPL = 16 / ((C ? 2 : 1) * static_cast<int>(sizeof(FT)));  // rows per lane
  FT r[RPL], i[C ? RPL : 1];  // kept in the storage type, widened where multiplied
  __device__ __forceinline__ void load(const FT* p) {
    if constexpr (std::is_same<FT, double>::value && !C) {
      const double2 v = *reinterpret_cast<const double2*>(p);
      r[0] = v.x, r[1] = v.y;
    } else if constexpr (std::is_same<FT, double>::value) {
      const double2 v = *reinterpret_cast<const double2*>(p);
      r[0] = v.x, i[0] = v.y;
    } else if constexpr (!C) {
      const float4 v = *reinterpret_cast<const float4*>(p);
      r[0] = v.x, r[1] = v.y, r[2] = v.z, r[3] = v.w;
    } else {
      const float4 v = *reinterpret_cast<const float4*>(p);
      r[0] = v.x, i[0] = v.y, r[1] = v.z, i[1] = v.w;
    }
  }
};

template <bool C, typename FT, int DD, int UB>
__device__ __forceinline__ void leaf_wave_v(int c, const LeafArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int RPL = RowVec<C, FT>::RPL;
  constexpr int H = DD / RPL;
  constexpr int NG = 64 / H;
  constexpr int JC = (DD + NG - 1) / NG;
  const int lane = threadIdx.x & 63;
  const int g0 = lane / H;
  const int g = g0 < NG ? g0 : NG - 1;  // spare lanes repeat the last group and store nothing
  const int l = lane - g0 * H < H ? lane - g0 * H : 0;
  const int p0 = a.rp[c], p1 = a.rp[c + 1];
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  const double* __restrict__ xs = a.xs;
  double yr[RPL], yi[C ? RPL : 1];
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    yr[q] = 0.0;
    if constexpr (C) yi[q] = 0.0;
  }
  // the source clusters of 64 entries at a time, one per lane, read with lane reads; the source
  // vector of a block with one coalesced load (lane j: entry j), its entries handed to the
  // groups' lanes by lane permutes (read straight from global memory, each entry would be a
  // load of the same few addresses by the whole wave, waiting on the source index)
  const int le = lane < DD ? lane : 0;
  for (int q0 = p0; q0 < p1; q0 += 64) {
    const int srcv = q0 + lane < p1 ? a.src[q0 + lane] : 0;
    const int q1 = p1 - q0 < 64 ? p1 : q0 + 64;
    for (int p = q0; p < q1; p += UB) {
      RowVec<C, FT> fv[UB][JC];
      double xor_[UB], xoi[UB];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        const int pu = p + u < q1 ? p + u : q1 - 1;
        const double* x = xs + S * (static_cast<int64_t>(__builtin_amdgcn_readlane(srcv, pu - q0)) * DD + le);
        if constexpr (C) {
          const double2 v = *reinterpret_cast<const double2*>(x);
          xor_[u] = v.x, xoi[u] = v.y;
        } else {
          xor_[u] = x[0], xoi[u] = 0.0;
        }
        const FT* f = F + S * (static_cast<int64_t>(pu) * a.fstride);
#pragma unroll
        for (int jj = 0; jj < JC; ++jj) {
          const int j = g * JC + jj < DD ? g * JC + jj : DD - 1;
          fv[u][jj].load(f + S * (j * DD + RPL * l));
        }
      }
#pragma unroll
      for (int u = 0; u < UB; ++u)
#pragma unroll
        for (int jj = 0; jj < JC; ++jj) {
          const bool in = g * JC + jj < DD && p + u < q1;
          const int j = g * JC + jj < DD ? g * JC + jj : DD - 1;
          const double xr = in ? __shfl(xor_[u], j, 64) : 0.0;
          const double xi = C && in ? __shfl(xoi[u], j, 64) : 0.0;
#pragma unroll
          for (int q = 0; q < RPL; ++q) {
            const double fr = static_cast<double>(fv[u][jj].r[q]);
            if constexpr (C) {
              const double fi = static_cast<double>(fv[u][jj].i[q]);
              yr[q] += fr * xr - fi * xi;
              yi[q] += fr * xi + fi * xr;
            } else {
              yr[q] += fr * xr;
            }
          }
        }
    }
  }
  // group 0 collects the other groups' sums
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    double sr = yr[q], si = C ? yi[q] : 0.0;
#pragma unroll
    for (int k = 1; k < NG; ++k) {
      const int src = lane + k * H < 64 ? lane + k * H : lane;
      const double tr = __shfl(yr[q], src, 64);
      const double ti = C ? __shfl(yi[q], src, 64) : 0.0;
      if (lane + k * H < 64) sr += tr, si += ti;
    }
    yr[q] = sr;
    if constexpr (C) yi[q] = si;
  }
  if (g0 == 0) {
    double* y = a.ys + S * (static_cast<int64_t>(c) * DD + RPL * l);
#pragma unroll
    for (int q = 0; q < RPL; ++q) {
      y[S * q] = yr[q];
      if constexpr (C) y[S * q + 1] = yi[q];
    }
  }
}

// FP32 coupling blocks with columns padded to whole 16-byte row vectors (LD rows): a group of
// LD / RPL lanes owns a block, NG groups take every NG-th block; padding rows are zero.
template <bool C, int CD, int LD, int UB>
__device__ __forceinline__ void coupling_wave_v(int t, const CplArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int RPL = RowVec<C, float>::RPL;
  constexpr int H = LD / RPL;
  constexpr int NG = 64 / H;
  const int lane = threadIdx.x & 63;
  const int g0 = lane / H;
  const int g = g0 < NG ? g0 : NG - 1;
  const int l = lane - g0 * H < H ? lane - g0 * H : 0;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const float* __restrict__ F = static_cast<const float*>(a.F);
  double yr[RPL], yi[C ? RPL : 1];
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    yr[q] = 0.0;
    if constexpr (C) yi[q] = 0.0;
  }
  for (int p = p0 + g; p < p1; p += NG * UB) {
    RowVec<C, float> fv[UB][CD];
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int pu = p + NG * u < p1 ? p + NG * u : p;
      const float* f = F + S * (static_cast<int64_t>(pu) * a.fstride + a.fcomp);
#pragma unroll
      for (int j = 0; j < CD; ++j) fv[u][j].load(f + S * (j * LD + RPL * l));
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const bool ok = p + NG * u < p1;
      const int pu = ok ? p + NG * u : p;
      const double* x = a.fw + S * (off + static_cast<int64_t>(a.src[pu]) * CD);
      // FP32 entries, FP64 sums (FP64 multiply-adds issue at the FP32 rate here, and the reduced
      // operator's accuracy sets the Krylov step count)
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        const double xr = ok ? x[S * j] : 0.0;
        const double xi = (C && ok) ? x[S * j + 1] : 0.0;
#pragma unroll
        for (int q = 0; q < RPL; ++q) {
          const double fr = static_cast<double>(fv[u][j].r[q]);
          if constexpr (C) {
            const double fi = static_cast<double>(fv[u][j].i[q]);
            yr[q] += fr * xr - fi * xi;
            yi[q] += fr * xi + fi * xr;
          } else {
            yr[q] += fr * xr;
          }
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    double sr = yr[q], si = C ? yi[q] : 0.0;
#pragma unroll
    for (int k = 1; k < NG; ++k) {
      const int src = lane + k * H < 64 ? lane + k * H : lane;
      const double tr = __shfl(yr[q], src, 64);
      const double ti = C ? __shfl(yi[q], src, 64) : 0.0;
      if (lane + k * H < 64) sr += tr, si += ti;
    }
    yr[q] = sr;
    if constexpr (C) yi[q] = si;
  }
  if (g0 == 0) {
    double* y = a.bw + S * (off + static_cast<int64_t>(T.y) * CD);
#pragma unroll
    for (int q = 0; q < RPL; ++q) {
      const int row = RPL * l + q;
      if (row >= CD) continue;
      y[S * row] = yr[q];
      if constexpr (C) y[S * row + 1] = yi[q];
    }
  }
}

template <int CD, int UB>
__device__ __forceinline__ void coupling_wave_r2(int t, const CplArgs& a) {
  constexpr int H = CD / 2;
  constexpr int NG = 64 / H;  // H is a power of two here
  const int lane = threadIdx.x & 63;
  const int g = lane / H, l = lane % H;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const double* __restrict__ F = static_cast<const double*>(a.F);
  double y0 = 0.0, y1 = 0.0;
  for (int p = p0 + g; p < p1; p += NG * UB) {
    double2 fv[UB][CD];
    double xv[UB][CD];
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const bool ok = p + NG * u < p1;
      const int pu = ok ? p + NG * u : p;
      const double* f = F + static_cast<int64_t>(pu) * a.fstride + a.fcomp;
      const double* x = a.fw + off + static_cast<int64_t>(a.src[pu]) * CD;
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        fv[u][j] = *reinterpret_cast<const double2*>(f + j * CD + 2 * l);
        xv[u][j] = ok ? x[j] : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < UB; ++u)
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        y0 += fv[u][j].x * xv[u][j];
        y1 += fv[u][j].y * xv[u][j];
      }
  }
#pragma unroll
  for (int m = H; m < 64; m <<= 1) {
    y0 += __shfl_xor(y0, m, 64);
    y1 += __shfl_xor(y1, m, 64);
  }
  if (g == 0) {
    double* y = a.bw + off + static_cast<int64_t>(T.y) * CD + 2 * l;
    y[0] = y0;
    y[1] = y1;
  }
}

// ------------------------------------------------------------------ symmetric coupling (single RHS)
// Coupling blocks of the scalar kernels come in transposed pairs: the block of (level, s, t) is the
// transpose of (level, t, s) (the kernel is symmetric in its arguments, the node sets are per
// level). A single-RHS sweep can therefore read only the upper blocks (t < s): the wave owning t
// adds B x_s to its own rows and leaves u = B^T x_t, which belongs to s, in a per-block partial
// vector; k_sym_gather then adds each target's partials in a fixed order (no atomics, the same
// bits on every run). Each upper block is read once for both products.

// Column sums of a W-lane group (W a power of two, groups W-aligned within the wave): lane li
// supplies its partial value v(j) of every column j < W*R; on return out[r] holds the group's sum
// of column R*li + r. Recursive halving: under mask m each lane keeps the half of its columns
// selected by (li & m) and adds its partner's copy of that half.
// the partner value of a recursive-halving round with mask m inside rows of 16 lanes, through a
// DPP lane move (no LDS): m = 8 pairs lane i with 15 - i (row mirror), m = 4 with 7 - i (half-row
// mirror), m = 2 and 1 with i ^ 2 and i ^ 1 (quad permutes).  Each partner differs from the lane
// in bit m and, with the rounds taken from the largest mask down, agrees in every bit an earlier
// round split on, so both hold the same columns.  Larger masks go through the LDS permute.
template <int M>
__device__ __forceinline__ double halving_partner(double v) {
  constexpr int CTRL = M == 8 ? 0x140 : M == 4 ? 0x141 : M == 2 ? 0x4E : 0xB1;
  if constexpr (M >= 16) {
    return __shfl_xor(v, M, 64);
  } else {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
  }
}

// rounds m, m / 2, ..., 1 of the recursive halving on h (m * 2 * R live values)
template <int M, int R, int NH>
__device__ __forceinline__ void halving_rounds(int li, double (&h)[NH]) {
  if constexpr (M >= 1) {
    const bool up = (li & M) != 0;
#pragma unroll
    for (int k = 0; k < M * R; ++k) {
      const double lo = h[k], hi = h[k + M * R];
      h[k] = (up ? hi : lo) + halving_partner<M>(up ? lo : hi);
    }
    halving_rounds<M / 2, R>(li, h);
  }
}

template <int W, int R, class V>
__device__ __forceinline__ void group_column_sums(int li, V v, double (&out)[R]) {
  constexpr int N = W * R;
  if constexpr (W == 1) {
#pragma unroll
    for (int r = 0; r < R; ++r) out[r] = v(r);
  } else {
    constexpr int M0 = W / 2;
    double h[N / 2];
    const bool up0 = (li & M0) != 0;
#pragma unroll
    for (int k = 0; k < N / 2; ++k) {
      const double lo = v(k), hi = v(k + N / 2);
      h[k] = (up0 ? hi : lo) + halving_partner<M0>(up0 ? lo : hi);
    }
    halving_rounds<M0 / 2, R>(li, h);
#pragma unroll
    for (int r = 0; r < R; ++r) out[r] = h[r];
  }
}

__host__ __device__ constexpr int pow2_at_least(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// one row per lane: FP64 blocks (complex, or real sizes without the two-row form), or the
// padded FP32 copy of complex blocks (column stride LD; 8-byte entries, half the registers of
// the 16-byte row-vector form)
template <bool C, int CD, int UB, typename FT = double, int LD = CD>
__device__ __forceinline__ void coupling_wave_sym(int t, const CplArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int W = pow2_at_least(CD);
  static_assert(W <= 64, "block rows exceed a wave");
  constexpr int G = 64 / W;
  const int lane = threadIdx.x & 63;
  const int g = lane / W, li = lane % W;
  const bool act = li < CD;
  const int i = act ? li : 0;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  const double* xt = a.fw + S * (off + static_cast<int64_t>(T.y) * CD + i);
  const double tr = act ? xt[0] : 0.0, ti = (C && act) ? xt[1] : 0.0;
  double ar = 0.0, ai = 0.0;
  for (int p = p0 + g; p < p1; p += G * UB) {
    FT fr[UB][CD], fi[UB][C ? CD : 1];
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int pu = p + G * u < p1 ? p + G * u : p;
      const FT* f = F + S * (static_cast<int64_t>(a.blk[pu]) * a.fstride + a.fcomp);
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        if constexpr (C && std::is_same<FT, float>::value) {
          const float2 v = *reinterpret_cast<const float2*>(f + S * (j * LD + i));
          fr[u][j] = v.x;
          fi[u][j] = v.y;
        } else {
          fr[u][j] = f[S * (j * LD + i)];
          if constexpr (C) fi[u][j] = f[S * (j * LD + i) + 1];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const bool ok = p + G * u < p1;
      const int pu = ok ? p + G * u : p;
      const double* x = a.fw + S * (off + static_cast<int64_t>(a.src[pu]) * CD);
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        const double xr = ok ? x[S * j] : 0.0;
        const double xi = (C && ok) ? x[S * j + 1] : 0.0;
        const double er = static_cast<double>(fr[u][j]), ei = C ? static_cast<double>(fi[u][C ? j : 0]) : 0.0;
        if constexpr (C) {
          ar += er * xr - ei * xi;
          ai += er * xi + ei * xr;
        } else {
          ar += er * xr;
        }
      }
      double cr[1], ci[1];
      group_column_sums<W, 1>(
          li,
          [&](int j) {
            const int jj = j < CD ? j : 0;
            const double er = static_cast<double>(fr[u][jj]), ei = C ? static_cast<double>(fi[u][C ? jj : 0]) : 0.0;
            return j < CD ? (C ? er * tr - ei * ti : er * tr) : 0.0;
          },
          cr);
      if constexpr (C)
        group_column_sums<W, 1>(
            li,
            [&](int j) {
              const int jj = j < CD ? j : 0;
              return j < CD ? static_cast<double>(fr[u][jj]) * ti + static_cast<double>(fi[u][jj]) * tr : 0.0;
            },
            ci);
      const int sl = a.slot[pu];
      if (ok && act && sl >= 0) {  // a diagonal near-field leaf (slot -1) has no transposed product
        double* pp = a.part + S * (static_cast<int64_t>(sl) * CD + li);
        pp[0] = cr[0];
        if constexpr (C) pp[1] = ci[0];
      }
    }
  }
#pragma unroll
  for (int m = W; m < 64; m <<= 1) {
    ar += __shfl_xor(ar, m, 64);
    if constexpr (C) ai += __shfl_xor(ai, m, 64);
  }
  if (g == 0 && act) {
    double* y = a.bw + S * (off + static_cast<int64_t>(T.y) * CD + li);
    y[0] = ar;
    if constexpr (C) y[1] = ai;
  }
}

// Complex blocks from the lower side: for the loop's cluster c (its x_c in LDS, the same for every
// entry) each entry names a partner s > c and the stored block B = F(s, c) (rows of s, columns of
// c), the transpose of the upper block F(c, s).  The wave takes one block at a time: lane i of
// half h holds row i of the block's h-th column half.
//  * B x_c: a dot product inside the lane over its half, the two halves added across the wave,
//    is the entry's partial for the rows of s;
//  * B^T x_s = F(c, s) x_s adds B(i, j) x_s(i) into the lane's column accumulators (x_s(i) is one
//    coalesced load per lane), summed over the half's lanes once, after the loop, into y_c.
// The upper-block form needs a column sum over the lanes for every block; this form one per loop.
template <bool C, int CD, int UB, typename FT = double, int LD = CD>
__device__ __forceinline__ void coupling_wave_lsym(int t, const CplArgs& a) {
  static_assert(C, "complex blocks");
  static_assert(CD <= 32, "block rows exceed half a wave");
  constexpr int S = 2;
  constexpr int JH = (CD + 1) / 2;  // columns of the first half (the second has CD - JH)
  __shared__ double xl[4][S * CD];  // x_c of each wave of the workgroup
  const int lane = threadIdx.x & 63;
  const int wv = static_cast<int>(threadIdx.x >> 6);
  const int h = lane >> 5, li = lane & 31;
  const bool act = li < CD;
  const int i = act ? li : 0;
  const int j0 = h * JH;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  {
    const double* xc = a.fw + S * (off + static_cast<int64_t>(T.y) * CD);
    if (lane < S * CD) xl[wv][lane] = xc[lane];
  }
  __builtin_amdgcn_wave_barrier();
  double acr[JH], aci[JH];
#pragma unroll
  for (int jj = 0; jj < JH; ++jj) acr[jj] = 0.0, aci[jj] = 0.0;
  // block, partner and partial slot of 64 entries at a time, one per lane, read by the block
  // loop with lane reads (no dependent load before each block)
  for (int q0 = p0; q0 < p1; q0 += 64) {
    const bool lq = q0 + lane < p1;
    const int blkv = lq ? a.blk[q0 + lane] : 0;
    const int srcv = lq ? a.src[q0 + lane] : 0;
    const int slotv = lq ? a.slot[q0 + lane] : 0;
    const int q1 = p1 - q0 < 64 ? p1 : q0 + 64;
    for (int p = q0; p < q1; p += UB) {
      FT fr[UB][JH], fi[UB][JH];
      double sr[UB], si[UB];
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        const bool ok = p + u < q1;
        const int e = (ok ? p + u : p) - q0;
        const double2 xs = *reinterpret_cast<const double2*>(
            a.fw + S * (off + static_cast<int64_t>(__builtin_amdgcn_readlane(srcv, e)) * CD + i));
        sr[u] = ok && act ? xs.x : 0.0;  // idle lanes and spare entries add nothing to the columns
        si[u] = ok && act ? xs.y : 0.0;
        const FT* f = F + S * (static_cast<int64_t>(__builtin_amdgcn_readlane(blkv, e)) * a.fstride + a.fcomp);
#pragma unroll
        for (int jj = 0; jj < JH; ++jj) {
          // the second half is one column short when CD is odd: its last slot reads column j0
          // and counts as zero
          const bool has = jj < CD - JH || h == 0;
          const int j = has ? j0 + jj : j0;
          if constexpr (std::is_same<FT, float>::value) {
            const float2 v = *reinterpret_cast<const float2*>(f + S * (j * LD + i));
            fr[u][jj] = has ? v.x : 0.0f;
            fi[u][jj] = has ? v.y : 0.0f;
          } else {
            const double2 v = *reinterpret_cast<const double2*>(f + S * (j * LD + i));
            fr[u][jj] = has ? v.x : 0.0;
            fi[u][jj] = has ? v.y : 0.0;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < UB; ++u) {
        const bool ok = p + u < q1;
        const int e = (ok ? p + u : p) - q0;
        // x_c is read from LDS inside the loop (held in registers across it, it would take 2 * CD)
        int base = j0;
        asm volatile("" : "+v"(base));
        double dr = 0.0, di = 0.0;
#pragma unroll
        for (int jj = 0; jj < JH; ++jj) {
          const int jx = jj < CD - JH ? jj : (h == 0 ? jj : 0);
          const double2 xc = *reinterpret_cast<const double2*>(&xl[wv][S * (base + jx)]);
          const double er = static_cast<double>(fr[u][jj]), ei = static_cast<double>(fi[u][jj]);
          dr += er * xc.x - ei * xc.y;
          di += er * xc.y + ei * xc.x;
          acr[jj] += er * sr[u] - ei * si[u];
          aci[jj] += er * si[u] + ei * sr[u];
        }
        dr += __shfl_xor(dr, 32, 64);
        di += __shfl_xor(di, 32, 64);
        if (ok && act && h == 0) {
          double2* pp = reinterpret_cast<double2*>(
              a.part + S * (static_cast<int64_t>(__builtin_amdgcn_readlane(slotv, e)) * CD + li));
          *pp = make_double2(dr, di);
        }
      }
    }
  }
  // column sums over each half's lanes: lane li of half h ends with column j0 + li
  double cr[1], ci[1];
  group_column_sums<32, 1>(li, [&](int k) { return k < JH ? acr[k < JH ? k : 0] : 0.0; }, cr);
  group_column_sums<32, 1>(li, [&](int k) { return k < JH ? aci[k < JH ? k : 0] : 0.0; }, ci);
  if (li < (h ? CD - JH : JH)) {
    double2* y = reinterpret_cast<double2*>(a.bw + S * (off + static_cast<int64_t>(T.y) * CD + j0 + li));
    *y = make_double2(cr[0], ci[0]);
  }
}

// FP32 blocks with columns padded to whole 16-byte row vectors (LD rows): a group of W lanes
// (W = LD / RPL rounded up to a power of two; lanes past LD / RPL idle) owns a block
template <bool C, int CD, int LD, int UB>
__device__ __forceinline__ void coupling_wave_v_sym(int t, const CplArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int RPL = RowVec<C, float>::RPL;
  constexpr int H = LD / RPL;
  constexpr int W = pow2_at_least(H);
  constexpr int NG = 64 / W;
  constexpr int R = (CD + W - 1) / W;  // columns per lane after the column sums
  const int lane = threadIdx.x & 63;
  const int g = lane / W, l = lane % W;
  const bool act = l < H;
  const int lc = act ? l : 0;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const float* __restrict__ F = static_cast<const float*>(a.F);
  // x_t at this lane's rows
  double tr[RPL], ti[RPL];
  {
    const double* xt = a.fw + S * (off + static_cast<int64_t>(T.y) * CD);
#pragma unroll
    for (int q = 0; q < RPL; ++q) {
      const int row = RPL * l + q;
      const bool in = act && row < CD;
      tr[q] = in ? xt[S * (in ? row : 0)] : 0.0;
      ti[q] = (C && in) ? xt[S * (in ? row : 0) + 1] : 0.0;
    }
  }
  double yr[RPL], yi[C ? RPL : 1];
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    yr[q] = 0.0;
    if constexpr (C) yi[q] = 0.0;
  }
#pragma unroll 1
  for (int p = p0 + g; p < p1; p += NG * UB) {
    RowVec<C, float> fv[UB][CD];
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int pu = p + NG * u < p1 ? p + NG * u : p;
      const float* f = F + S * (static_cast<int64_t>(a.blk[pu]) * a.fstride + a.fcomp);
#pragma unroll
      for (int j = 0; j < CD; ++j) fv[u][j].load(f + S * (j * LD + RPL * lc));
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const bool ok = p + NG * u < p1;
      const int pu = ok ? p + NG * u : p;
      // F^T x_t first: this lane's rows of column j, summed over the group right away (xor
      // all-reduce: every lane ends with the same bits); lane j % W keeps column j. The partials
      // are stored before the row products (fewer registers held across the stores)
      double cr[R], ci[R];
#pragma unroll
      for (int r = 0; r < R; ++r) cr[r] = 0.0, ci[r] = 0.0;
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        double sr = 0.0, si = 0.0;
#pragma unroll
        for (int q = 0; q < RPL; ++q) {
          const double fr = static_cast<double>(fv[u][j].r[q]);
          if constexpr (C) {
            const double fi = static_cast<double>(fv[u][j].i[q]);
            sr += fr * tr[q] - fi * ti[q];
            si += fr * ti[q] + fi * tr[q];
          } else {
            sr += fr * tr[q];
          }
        }
#pragma unroll
        for (int m = W / 2; m >= 1; m >>= 1) {
          sr += __shfl_xor(sr, m, 64);
          if constexpr (C) si += __shfl_xor(si, m, 64);
        }
        if (l == j % W) {
          cr[j / W] = sr;
          if constexpr (C) ci[j / W] = si;
        }
      }
      if (ok) {
        double* pp = a.part + S * static_cast<int64_t>(a.slot[pu]) * CD;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int col = r * W + l;
          if (col < CD) {
            pp[S * col] = cr[r];
            if constexpr (C) pp[S * col + 1] = ci[r];
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      const double* x = a.fw + S * (off + static_cast<int64_t>(a.src[pu]) * CD);
      // row products in two column halves (half of the x values live at a time)
      constexpr int JH = (CD + 1) / 2;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (half) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = half * JH; j < (half ? CD : JH); ++j) {
          const double xr = ok ? x[S * j] : 0.0;
          const double xi = (C && ok) ? x[S * j + 1] : 0.0;
#pragma unroll
          for (int q = 0; q < RPL; ++q) {
            const double fr = static_cast<double>(fv[u][j].r[q]);
            if constexpr (C) {
              const double fi = static_cast<double>(fv[u][j].i[q]);
              yr[q] += fr * xr - fi * xi;
              yi[q] += fr * xi + fi * xr;
            } else {
              yr[q] += fr * xr;
            }
          }
        }
      }
    }
  }
  // the NG groups' row sums
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
#pragma unroll
    for (int m = W; m < 64; m <<= 1) {
      yr[q] += __shfl_xor(yr[q], m, 64);
      if constexpr (C) yi[q] += __shfl_xor(yi[q], m, 64);
    }
  }
  if (g == 0 && act) {
    double* y = a.bw + S * (off + static_cast<int64_t>(T.y) * CD);
#pragma unroll
    for (int q = 0; q < RPL; ++q) {
      const int row = RPL * l + q;
      if (row >= CD) continue;
      y[S * row] = yr[q];
      if constexpr (C) y[S * row + 1] = yi[q];
    }
  }
}

// real FP64 blocks, two rows per lane
template <int CD, int UB>
__device__ __forceinline__ void coupling_wave_r2_sym(int t, const CplArgs& a) {
  constexpr int H = CD / 2;
  constexpr int NG = 64 / H;  // H is a power of two here
  const int lane = threadIdx.x & 63;
  const int g = lane / H, l = lane % H;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const double* __restrict__ F = static_cast<const double*>(a.F);
  const double* xt = a.fw + off + static_cast<int64_t>(T.y) * CD + 2 * l;
  const double t0 = xt[0], t1 = xt[1];
  double y0 = 0.0, y1 = 0.0;
  for (int p = p0 + g; p < p1; p += NG * UB) {
    double2 fv[UB][CD];
    double xv[UB][CD];
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const bool ok = p + NG * u < p1;
      const int pu = ok ? p + NG * u : p;
      const double* f = F + static_cast<int64_t>(a.blk[pu]) * a.fstride + a.fcomp;
      const double* x = a.fw + off + static_cast<int64_t>(a.src[pu]) * CD;
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        fv[u][j] = *reinterpret_cast<const double2*>(f + j * CD + 2 * l);
        xv[u][j] = ok ? x[j] : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < UB; ++u) {
#pragma unroll
      for (int j = 0; j < CD; ++j) {
        y0 += fv[u][j].x * xv[u][j];
        y1 += fv[u][j].y * xv[u][j];
      }
      const bool ok = p + NG * u < p1;
      const int pu = ok ? p + NG * u : p;
      double c[2];
      group_column_sums<H, 2>(l, [&](int j) { return fv[u][j].x * t0 + fv[u][j].y * t1; }, c);
      if (ok) {
        double* pp = a.part + static_cast<int64_t>(a.slot[pu]) * CD + 2 * l;
        pp[0] = c[0];
        pp[1] = c[1];
      }
    }
  }
#pragma unroll
  for (int m = H; m < 64; m <<= 1) {
    y0 += __shfl_xor(y0, m, 64);
    y1 += __shfl_xor(y1, m, 64);
  }
  if (g == 0) {
    double* y = a.bw + off + static_cast<int64_t>(T.y) * CD + 2 * l;
    y[0] = y0;
    y[1] = y1;
  }
}

// bw[s] += the partials of the upper blocks (t, s), stored contiguously in gather order: one
// thread per (target, entry of its S*CD doubles), independent loads, added in list order
template <bool C, int CD>
__global__ __launch_bounds__(256) void k_sym_gather(int ng, const int2* __restrict__ gtgt, const int* __restrict__ grp,
                                                    const double* __restrict__ part,
                                                    const int64_t* __restrict__ lvl_off, double* bw) {
  constexpr int S = C ? 2 : 1;
  constexpr int E = S * CD;  // doubles per target (even: read as 16-byte pairs)
  static_assert(E % 2 == 0, "pairs of doubles");
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(ng) * (E / 2)) return;
  const int w = static_cast<int>(gid / (E / 2)), e = 2 * static_cast<int>(gid - static_cast<int64_t>(w) * (E / 2));
  const int2 T = gtgt[w];
  double2* y = reinterpret_cast<double2*>(bw + S * (lvl_off[T.x] + static_cast<int64_t>(T.y) * CD) + e);
  const int q0 = grp[w], q1 = grp[w + 1];
  const double* pp = part + static_cast<int64_t>(q0) * E + e;
  // eight 16-byte loads in flight, then added in slot order (a target receives 16 partials on
  // average)
  double2 s = *y;
  int q = 0;
  for (; q + 8 <= q1 - q0; q += 8) {
    double2 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const double2*>(pp + static_cast<int64_t>(q + u) * E);
#pragma unroll
    for (int u = 0; u < 8; ++u) s.x += v[u].x, s.y += v[u].y;
  }
  for (; q < q1 - q0; ++q) {
    const double2 v = *reinterpret_cast<const double2*>(pp + static_cast<int64_t>(q) * E);
    s.x += v.x, s.y += v.y;
  }
  *y = s;
}

// the two sweeps of a single-RHS product in one launch: workgroups [0, nb_near) run the near
// field, the rest the coupling blocks, so both streams of leaves share the memory system
template <bool C, int DD, typename FT, int CD, int UBN, int UBC, typename NFT, bool SYM, bool NSYM>
__device__ __forceinline__ void sweep_fused_body(const LeafArgs& la, const CplArgs& ca, int nb_near,
                                                 const CplArgs& na) {
  const int b = static_cast<int>(blockIdx.x);
  const int w = static_cast<int>(threadIdx.x >> 6);
  // real FP64 blocks: two rows per lane (16-byte loads)
  // near-field rows of 16-byte vectors: real FP64 (2 rows per lane), FP32 (4 real, 2 complex)
  constexpr bool R2N = (!C || std::is_same<NFT, float>::value) && DD % RowVec<C, NFT>::RPL == 0;
  constexpr bool R2C = !C && std::is_same<FT, double>::value && (CD == 16 || CD == 32);
  // FP32 coupling copies are stored with columns padded to LDV rows (see the FP32 conversion)
  constexpr int RPLC = RowVec<C, float>::RPL;
  constexpr int LDV = (CD + RPLC - 1) / RPLC * RPLC;
  constexpr bool VC = std::is_same<FT, float>::value;
  if (b < nb_near) {
    const int c = __builtin_amdgcn_readfirstlane(b * 4 + w);
    if (c < la.ncl) {
      if constexpr (SYM && NSYM && std::is_same<NFT, double>::value) {
        // upper and diagonal near-field leaves with transposed partials
        if (na.rp) {
          coupling_wave_sym<C, DD, UBN>(c, na);
          return;
        }
      }
      if constexpr (R2N)
        leaf_wave_v<C, NFT, DD, UBN>(c, la);
      else
        leaf_wave<C, DD, UBN, NFT>(c, la);
    }
  } else {
    const int t = __builtin_amdgcn_readfirstlane((b - nb_near) * 4 + w);
    if (t < ca.ntgt) {
      if constexpr (SYM) {
        // one block per pair (the launcher checks the padded FP32 layout): the upper blocks of
        // real kernels, the lower ones of complex kernels
        if constexpr (R2C)
          coupling_wave_r2_sym<CD, UBC>(t, ca);
        else if constexpr (VC && C)
          coupling_wave_lsym<C, CD, UBC, float, LDV>(t, ca);
        else if constexpr (VC)
          coupling_wave_v_sym<C, CD, LDV, UBC>(t, ca);
        else if constexpr (C)
          coupling_wave_lsym<C, CD, UBC>(t, ca);
        else
          coupling_wave_sym<C, CD, UBC>(t, ca);
      } else if constexpr (R2C)
        coupling_wave_r2<CD, UBC>(t, ca);
      else if constexpr (VC) {
        if (ca.ld == LDV && ca.Fc == nullptr) {
          coupling_wave_v<C, CD, LDV, UBC>(t, ca);
        } else {
          coupling_wave<C, FT, CD, 1, UBC>(t, ca);
        }
      } else {
        coupling_wave<C, FT, CD, 1, UBC>(t, ca);
      }
    }
  }
}

// every block of both sweeps (SYM false), or the upper coupling blocks with transposed partials
// (SYM true; NSYM: the upper near-field leaves as well, a separate instantiation because its
// registers would otherwise bound the occupancy of the coupling-only form)
template <bool C, int DD, typename FT, int CD, int UBN, int UBC, typename NFT = double>
__global__ __launch_bounds__(256) void k_sweep_fused(LeafArgs la, CplArgs ca, int nb_near, CplArgs na) {
  sweep_fused_body<C, DD, FT, CD, UBN, UBC, NFT, false, false>(la, ca, nb_near, na);
}

template <bool C, int DD, typename FT, int CD, int UBN, int UBC, typename NFT, bool NSYM>
__global__ __launch_bounds__(256) void k_sweep_fused_sym(LeafArgs la, CplArgs ca, int nb_near, CplArgs na) {
  sweep_fused_body<C, DD, FT, CD, UBN, UBC, NFT, true, NSYM>(la, ca, nb_near, na);
}

// ------------------------------------------------------------------ many right-hand sides
// Block rows of row owners (leaf clusters or coupling targets), 64 columns per workgroup.
// Addresses: X(s, j, k) = x[S * (xoff + s * xcs + k * xks + j)], Y(r, i, k) likewise with the
// owner's cluster; coupling owners shift both by their level's start.
struct MultiArgs {
  int nown, nrhs;
  const int2* tgt;  // coupling: (level, cluster) of each owner; near field: null (owner = cluster)
  const int64_t* lvl_off;
  const int* rp;
  const int* src;
  const void* F;
  int64_t fstride, fcomp;
  int ldf;  // column stride of the blocks
  const double* x;
  int64_t xoff, xcs, xks, xrs;  // offset, cluster, column (RHS) and row strides of x
  double* y;
  int64_t yoff, ycs, yks, yrs;
  int accumulate;
  // block list of owner r: 0 = CSR (rp, src; block p); implicit lists of the tree steps:
  // 1 = blocks 4r..4r+3 on sources 4r..4r+3, block index p % 4 (children to parent);
  // 2 = one block on source r / 4, block index r % 4 (parent to child);
  // 3 = one block on source r, block index 0 (leaf moments and leaf rows)
  int mode;
};

// ------------------------------------------------------------------ block rows staged in LDS (many RHS)
// One workgroup (4 waves) per owner and 64 right-hand sides: y_owner (ROUT x 64) = sum over the
// owner's blocks of F_p (ROUT x RIN) x_src(p) (RIN x 64). Each block and the x tile it multiplies
// are copied to LDS with coalesced 8-byte loads by all 256 threads; the next block's copy is in
// flight (registers) while the current one is multiplied. Wave w owns output rows
// [w*RPW, w*RPW + RPW); its lanes are the 64 right-hand sides, reading the x tile row by row
// (consecutive lanes, consecutive LDS words) and the block entries as LDS broadcasts. Sums in
// FP64 whatever the block type. XC: complex vectors; FC: complex blocks (real blocks with
// complex vectors are the tree steps of an oscillatory kernel).
template <bool XC, bool FC, typename FT, int ROUT, int RIN>
__global__ __launch_bounds__(256) void k_multi_lds(MultiArgs a) {
  static_assert(XC || !FC, "complex blocks need complex vectors");
  constexpr int SX = XC ? 2 : 1, SF = FC ? 2 : 1;
  constexpr int RPW = (ROUT + 3) / 4;
  constexpr int LDMAX = (ROUT + 3) / 4 * 4;
  constexpr int FU_MAX = SF * LDMAX * RIN;  // 8-byte units of the largest (FP64) block
  constexpr int XU = RIN * 64 * SX;         // 8-byte units of an x tile
  constexpr int NFU = (FU_MAX + 255) / 256, NXU = (XU + 255) / 256;
  __shared__ uint2 Fs[FU_MAX];
  __shared__ double Xs[XU];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int r = blockIdx.x;
  const int k0 = static_cast<int>(blockIdx.y) * 64;
  const int kmax = a.nrhs - 1 - k0;  // last valid lane of this tile
  int cl = r;
  int64_t xo = a.xoff, yo = a.yoff;
  if (a.tgt) {
    const int2 T = a.tgt[r];
    cl = T.y;
    const int64_t lo = a.lvl_off[T.x] * a.nrhs;
    xo += lo;
    yo += lo;
  }
  const int mode = a.mode;
  int p0, p1;
  if (mode == 0) {
    p0 = a.rp[r];
    p1 = a.rp[r + 1];
  } else if (mode == 1) {
    p0 = 4 * r;
    p1 = p0 + 4;
  } else {
    p0 = r;
    p1 = r + 1;
  }
  const int fu = static_cast<int>((static_cast<int64_t>(SF) * a.ldf * RIN * sizeof(FT)) / 8);
  const uint2* __restrict__ F8 = static_cast<const uint2*>(a.F);
  const int64_t fblk = static_cast<int64_t>(SF) * a.fstride * sizeof(FT) / 8;  // 8-byte units per block index
  const int64_t fc8 = static_cast<int64_t>(SF) * a.fcomp * sizeof(FT) / 8;
  uint2 pf[NFU];
  double px[NXU];
  auto fetch = [&](int p) {
    const int bi = mode == 0 ? p : (mode == 3 ? 0 : (p & 3));
    const int sc = mode == 0 ? a.src[p] : (mode == 2 ? (p >> 2) : p);
    const uint2* f = F8 + static_cast<int64_t>(bi) * fblk + fc8;
#pragma unroll
    for (int q = 0; q < NFU; ++q) {
      const int u = tid + 256 * q;
      if (u < fu) pf[q] = f[u];
    }
    const double* x = a.x + SX * (xo + static_cast<int64_t>(sc) * a.xcs);
#pragma unroll
    for (int q = 0; q < NXU; ++q) {
      const int u = tid + 256 * q;
      if (XU % 256 == 0 || u < XU) {
        const int j = u / (64 * SX), rem = u - j * (64 * SX);
        int kl = rem / SX;
        kl = kl <= kmax ? kl : kmax;
        px[q] = x[SX * (static_cast<int64_t>(j) * a.xrs + static_cast<int64_t>(k0 + kl) * a.xks) + (rem % SX)];
      }
    }
  };
  auto commit = [&]() {
#pragma unroll
    for (int q = 0; q < NFU; ++q) {
      const int u = tid + 256 * q;
      if (u < fu) Fs[u] = pf[q];
    }
#pragma unroll
    for (int q = 0; q < NXU; ++q) {
      const int u = tid + 256 * q;
      if (XU % 256 == 0 || u < XU) Xs[u] = px[q];
    }
  };
  double ar[RPW], ai[XC ? RPW : 1];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    ar[i] = 0.0;
    if constexpr (XC) ai[i] = 0.0;
  }
  const int i0 = w * RPW;
  const FT* Fl = reinterpret_cast<const FT*>(Fs);
  if (p0 < p1) fetch(p0);
  for (int p = p0; p < p1; ++p) {
    __syncthreads();  // the previous block is no longer read
    commit();
    __syncthreads();
    if (p + 1 < p1) fetch(p + 1);
#pragma unroll 2
    for (int j = 0; j < RIN; ++j) {
      const double xr = Xs[SX * (j * 64 + lane)];
      const double xi = XC ? Xs[SX * (j * 64 + lane) + 1] : 0.0;
      const FT* fj = Fl + SF * (j * a.ldf);
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const int ii = (ROUT % 4 == 0 || i0 + i < ROUT) ? i0 + i : ROUT - 1;
        const double fr = static_cast<double>(fj[SF * ii]);
        if constexpr (FC) {
          const double fi = static_cast<double>(fj[SF * ii + 1]);
          ar[i] += fr * xr - fi * xi;
          ai[i] += fr * xi + fi * xr;
        } else if constexpr (XC) {
          ar[i] += fr * xr;
          ai[i] += fr * xi;
        } else {
          ar[i] += fr * xr;
        }
      }
    }
  }
  if (lane > kmax) return;
  double* y = a.y + SX * (yo + static_cast<int64_t>(cl) * a.ycs + static_cast<int64_t>(k0 + lane) * a.yks);
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (ROUT % 4 != 0 && i0 + i >= ROUT) continue;
    double* yi_ = y + SX * static_cast<int64_t>(i0 + i) * a.yrs;
    double vr = ar[i], vi = XC ? ai[i] : 0.0;
    if (a.accumulate) {
      vr += yi_[0];
      if constexpr (XC) vi += yi_[1];
    }
    yi_[0] = vr;
    if constexpr (XC) yi_[1] = vi;
  }
}

// ------------------------------------------------------------------ block rows on the matrix cores (many RHS)
// Same product as k_multi_lds, on FP64 MFMA (v_mfma_f64_16x16x4f64): y_owner (ROUT x 64) = sum over
// the owner's blocks of F_p (ROUT x RIN) x_src(p) (RIN x 64); wave w computes the 16 right-hand
// sides [16w, 16w + 16) for all row tiles. Operand layout of the instruction: A(i, k) on lane
// i + 16k, B(k, j) on lane j + 16k, D(i, j) on lane j + 16 (i % 4), element i / 4.
// The block (widened to FP64) is staged in LDS as planes of real and of imaginary parts, zero-padded
// to whole 16-row tiles and 4-column steps, so that the 16 lanes of a row tile read 16 consecutive
// doubles. Complex blocks times complex vectors are three real products (Gauss: Fr Xr, Fi Xi and
// (Fr + Fi)(Xr + Xi)), real blocks times complex vectors two. Complex blocks with 4 rows past the
// last full tile (36 = 2 x 16 + 4) compute those rows in one more tile, real parts in its rows 0-3
// and imaginary parts in rows 4-7, as [Fr, -Fi; Fi, Fr] [Xr; Xi] (two products per column step).
// Two forms:
// * XL = false (tree steps): the x tile is staged in LDS like the block, one block at a time,
//   one workgroup per owner;
// * XL = true (block sweeps): x is not shared between waves (each wave multiplies its own 16
//   columns), so every lane loads its operands itself; the blocks alternate between two LDS
//   buffers (one barrier per block), and each workgroup runs over several owners, the next
//   owner's first block fetched during the last block of the current one.
// Owners go to XCDs in contiguous ranges (workgroups are handed to the 8 XCDs in turn): neighbouring
// owners share most of their source clusters, and each XCD has its own L2.
typedef double bmi_d4 __attribute__((ext_vector_type(4)));

// the owner range [start, start + cnt) of XCD k for nown owners
__device__ __forceinline__ void xcd_range(int k, int nown, int& start, int& cnt) {
  const int q = nown >> 3, rem = nown & 7;
  start = k * q + (k < rem ? k : rem);
  cnt = q + (k < rem ? 1 : 0);
}

template <bool XC, bool FC, typename FT, int ROUT, int RIN, bool XL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_multi_mfma(MultiArgs a) {
  static_assert(XC || !FC, "complex blocks need complex vectors");
  constexpr int SX = XC ? 2 : 1, SF = FC ? 2 : 1;
  constexpr int MT = (ROUT + 15) / 16, KS = (RIN + 3) / 4;
  constexpr int NP = MT == 1 ? 2 : 1;  // independent accumulator chains per tile
  constexpr bool TAIL = FC && MT >= 2 && ROUT % 16 == 4;
  constexpr int MTF = TAIL ? MT - 1 : MT;  // tiles of the three-product form
  constexpr int FLD = MT * 16;             // LDS column stride of a plane
  constexpr int PL = KS * 4 * FLD;         // doubles per plane
  constexpr int LDMAX = (ROUT + 3) / 4 * 4;
  constexpr int NFE = (LDMAX * RIN + 255) / 256;  // block elements per thread (bound)
  constexpr int NBUF = XL ? 2 : 1;
  constexpr int XPL = XL ? 0 : KS * 4 * 64;       // doubles per x plane (staged x)
  constexpr int NXE = (RIN * 64 + 255) / 256;     // staged x elements per thread
  __shared__ double Fs[NBUF * SF * PL + SX * XPL];
  double* Xs = Fs + NBUF * SF * PL;
  // LDS positions: entry (column c, row i) of a block plane and (row j, column k) of an x plane.
  // Odd columns (rows) swap their halves of 16 doubles where the stride is an even multiple of
  // 16, so the two lane quarters of a half-wave (consecutive columns) fall on different banks.
  auto fpos = [](int c, int i) { return c * FLD + (MT % 2 == 0 ? (i ^ ((c & 1) << 4)) : i); };
  auto xpos = [](int j, int k) { return j * 64 + (k ^ ((j & 1) << 4)); };
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int n = w * 16 + li;  // this lane's column of the x tile
  const int k0 = static_cast<int>(blockIdx.y) * 64;
  const int kmax = a.nrhs - 1 - k0;
  const int kc = n <= kmax ? n : kmax;  // columns past the last right-hand side repeat it
  const int mode = a.mode;
  struct Own {
    int cl, p0, p1;
    int64_t xo, yo;
  };
  auto owner = [&](int r) {
    Own o;
    o.cl = r;
    o.xo = a.xoff;
    o.yo = a.yoff;
    if (a.tgt) {
      const int2 T = a.tgt[r];
      o.cl = T.y;
      const int64_t lo = a.lvl_off[T.x] * a.nrhs;
      o.xo += lo;
      o.yo += lo;
    }
    if (mode == 0) {
      o.p0 = a.rp[r];
      o.p1 = a.rp[r + 1];
    } else if (mode == 1) {
      o.p0 = 4 * r;
      o.p1 = o.p0 + 4;
    } else {
      o.p0 = r;
      o.p1 = r + 1;
    }
    return o;
  };
  auto source = [&](int p) { return mode == 0 ? a.src[p] : (mode == 2 ? (p >> 2) : p); };
  // zero padding: rows [ROUT, RREAD) of every column and columns [RIN, KS * 4) of the block rows
  // (and x rows [RIN, KS * 4) when x is staged); the copies below write inside only
  {
    constexpr int RREAD = TAIL ? ROUT : MT * 16;
    constexpr int PR = RREAD > ROUT ? RREAD - ROUT : 1;
    constexpr int NZR = KS * 4 * (RREAD - ROUT), NZ = NZR + (KS * 4 - RIN) * ROUT;
    for (int u = tid; u < NBUF * SF * NZ; u += 256) {
      const int pl = u / NZ, v = u - pl * NZ;
      int c, i;
      if (v < NZR) {
        c = v / PR;
        i = ROUT + (v - c * PR);
      } else {
        c = RIN + (v - NZR) / ROUT;
        i = (v - NZR) - (c - RIN) * ROUT;
      }
      Fs[pl * PL + fpos(c, i)] = 0.0;
    }
    if constexpr (!XL) {
      constexpr int NZX = (KS * 4 - RIN) * 64;
      for (int u = tid; u < SX * NZX; u += 256) {
        const int pl = u / NZX, v = u - pl * NZX;
        Xs[pl * XPL + xpos(RIN + (v >> 6), v & 63)] = 0.0;
      }
    }
  }
  const int ldf = a.ldf;
  const int fe = ldf * RIN;
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  FT pfr[NFE], pfi[FC ? NFE : 1];
  double pxr[XL ? 1 : NXE], pxi[XC && !XL ? NXE : 1];  // staged x: the thread's share of the tile
  double xr[XL ? KS : 1], xi[XC && XL ? KS : 1];      // lane-loaded x: (row 4 ks + lk, column n)
  // block p into registers (and, staged x, its x tile)
  auto fetch = [&](const Own& o, int p) {
    const int bi = mode == 0 ? p : (mode == 3 ? 0 : (p & 3));
    const FT* f = F + SF * (static_cast<int64_t>(bi) * a.fstride + a.fcomp);
#pragma unroll
    for (int q = 0; q < NFE; ++q) {
      const int e = tid + 256 * q;
      if (e < fe) {
        pfr[q] = f[SF * e];
        if constexpr (FC) pfi[q] = f[SF * e + 1];
      }
    }
    if constexpr (!XL) {
      const double* x = a.x + SX * (o.xo + static_cast<int64_t>(source(p)) * a.xcs);
#pragma unroll
      for (int q = 0; q < NXE; ++q) {
        const int e = tid + 256 * q;
        if ((RIN * 64) % 256 == 0 || e < RIN * 64) {
          const int j = e >> 6;
          int kl = e & 63;
          kl = kl <= kmax ? kl : kmax;
          const double* xe = x + SX * (static_cast<int64_t>(j) * a.xrs + static_cast<int64_t>(k0 + kl) * a.xks);
          pxr[q] = xe[0];
          if constexpr (XC) pxi[q] = xe[1];
        }
      }
    }
  };
  // the lane's x operands of block p (lane-loaded x)
  auto load_x = [&](const Own& o, int p) {
    const double* x = a.x + SX * (o.xo + static_cast<int64_t>(source(p)) * a.xcs + static_cast<int64_t>(k0 + kc) * a.xks);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kr = ks * 4 + lk;
      if (RIN % 4 == 0 || kr < RIN) {
        const double* xe = x + SX * static_cast<int64_t>(kr) * a.xrs;
        xr[ks] = xe[0];
        if constexpr (XC) xi[ks] = xe[1];
      } else {
        xr[ks] = 0.0;
        if constexpr (XC) xi[ks] = 0.0;
      }
    }
  };
  auto commit = [&](int buf) {
    double* Fb = Fs + buf * (SF * PL);
#pragma unroll
    for (int q = 0; q < NFE; ++q) {
      const int e = tid + 256 * q;
      if (e < fe) {
        const int c = e / ldf, i = e - c * ldf;
        if (i < ROUT) {
          Fb[fpos(c, i)] = static_cast<double>(pfr[q]);
          if constexpr (FC) Fb[PL + fpos(c, i)] = static_cast<double>(pfi[q]);
        }
      }
    }
    if constexpr (!XL) {
#pragma unroll
      for (int q = 0; q < NXE; ++q) {
        const int e = tid + 256 * q;
        if ((RIN * 64) % 256 == 0 || e < RIN * 64) {
          const int j = e >> 6, kl = e & 63;
          Xs[xpos(j, kl)] = pxr[q];
          if constexpr (XC) Xs[XPL + xpos(j, kl)] = pxi[q];
        }
      }
    }
  };
  // complex blocks: P1 = Fr Xr (accr), P2 = Fi Xi (accq), P3 = (Fr + Fi)(Xr + Xi) (acci);
  // Re = P1 - P2, Im = P3 - P1 - P2; the tail tile accumulates in accr[MT - 1]
  bmi_d4 accr[MT][NP], acci[XC ? MT : 1][NP], accq[FC ? MT : 1][NP];
  auto reset = [&]() {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int h = 0; h < NP; ++h) {
        accr[m][h] = bmi_d4{0.0, 0.0, 0.0, 0.0};
        if constexpr (XC) acci[m][h] = bmi_d4{0.0, 0.0, 0.0, 0.0};
        if constexpr (FC) accq[m][h] = bmi_d4{0.0, 0.0, 0.0, 0.0};
      }
  };
  // the products of one staged block (planes at Fb)
  auto multiply = [&](const double* Fb) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kr = ks * 4 + lk;
      const int h = NP == 2 ? (ks & 1) : 0;
      const double br = XL ? xr[XL ? ks : 0] : Xs[xpos(kr, n)];
      const double bi = XC ? (XL ? xi[XL ? ks : 0] : Xs[XPL + xpos(kr, n)]) : 0.0;
      const double bs = br + bi;
      if constexpr (TAIL) {
        const int tr = MTF * 16 + (li & 3);
        const double tfr = Fb[fpos(kr, tr)], tfi = Fb[PL + fpos(kr, tr)];
        const double a1 = li < 4 ? tfr : (li < 8 ? tfi : 0.0);
        const double a2 = li < 4 ? -tfi : (li < 8 ? tfr : 0.0);
        accr[MT - 1][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, br, accr[MT - 1][h], 0, 0, 0);
        accr[MT - 1][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a2, bi, accr[MT - 1][h], 0, 0, 0);
      }
#pragma unroll
      for (int m = 0; m < MTF; ++m) {
        const double fr = Fb[fpos(kr, m * 16 + li)];
        if constexpr (FC) {
          const double fi = Fb[PL + fpos(kr, m * 16 + li)];
          accr[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr, br, accr[m][h], 0, 0, 0);
          accq[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fi, bi, accq[m][h], 0, 0, 0);
          acci[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr + fi, bs, acci[m][h], 0, 0, 0);
        } else if constexpr (XC) {
          accr[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr, br, accr[m][h], 0, 0, 0);
          acci[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr, bi, acci[m][h], 0, 0, 0);
        } else {
          accr[m][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr, br, accr[m][h], 0, 0, 0);
        }
      }
    }
  };
  // the owner's rows from the accumulators (zero: rows of an owner without blocks)
  auto write_rows = [&](const Own& o, bool zero) {
    if (n > kmax) return;
    if (zero && a.accumulate) return;
    double* y = a.y + SX * (o.yo + static_cast<int64_t>(o.cl) * a.ycs + static_cast<int64_t>(k0 + n) * a.yks);
    auto put = [&](int row, double vr, double vi) {
      double* yr = y + SX * static_cast<int64_t>(row) * a.yrs;
      if (zero) vr = vi = 0.0;
      if (a.accumulate) {
        vr += yr[0];
        if constexpr (XC) vi += yr[1];
      }
      yr[0] = vr;
      if constexpr (XC) yr[1] = vi;
    };
    if constexpr (TAIL) put(MTF * 16 + lk, accr[MT - 1][0][0], accr[MT - 1][0][1]);
#pragma unroll
    for (int m = 0; m < MTF; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = m * 16 + 4 * v + lk;
        if (ROUT % 16 != 0 && row >= ROUT) continue;
        double vr = accr[m][0][v], vi = 0.0;
        if constexpr (NP == 2) vr += accr[m][1][v];
        if constexpr (XC) {
          vi = acci[m][0][v];
          if constexpr (NP == 2) vi += acci[m][1][v];
        }
        if constexpr (FC) {
          double q = accq[m][0][v];
          if constexpr (NP == 2) q += accq[m][1][v];
          vi -= vr + q;  // P3 - (P1 + P2)
          vr -= q;       // P1 - P2
        }
        put(row, vr, vi);
      }
  };
  reset();
  if constexpr (!XL) {
    const Own o = owner(static_cast<int>(blockIdx.x));
    if (o.p0 < o.p1) fetch(o, o.p0);
    for (int p = o.p0; p < o.p1; ++p) {
      __syncthreads();  // previous block no longer read (first pass: zero fill done)
      commit(0);
      __syncthreads();
      if (p + 1 < o.p1) fetch(o, p + 1);
      multiply(Fs);
    }
    write_rows(o, false);
  } else {
    // this workgroup's owners: start + slot, start + slot + S, ... of its XCD's range
    int start, cnt;
    xcd_range(static_cast<int>(blockIdx.x & 7), a.nown, start, cnt);
    const int slot = static_cast<int>(blockIdx.x >> 3), S = static_cast<int>(gridDim.x >> 3);
    // the first owner with blocks from index t on; owners without blocks get their rows here
    auto advance = [&](int t, Own& o) {
      for (; t < cnt; t += S) {
        o = owner(start + t);
        if (o.p0 < o.p1) break;
        write_rows(o, true);
      }
      return t;
    };
    Own cur;
    int oi = advance(slot, cur);
    if (oi >= cnt) return;
    int p = cur.p0;
    fetch(cur, p);
    __syncthreads();  // zero fill done
    commit(0);
    load_x(cur, p);
    __syncthreads();
    int buf = 0;
    while (true) {
      // the next block: the owner's next, or the first of this workgroup's next owner
      Own nx = cur;
      int pn = p + 1, on = oi;
      if (pn >= cur.p1) {
        on = advance(oi + S, nx);
        pn = nx.p0;
      }
      const bool more = on < cnt;
      if (more) fetch(nx, pn);
      multiply(Fs + buf * (SF * PL));
      if (on != oi || !more) {
        write_rows(cur, false);
        reset();
      }
      if (!more) break;
      // the other buffer was last read before the previous barrier
      commit(1 - buf);
      load_x(nx, pn);
      __syncthreads();
      buf ^= 1;
      cur = nx;
      p = pn;
      oi = on;
    }
  }
}

// FP32 blocks of a reduced operator on the FP32 matrix cores (v_mfma_f32_16x16x4f32, twice the
// FP64 rate): the block and its x tile (rounded to FP32) are staged in LDS; each block's product
// is accumulated in FP32 from zero and then added to FP64 sums, so only the rows x columns of one
// block (at most RIN terms) are summed in FP32 and the sum over the owner's blocks is FP64.
// Operand layout: A(i, k) on lane i + 16k, B(k, j) on lane j + 16k, D(i, j) on lane
// j + 16 (i / 4), element i % 4 (checked on the device).
typedef float bmi_f4 __attribute__((ext_vector_type(4)));

template <bool C, int ROUT, int RIN>
__global__ __launch_bounds__(256) void k_multi_mfma32(MultiArgs a) {
  constexpr int S = C ? 2 : 1;
  constexpr int MT = (ROUT + 15) / 16, KS = (RIN + 3) / 4;
  constexpr int FLD = MT * 16;
  constexpr int LDMAX = (ROUT + 3) / 4 * 4;
  constexpr int NFE = (LDMAX * RIN + 255) / 256;
  constexpr int NXE = (RIN * 64 + 255) / 256;
  __shared__ float Fs[S * KS * 4 * FLD];
  __shared__ float Xs[S * KS * 4 * 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int r = blockIdx.x;
  const int k0 = static_cast<int>(blockIdx.y) * 64;
  const int kmax = a.nrhs - 1 - k0;
  int cl = r;
  int64_t xo = a.xoff, yo = a.yoff;
  if (a.tgt) {
    const int2 T = a.tgt[r];
    cl = T.y;
    const int64_t lo = a.lvl_off[T.x] * a.nrhs;
    xo += lo;
    yo += lo;
  }
  const int p0 = a.rp[r], p1 = a.rp[r + 1];
  for (int u = tid; u < S * KS * 4 * FLD; u += 256) Fs[u] = 0.0f;
  for (int u = tid; u < S * KS * 4 * 64; u += 256) Xs[u] = 0.0f;
  const int ldf = a.ldf;
  const int fe = ldf * RIN;
  const float* __restrict__ F = static_cast<const float*>(a.F);
  float pfr[NFE], pfi[C ? NFE : 1];
  float pxr[NXE], pxi[C ? NXE : 1];
  auto fetch = [&](int p) {
    const float* f = F + S * (static_cast<int64_t>(p) * a.fstride + a.fcomp);
#pragma unroll
    for (int q = 0; q < NFE; ++q) {
      const int e = tid + 256 * q;
      if (e < fe) {
        pfr[q] = f[S * e];
        if constexpr (C) pfi[q] = f[S * e + 1];
      }
    }
    const double* x = a.x + S * (xo + static_cast<int64_t>(a.src[p]) * a.xcs);
#pragma unroll
    for (int q = 0; q < NXE; ++q) {
      const int e = tid + 256 * q;
      if ((RIN * 64) % 256 == 0 || e < RIN * 64) {
        const int j = e >> 6;
        int kl = e & 63;
        kl = kl <= kmax ? kl : kmax;
        const double* xe = x + S * (static_cast<int64_t>(j) * a.xrs + static_cast<int64_t>(k0 + kl) * a.xks);
        pxr[q] = static_cast<float>(xe[0]);
        if constexpr (C) pxi[q] = static_cast<float>(xe[1]);
      }
    }
  };
  auto commit = [&]() {
#pragma unroll
    for (int q = 0; q < NFE; ++q) {
      const int e = tid + 256 * q;
      if (e < fe) {
        const int c = e / ldf, i = e - c * ldf;
        if (i < ROUT) {
          Fs[S * (c * FLD + i)] = pfr[q];
          if constexpr (C) Fs[S * (c * FLD + i) + 1] = pfi[q];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < NXE; ++q) {
      const int e = tid + 256 * q;
      if ((RIN * 64) % 256 == 0 || e < RIN * 64) {
        Xs[S * e] = pxr[q];
        if constexpr (C) Xs[S * e + 1] = pxi[q];
      }
    }
  };
  double sr[MT][4], si[C ? MT : 1][4];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      sr[m][v] = 0.0;
      if constexpr (C) si[m][v] = 0.0;
    }
  const int li = lane & 15, lk = lane >> 4;
  const int n = w * 16 + li;
  const bmi_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  if (p0 < p1) fetch(p0);
  for (int p = p0; p < p1; ++p) {
    __syncthreads();
    commit();
    __syncthreads();
    if (p + 1 < p1) fetch(p + 1);
    bmi_f4 ar[MT], ai[C ? MT : 1];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      ar[m] = zero;
      if constexpr (C) ai[m] = zero;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kr = ks * 4 + lk;
      const float br = Xs[S * (kr * 64 + n)];
      const float bi = C ? Xs[S * (kr * 64 + n) + 1] : 0.0f;
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float fr = Fs[S * (kr * FLD + m * 16 + li)];
        if constexpr (C) {
          const float fi = Fs[S * (kr * FLD + m * 16 + li) + 1];
          ar[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(fr, br, ar[m], 0, 0, 0);
          ai[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(fr, bi, ai[m], 0, 0, 0);
          ar[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(-fi, bi, ar[m], 0, 0, 0);
          ai[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(fi, br, ai[m], 0, 0, 0);
        } else {
          ar[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(fr, br, ar[m], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        sr[m][v] += static_cast<double>(ar[m][v]);
        if constexpr (C) si[m][v] += static_cast<double>(ai[m][v]);
      }
  }
  if (n > kmax) return;
  double* y = a.y + S * (yo + static_cast<int64_t>(cl) * a.ycs + static_cast<int64_t>(k0 + n) * a.yks);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = m * 16 + 4 * lk + v;
      if (ROUT % 16 != 0 && row >= ROUT) continue;
      double vr = sr[m][v], vi = C ? si[m][v] : 0.0;
      double* yr = y + S * static_cast<int64_t>(row) * a.yrs;
      if (a.accumulate) {
        vr += yr[0];
        if constexpr (C) vi += yr[1];
      }
      yr[0] = vr;
      if constexpr (C) yr[1] = vi;
    }
}

// ------------------------------------------------------------------ RHS-fastest layout (many RHS)
// With many right-hand sides the internal vectors keep the RHS index fastest, so that a wave's 64
// lanes (64 right-hand sides) read and write 64 consecutive entries:
//   super vectors  v_t[(row * nrhs + k)]            (S doubles per entry)
//   multipole      m_t[((lvl_off[l] + c * rows + r) * nrhs + k)]
// T * X reads the caller's column-major X; T^T * (ys + yf) writes the caller's column-major Y.
template <bool C>
__global__ void k_spmv_tin(int nrows, int nrhs, const int* __restrict__ rp, const int* __restrict__ ci,
                           const double* __restrict__ v, const double* __restrict__ X, int64_t ldx,
                           double* __restrict__ Yt) {
  constexpr int S = C ? 2 : 1;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(nrows) * nrhs) return;
  const int k = static_cast<int>(gid % nrhs), row = static_cast<int>(gid / nrhs);
  const double* xk = X + S * static_cast<int64_t>(k) * ldx;
  double ar = 0.0, ai = 0.0;
  for (int p = rp[row]; p < rp[row + 1]; ++p) {
    const int c = ci[p];
    ar += v[p] * xk[S * c];
    if constexpr (C) ai += v[p] * xk[S * c + 1];
  }
  Yt[S * gid] = ar;
  if constexpr (C) Yt[S * gid + 1] = ai;
}

template <bool C>
__global__ void k_spmv_tout(int nrows, int nrhs, const int* __restrict__ rp, const int* __restrict__ ci,
                            const double* __restrict__ v, const double* __restrict__ At, const double* __restrict__ Bt,
                            double* Y, int64_t ldy, double ar_, double ai_, double br_, double bi_, int use_beta) {
  constexpr int S = C ? 2 : 1;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(nrows) * nrhs) return;
  const int k = static_cast<int>(gid % nrhs), row = static_cast<int>(gid / nrhs);
  double sr = 0.0, si = 0.0;
  for (int p = rp[row]; p < rp[row + 1]; ++p) {
    const int64_t q = S * (static_cast<int64_t>(ci[p]) * nrhs + k);
    double xr = At[q], xi = C ? At[q + 1] : 0.0;
    if (Bt) {
      xr += Bt[q];
      if constexpr (C) xi += Bt[q + 1];
    }
    sr += v[p] * xr;
    if constexpr (C) si += v[p] * xi;
  }
  double* y = Y + S * (static_cast<int64_t>(k) * ldy + row);
  if constexpr (C) {
    double r = ar_ * sr - ai_ * si, im = ar_ * si + ai_ * sr;
    if (use_beta) {
      const double yr = y[0], yi = y[1];
      r += br_ * yr - bi_ * yi;
      im += br_ * yi + bi_ * yr;
    }
    y[0] = r;
    y[1] = im;
  } else {
    double r = ar_ * sr;
    if (use_beta) r += br_ * y[0];
    y[0] = r;
  }
}

// ------------------------------------------------------------------ coupling evaluated on the fly
// Reduced-precision far field without stored coupling blocks: the interpolated kernel
// F(i, j) = w_i w_j k(|x_i - y_j|) of an admissible block (the entry k_coupling_assemble stores)
// is recomputed in FP32 from the Chebyshev surface points of the two clusters, which costs far
// fewer bytes than reading the block.  Points are kept as FP32 offsets from their cluster's first
// point, whose FP64 position gives the block's centre shift, so |x_i - y_j| keeps FP32 relative
// precision for close clusters; each block's FP32 partial sums are added in FP64.
struct FlyArgs {
  int ntgt;
  const int2* tgt;
  const int* rp;
  const int* src;
  const int64_t* lvl_off;  // per level, in clusters x CD rows
  const float4* pts;       // [level cluster][node]: offset from the cluster's node 0 (x, y, z), weight
  const double4* org;      // [level cluster]: node 0 (x, y, z)
  const double* fw;
  double* bw;
  float krev, kim;         // kappa / (2 pi) (phase in revolutions), Im kappa
};

template <bool C, int CD>
__device__ __forceinline__ void coupling_fly_wave(int t, const FlyArgs& a) {
  constexpr int S = C ? 2 : 1;
  constexpr int CDP = CD <= 16 ? 16 : (CD <= 32 ? 32 : 64);
  constexpr int G = 64 / CDP;
  const int lane = threadIdx.x & 63;
  const int g = lane / CDP, li = lane % CDP;
  const int i = li < CD ? li : 0;
  const int2 T = a.tgt[t];
  const int64_t off = a.lvl_off[T.x];  // rows of the level start (one RHS)
  const int64_t coff = off / CD;       // clusters of the level start
  const int p0 = a.rp[t], p1 = a.rp[t + 1];
  const double4 ot = a.org[coff + T.y];
  const float4 xi = a.pts[(coff + T.y) * CD + i];
  double ar = 0.0, ai = 0.0;
  for (int p = p0 + g; p < p1; p += G) {
    const int s2 = a.src[p];
    const double4 os = a.org[coff + s2];
    // x_i - y_j = (o_t - o_s) + (xi - yj)
    const float ex = static_cast<float>(ot.x - os.x) + xi.x;
    const float ey = static_cast<float>(ot.y - os.y) + xi.y;
    const float ez = static_cast<float>(ot.z - os.z) + xi.z;
    const float4* yp = a.pts + (coff + s2) * CD;
    const double* x = a.fw + S * (off + static_cast<int64_t>(s2) * CD);
    float br = 0.f, bi = 0.f;
#pragma unroll
    for (int j = 0; j < CD; ++j) {
      const float4 y = yp[j];
      const float dx = ex - y.x, dy = ey - y.y, dz = ez - y.z;
      const float r2 = dx * dx + dy * dy + dz * dz;
      const float rinv = __builtin_amdgcn_rsqf(r2);
      if constexpr (C) {
        const float vr = y.w * static_cast<float>(x[2 * j]), vi = y.w * static_cast<float>(x[2 * j + 1]);
        const float r = r2 * rinv;
        float mag = rinv;
        if (a.kim != 0.f) mag *= __expf(a.kim * r);
        float ph = r * a.krev;
        ph -= rintf(ph);
        const float cs = __builtin_amdgcn_cosf(ph), sn = __builtin_amdgcn_sinf(ph);
        const float kr = mag * cs, ki = -mag * sn;
        br += kr * vr - ki * vi;
        bi += kr * vi + ki * vr;
      } else {
        br += rinv * (y.w * static_cast<float>(x[j]));
      }
    }
    ar += static_cast<double>(br);
    if constexpr (C) ai += static_cast<double>(bi);
  }
#pragma unroll
  for (int m = CDP; m < 64; m <<= 1) {
    ar += __shfl_xor(ar, m, 64);
    if constexpr (C) ai += __shfl_xor(ai, m, 64);
  }
  if (g == 0 && li < CD) {
    const double wq = static_cast<double>(xi.w) * (0.25 * M_1_PI);
    double* y = a.bw + S * (off + static_cast<int64_t>(T.y) * CD + li);
    y[0] = ar * wq;
    if constexpr (C) y[1] = ai * wq;
  }
}

// single-RHS product sweep of the reduced operator: FP32 near-field blocks and the coupling
// evaluated on the fly in one launch.  Near-field workgroups stream HBM, coupling workgroups
// compute; the two kinds are interleaved along the grid so that both run at once on every CU.
template <bool C, int DD, int CD, int UBN>
__global__ __launch_bounds__(256) void k_sweep_fly(LeafArgs la, FlyArgs fa, int nb_near, int nb_cpl) {
  const int64_t b = blockIdx.x, tot = static_cast<int64_t>(nb_near) + nb_cpl;
  const int64_t cb = b * nb_cpl / tot, cb1 = (b + 1) * nb_cpl / tot;
  const int w = static_cast<int>(threadIdx.x >> 6);
  if (cb1 > cb) {
    const int t = __builtin_amdgcn_readfirstlane(static_cast<int>(cb) * 4 + w);
    if (t < fa.ntgt) coupling_fly_wave<C, CD>(t, fa);
  } else {
    const int c = __builtin_amdgcn_readfirstlane(static_cast<int>(b - cb) * 4 + w);
    if (c < la.ncl) {
      if constexpr (DD % RowVec<C, float>::RPL == 0)
        leaf_wave_v<C, float, DD, UBN>(c, la);
      else
        leaf_wave<C, DD, UBN, float>(c, la);
    }
  }
}

// FP32 node tables of one level for the on-the-fly coupling: offsets from the cluster's node 0
// and the weights, from the FP64 table of k_cluster_points
__global__ void k_fly_points(const double* __restrict__ pts, int ncl, int np2, float4* __restrict__ out,
                             double4* __restrict__ org) {
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(ncl) * np2) return;
  const int64_t c = gid / np2;
  const double* p = pts + gid * CP_STRIDE;
  const double* o = pts + c * np2 * CP_STRIDE;
  out[gid] = make_float4(static_cast<float>(p[0] - o[0]), static_cast<float>(p[1] - o[1]),
                         static_cast<float>(p[2] - o[2]), static_cast<float>(p[3]));
  if (gid % np2 == 0) org[c] = make_double4(o[0], o[1], o[2], 0.0);
}

// FP32 copy of nb coupling blocks (cd x cd, column-major, S doubles per entry) with the columns
// padded to ld rows of zeros, so that rows can be read as 16-byte vectors
__global__ void k_to_fp32_blocks(const double* __restrict__ src, float* __restrict__ dst, int64_t nb, int cd, int ld,
                                 int S) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t per = static_cast<int64_t>(ld) * cd * S;
  if (i >= nb * per) return;
  const int64_t b = i / per;
  const int64_t r = i - b * per;
  const int s = static_cast<int>(r % S);
  const int64_t e = r / S;
  const int row = static_cast<int>(e % ld), col = static_cast<int>(e / ld);
  dst[i] = row < cd ? static_cast<float>(src[((b * cd + col) * cd + row) * S + s]) : 0.f;
}

// BF16 copy (round to nearest even of the FP32 value) of n doubles
__global__ void k_to_bf16(const double* __restrict__ src, unsigned short* __restrict__ dst, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsigned u = __float_as_uint(static_cast<float>(src[i]));
  u += 0x7FFFu + ((u >> 16) & 1u);
  dst[i] = static_cast<unsigned short>(u >> 16);
}

// ------------------------------------------------------------------ host launchers
static inline int nblk(int64_t n) { return static_cast<int>((n + 255) / 256); }

void launch_spmv(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* x,
                 int64_t ldx, double* y, int64_t ldy, const double* alpha, const double* beta, hipStream_t st,
                 const double* x2, bool long_rows) {
  const int64_t n = static_cast<int64_t>(nrows) * nrhs;
  if (n == 0) return;
  const double ar = alpha ? alpha[0] : 1.0, ai = alpha ? alpha[1] : 0.0;
  const double br = beta ? beta[0] : 0.0, bi = beta ? beta[1] : 0.0;
  const int ub = (beta && (br != 0.0 || bi != 0.0)) ? 1 : 0;
  if (long_rows) {
    const int64_t nt = n * 16;
    if (cplx)
      hipLaunchKernelGGL((k_spmv_sub<true, 16>), dim3(nblk(nt)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, x, x2, ldx,
                         y, ldy, ar, ai, br, bi, ub);
    else
      hipLaunchKernelGGL((k_spmv_sub<false, 16>), dim3(nblk(nt)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, x, x2, ldx,
                         y, ldy, ar, ai, br, bi, ub);
    BMI_CHECK_HIP(hipGetLastError());
    return;
  }
  if (cplx)
    hipLaunchKernelGGL(k_spmv<true>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, x, x2, ldx, y, ldy,
                       ar, ai, br, bi, ub);
  else
    hipLaunchKernelGGL(k_spmv<false>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, x, x2, ldx, y, ldy,
                       ar, ai, br, bi, ub);
  BMI_CHECK_HIP(hipGetLastError());
}

bool wave_leaf_supported(int dd) { return dd == 16 || dd == 36; }
bool wave_coupling_supported(int cd) { return cd == 16 || cd == 25; }

void launch_coupling_apply(bool cplx, bool fp32, int variant, int ntgt, int nrhs, int cd, const int2* tgt,
                           const int* rp, const int* src, const void* F, int64_t fstride, const int64_t* lvl_off,
                           const double* fw, double* bw, hipStream_t st, const unsigned short* Fc, int ncoarse, int ld,
                           const PairSweep* pairs) {
  if (ld <= 0) ld = cd;
  const int64_t n = static_cast<int64_t>(ntgt) * nrhs * cd;
  if (n == 0) return;
  TimedScope ts("coupling_apply", st);
  // several columns, and single columns of block sizes without a wave-per-target kernel (the BF16
  // blocks of the coarsest levels are read by the wave kernels only)
  const RowsArgs ra{ntgt, nrhs, cd, ld, 1, tgt, lvl_off, rp, src, F, fstride, fw, 0,
                    static_cast<int64_t>(nrhs) * cd, cd, 1, bw, 0, static_cast<int64_t>(nrhs) * cd, cd, 1,
                    0, 1, 1};
  if (pairs) return launch_pair_rows(cplx, fp32, ra, *pairs, st);
  auto rows = [&] { launch_block_rows(cplx, fp32, ra, st); };
  if (nrhs > 1 && (!Fc || ncoarse == 0)) return rows();
  const dim3 wgrid(static_cast<unsigned>((ntgt + 3) / 4));
  // wave-per-target kernels for the block sizes of the configurations (np 4, 5)
#define BMI_CPL_W(CC, FTT, CDD)                                                                              \
  if (cplx == CC && fp32 == std::is_same<FTT, float>::value && cd == CDD) {                                  \
    const CplArgs ca{ntgt, nrhs, tgt, rp, src, F, fstride, 0, lvl_off, fw, bw, 0, Fc, ncoarse, ld};  \
    if (nrhs == 1 && variant == 1)                                                                            \
      hipLaunchKernelGGL((k_coupling_w<CC, FTT, CDD, 1, 2>), wgrid, dim3(256), 0, st, ca);                    \
    else if (nrhs == 1)                                                                                       \
      hipLaunchKernelGGL((k_coupling_w<CC, FTT, CDD, 1, 1>), wgrid, dim3(256), 0, st, ca);                    \
    else                                                                                                      \
      hipLaunchKernelGGL((k_coupling_w<CC, FTT, CDD, (CC ? 2 : 4), 1>), wgrid, dim3(256), 0, st, ca);         \
    BMI_CHECK_HIP(hipGetLastError());                                                                         \
    return;                                                                                                   \
  }
  BMI_CPL_W(false, double, 16)
  BMI_CPL_W(false, float, 16)
  BMI_CPL_W(true, double, 16)
  BMI_CPL_W(true, float, 16)
  BMI_CPL_W(false, double, 25)
  BMI_CPL_W(false, float, 25)
  BMI_CPL_W(true, double, 25)
  BMI_CPL_W(true, float, 25)
#undef BMI_CPL_W
  rows();
}

// near-field rows of every component: ys = A_near xs (blocks of the vd x vd component pairs dd x dd
// entries apart)
void launch_leaf(bool cplx, int variant, int ncl, int nrhs, int dd, int vd, const int* rp, const int* src,
                 const double* F, const double* xs, int64_t ldxs, int64_t xseg, double* ys, int64_t ldys,
                 int64_t yseg, hipStream_t st) {
  if (ncl <= 0 || nrhs <= 0) return;
  TimedScope ts("matvec_nearfield", st);
  const int64_t dblk = static_cast<int64_t>(dd) * dd;
  if (nrhs == 1 && vd == 1) {
    // wave-per-cluster kernels for the leaf sizes 4 (P+1)^2 of P = 1, 2
    const dim3 wgrid(static_cast<unsigned>((ncl + 3) / 4));
#define BMI_LEAF_W(CC, DDD)                                                                                     \
  if (cplx == CC && dd == DDD) {                                                                                \
    const LeafArgs la{ncl, rp, src, F, dblk, xs, ys};                                                           \
    if (variant == 1)                                                                                           \
      hipLaunchKernelGGL((k_leaf_w<CC, DDD, 2>), wgrid, dim3(256), 0, st, la);                               \
    else                                                                                                        \
      hipLaunchKernelGGL((k_leaf_w<CC, DDD, 1>), wgrid, dim3(256), 0, st, la);                               \
    BMI_CHECK_HIP(hipGetLastError());                                                                           \
    return;                                                                                                     \
  }
    BMI_LEAF_W(false, 16)
    BMI_LEAF_W(true, 16)
    BMI_LEAF_W(false, 36)
    BMI_LEAF_W(true, 36)
#undef BMI_LEAF_W
  }
  launch_block_rows(cplx, false,
                    RowsArgs{ncl, nrhs, dd, dd, vd, nullptr, nullptr, rp, src, F, dblk, xs, xseg, dd, ldxs, 1, ys,
                             yseg, dd, ldys, 1, 0, 1, 1},
                    st);
}

static bool launch_sweep_fused_sym(bool cplx, bool fp32, int leaf_variant, int cpl_variant, int ncl, int dd,
                                   const LeafArgs& la, int cd, const void* cF, int ld, const int64_t* lvl_off,
                                   const double* fw, double* bw, bool near32, const SymList& sl, const SymList* nsl,
                                   hipStream_t st) {
  CplArgs ca{sl.ntgt, 1, sl.tgt, sl.rp, sl.src, cF, static_cast<int64_t>(ld) * cd, 0, lvl_off, fw, bw, 0, nullptr,
             0, ld, sl.blk, sl.part, sl.slot};
  // near field from its upper and diagonal leaves (FP64 blocks): rows and vectors of the super
  // space, the row clusters as targets of one level at offset zero
  const bool nsym = nsl && !near32 && nsl->ntgt == ncl;
  CplArgs na{};
  if (nsym)
    na = CplArgs{nsl->ntgt, 1, nsl->tgt, nsl->rp, nsl->src, la.F, static_cast<int64_t>(dd) * dd, 0, nsl->lvl_off,
                 la.xs, la.ys, 0, nullptr, 0, dd, nsl->blk, nsl->part, nsl->slot};
  const int nbn = (ncl + 3) / 4, nbc = (sl.ntgt + 3) / 4;
  const dim3 grid(static_cast<unsigned>(nbn + nbc));
  bool launched = false;
  {
    TimedScope ts(tl_sweep_scope ? tl_sweep_scope : "matvec_sweep_upper", st);
#define BMI_FUSED_S(CC, DDD, FTT, CDD, UN, UC, NFTT)                                                                 \
  if (!launched && cplx == CC && dd == DDD && fp32 == std::is_same<FTT, float>::value && cd == CDD &&               \
      near32 == std::is_same<NFTT, float>::value && leaf_variant == UN - 1 && cpl_variant == UC - 1) {              \
    if (nsym && std::is_same<NFTT, double>::value)                                                                   \
      hipLaunchKernelGGL((k_sweep_fused_sym<CC, DDD, FTT, CDD, UN, UC, NFTT, true>), grid, dim3(256), 0, st, la,   \
                         ca, nbn, na);                                                                               \
    else                                                                                                             \
      hipLaunchKernelGGL((k_sweep_fused_sym<CC, DDD, FTT, CDD, UN, UC, NFTT, false>), grid, dim3(256), 0, st, la,  \
                         ca, nbn, na);                                                                               \
    BMI_CHECK_HIP(hipGetLastError());                                                                                \
    launched = true;                                                                                                 \
  }
#define BMI_FUSED_SV(CC, DDD, FTT, CDD, NFTT)                                                   \
  BMI_FUSED_S(CC, DDD, FTT, CDD, 1, 1, NFTT) BMI_FUSED_S(CC, DDD, FTT, CDD, 1, 2, NFTT)         \
  BMI_FUSED_S(CC, DDD, FTT, CDD, 2, 1, NFTT) BMI_FUSED_S(CC, DDD, FTT, CDD, 2, 2, NFTT)
    BMI_FUSED_SV(false, 36, double, 16, double)
    BMI_FUSED_SV(true, 36, double, 25, double)
    BMI_FUSED_SV(false, 36, float, 16, float)
    BMI_FUSED_SV(true, 36, float, 25, float)
#undef BMI_FUSED_SV
#undef BMI_FUSED_S
  }
  if (!launched) return false;
  if (nsym && nsl->ngather > 0) {
    TimedScope ts("matvec_sym_gather", st);
    const dim3 gg(static_cast<unsigned>(nblk(static_cast<int64_t>(nsl->ngather) * (cplx ? 2 : 1) * dd / 2)));
    if (cplx && dd == 36)
      hipLaunchKernelGGL((k_sym_gather<true, 36>), gg, dim3(256), 0, st, nsl->ngather, nsl->gtgt, nsl->grp, nsl->part,
                         nsl->lvl_off, la.ys);
    else if (!cplx && dd == 36)
      hipLaunchKernelGGL((k_sym_gather<false, 36>), gg, dim3(256), 0, st, nsl->ngather, nsl->gtgt, nsl->grp,
                         nsl->part, nsl->lvl_off, la.ys);
    else
      throw Error(BMI_UNSUPPORTED, "symmetric near-field gather not instantiated");
    BMI_CHECK_HIP(hipGetLastError());
  }
  if (sl.ngather > 0) {
    TimedScope ts("matvec_sym_gather", st);
    const dim3 gg(static_cast<unsigned>(nblk(static_cast<int64_t>(sl.ngather) * (cplx ? 2 : 1) * cd / 2)));
    if (cplx && cd == 25)
      hipLaunchKernelGGL((k_sym_gather<true, 25>), gg, dim3(256), 0, st, sl.ngather, sl.gtgt, sl.grp, sl.part,
                         lvl_off, bw);
    else if (!cplx && cd == 16)
      hipLaunchKernelGGL((k_sym_gather<false, 16>), gg, dim3(256), 0, st, sl.ngather, sl.gtgt, sl.grp, sl.part,
                         lvl_off, bw);
    else
      throw Error(BMI_UNSUPPORTED, "symmetric gather not instantiated");
    BMI_CHECK_HIP(hipGetLastError());
  }
  return true;
}

thread_local const char* tl_sweep_scope = nullptr;

bool sym_sweep_supported(bool cplx, int dd, int cd) { return dd == 36 && ((cplx && cd == 25) || (!cplx && cd == 16)); }

bool launch_sweep_fused(bool cplx, bool fp32, int leaf_variant, int cpl_variant, int ncl, int dd, const int* drp,
                        const int* dsrc, const void* dF, const double* xs, double* ys, int ntgt, int cd,
                        const int2* tgt, const int* crp, const int* csrc, const void* cF, const int64_t* lvl_off,
                        const double* fw, double* bw, hipStream_t st, const unsigned short* Fc, int ncoarse,
                        bool near32, int ld, const SymList* sym, const SymList* nsym) {
  const LeafArgs la{ncl, drp, dsrc, dF, static_cast<int64_t>(dd) * dd, xs, ys};
  if (ld <= 0) ld = cd;
  if (sym) {
    // upper blocks only: FP64 blocks, or the FP32 copy padded to whole row vectors
    const int rpl = fp32 ? (cplx ? 2 : 4) : 1;
    if (Fc || (fp32 && ld != (cd + rpl - 1) / rpl * rpl)) return false;
    return launch_sweep_fused_sym(cplx, fp32, leaf_variant, cpl_variant, ncl, dd, la, cd, cF, ld, lvl_off, fw, bw,
                                  near32, *sym, nsym, st);
  }
  const CplArgs ca{ntgt, 1, tgt, crp, csrc, cF, static_cast<int64_t>(ld) * cd, 0, lvl_off, fw, bw, 0, Fc, ncoarse, ld};
  const int nbn = (ncl + 3) / 4, nbc = (ntgt + 3) / 4;
  const dim3 grid(static_cast<unsigned>(nbn + nbc));
  TimedScope ts(tl_sweep_scope ? tl_sweep_scope : "matvec_sweep", st);
#define BMI_FUSED(CC, DDD, FTT, CDD, UN, UC, NFTT)                                                              \
  if (cplx == CC && dd == DDD && fp32 == std::is_same<FTT, float>::value && cd == CDD &&                        \
      near32 == std::is_same<NFTT, float>::value && leaf_variant == UN - 1 && cpl_variant == UC - 1) {          \
    hipLaunchKernelGGL((k_sweep_fused<CC, DDD, FTT, CDD, UN, UC, NFTT>), grid, dim3(256), 0, st, la, ca, nbn,    \
                       CplArgs{});                                                                                \
    BMI_CHECK_HIP(hipGetLastError());                                                                           \
    return true;                                                                                                \
  }
#define BMI_FUSED_V(CC, DDD, FTT, CDD, NFTT)                                                   \
  BMI_FUSED(CC, DDD, FTT, CDD, 1, 1, NFTT) BMI_FUSED(CC, DDD, FTT, CDD, 1, 2, NFTT)            \
  BMI_FUSED(CC, DDD, FTT, CDD, 2, 1, NFTT) BMI_FUSED(CC, DDD, FTT, CDD, 2, 2, NFTT)
  BMI_FUSED_V(false, 36, double, 16, double)
  BMI_FUSED_V(false, 36, float, 16, double)
  BMI_FUSED_V(true, 36, double, 25, double)
  BMI_FUSED_V(true, 36, float, 25, double)
  BMI_FUSED_V(true, 36, double, 16, double)
  BMI_FUSED_V(true, 36, float, 16, double)
  BMI_FUSED_V(false, 16, double, 16, double)
  BMI_FUSED_V(true, 16, double, 16, double)
  // reduced operators with the FP32 near-field copy
  BMI_FUSED_V(false, 36, float, 16, float)
  BMI_FUSED_V(false, 36, float, 25, float)
  BMI_FUSED_V(true, 36, float, 25, float)
  BMI_FUSED_V(true, 36, float, 16, float)
  BMI_FUSED_V(false, 16, float, 16, float)
  BMI_FUSED_V(true, 16, float, 16, float)
#undef BMI_FUSED_V
#undef BMI_FUSED
  return false;
}

void launch_fly_points(const double* pts, int ncl, int np2, float4* out, double4* org, hipStream_t st) {
  const int64_t n = static_cast<int64_t>(ncl) * np2;
  if (n == 0) return;
  hipLaunchKernelGGL(k_fly_points, dim3(nblk(n)), dim3(256), 0, st, pts, ncl, np2, out, org);
  BMI_CHECK_HIP(hipGetLastError());
}

bool launch_sweep_fly(bool cplx, int variant, int ncl, int dd, const int* drp, const int* dsrc, const float* dF32,
                      const double* xs, double* ys, int ntgt, int cd, const int2* tgt, const int* crp,
                      const int* csrc, const int64_t* lvl_off, const float4* pts, const double4* org,
                      double kre, double kim, const double* fw, double* bw, hipStream_t st) {
  const LeafArgs la{ncl, drp, dsrc, dF32, static_cast<int64_t>(dd) * dd, xs, ys};
  const FlyArgs fa{ntgt, tgt, crp, csrc, lvl_off, pts, org, fw, bw, static_cast<float>(kre * 0.5 * M_1_PI),
                   static_cast<float>(kim)};
  const int nbn = (ncl + 3) / 4, nbc = (ntgt + 3) / 4;
  const dim3 grid(static_cast<unsigned>(nbn + nbc));
  TimedScope ts("matvec_sweep", st);
#define BMI_FLY(CC, DDD, CDD)                                                                              \
  if (cplx == CC && dd == DDD && cd == CDD) {                                                              \
    if (variant == 1)                                                                                      \
      hipLaunchKernelGGL((k_sweep_fly<CC, DDD, CDD, 2>), grid, dim3(256), 0, st, la, fa, nbn, nbc);        \
    else                                                                                                   \
      hipLaunchKernelGGL((k_sweep_fly<CC, DDD, CDD, 1>), grid, dim3(256), 0, st, la, fa, nbn, nbc);        \
    BMI_CHECK_HIP(hipGetLastError());                                                                      \
    return true;                                                                                           \
  }
  BMI_FLY(false, 36, 16)
  BMI_FLY(false, 36, 25)
  BMI_FLY(false, 16, 16)
#undef BMI_FLY
  return false;
}

void launch_spmv_tin(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* X,
                     int64_t ldx, double* Yt, hipStream_t st) {
  const int64_t n = static_cast<int64_t>(nrows) * nrhs;
  if (n == 0) return;
  if (cplx)
    hipLaunchKernelGGL(k_spmv_tin<true>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, X, ldx, Yt);
  else
    hipLaunchKernelGGL(k_spmv_tin<false>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, X, ldx, Yt);
  BMI_CHECK_HIP(hipGetLastError());
}

void launch_spmv_tout(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* At,
                      const double* Bt, double* Y, int64_t ldy, const double* alpha, const double* beta,
                      hipStream_t st) {
  const int64_t n = static_cast<int64_t>(nrows) * nrhs;
  if (n == 0) return;
  const double ar = alpha ? alpha[0] : 1.0, ai = alpha ? alpha[1] : 0.0;
  const double br = beta ? beta[0] : 0.0, bi = beta ? beta[1] : 0.0;
  const int ub = (beta && (br != 0.0 || bi != 0.0)) ? 1 : 0;
  if (cplx)
    hipLaunchKernelGGL(k_spmv_tout<true>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, At, Bt, Y, ldy, ar,
                       ai, br, bi, ub);
  else
    hipLaunchKernelGGL(k_spmv_tout<false>, dim3(nblk(n)), dim3(256), 0, st, nrows, nrhs, rp, ci, v, At, Bt, Y, ldy, ar,
                       ai, br, bi, ub);
  BMI_CHECK_HIP(hipGetLastError());
}

// instantiations of k_multi_lds: block products (XC = FC) and the tree steps (real blocks)
static bool launch_lds(bool xc, bool fc, bool fp32, int rout, int rin, const MultiArgs& ma, dim3 grid,
                       hipStream_t st) {
#define BMI_LDS(X, FCC, FTT, RO, RI)                                                                \
  if (xc == X && fc == FCC && fp32 == std::is_same<FTT, float>::value && rout == RO && rin == RI) { \
    hipLaunchKernelGGL((k_multi_lds<X, FCC, FTT, RO, RI>), grid, dim3(256), 0, st, ma);            \
    BMI_CHECK_HIP(hipGetLastError());                                                               \
    return true;                                                                                    \
  }
#define BMI_LDS_BLK(X, R) BMI_LDS(X, X, double, R, R) BMI_LDS(X, X, float, R, R)
#define BMI_LDS_TREE(X, A, B) BMI_LDS(X, false, double, A, B) BMI_LDS(X, false, double, B, A)
  BMI_LDS_BLK(false, 16)
  BMI_LDS_BLK(false, 25)
  BMI_LDS_BLK(false, 36)
  BMI_LDS_BLK(true, 16)
  BMI_LDS_BLK(true, 25)
  BMI_LDS_BLK(true, 32)
  BMI_LDS_BLK(true, 36)
  BMI_LDS(true, false, double, 16, 16)
  BMI_LDS(true, false, double, 25, 25)
  BMI_LDS_TREE(false, 16, 36)
  BMI_LDS_TREE(false, 25, 16)
  BMI_LDS_TREE(false, 25, 36)
  BMI_LDS_TREE(true, 16, 36)
  BMI_LDS_TREE(true, 25, 16)
  BMI_LDS_TREE(true, 25, 36)
  BMI_LDS_TREE(true, 32, 16)
  BMI_LDS_TREE(true, 32, 36)
#undef BMI_LDS_TREE
#undef BMI_LDS_BLK
#undef BMI_LDS
  return false;
}

// compute units of the current device
static int device_cus() {
  static const int n = [] {
    int d = 0, v = 0;
    if (hipGetDevice(&d) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, d) !=
                                              hipSuccess || v < 8)
      v = 256;
    return v;
  }();
  return n;
}

// a block sweep: 8 S workgroups, S per XCD, each over every S-th owner of its XCD's range; S is
// what an XCD holds at once (measured, 64-RHS Helmholtz M = 5: near-field sweep 0.22 ms against
// 0.25 ms with one owner per workgroup, coupling sweep 0.44 against 0.47 ms)
template <bool X, typename FTT, int R>
static void launch_mfma_sweep(const MultiArgs& ma, unsigned rhs_tiles, hipStream_t st) {
  const void* fn = reinterpret_cast<const void*>(&k_multi_mfma<X, X, FTT, R, R, true>);
  static const int per_cu = [fn] {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, 256, 0) != hipSuccess || nb < 1) nb = 1;
    return nb;
  }();
  const int per_xcd = (ma.nown + 7) / 8;
  const int S = std::min(per_xcd, std::max(1, device_cus() / 8 * per_cu));
  if (S <= 0) return;
  hipLaunchKernelGGL((k_multi_mfma<X, X, FTT, R, R, true>), dim3(static_cast<unsigned>(8 * S), rhs_tiles, 1),
                     dim3(256), 0, st, ma);
  BMI_CHECK_HIP(hipGetLastError());
}

// block products (XL form) and tree steps (staged x) on the matrix cores
static bool launch_mfma(bool xc, bool fc, bool fp32, int rout, int rin, const MultiArgs& ma, dim3 grid,
                        hipStream_t st) {
#define BMI_MF(X, FCC, FTT, RO, RI)                                                                  \
  if (xc == X && fc == FCC && fp32 == std::is_same<FTT, float>::value && rout == RO && rin == RI) {  \
    hipLaunchKernelGGL((k_multi_mfma<X, FCC, FTT, RO, RI, false>), grid, dim3(256), 0, st, ma);      \
    BMI_CHECK_HIP(hipGetLastError());                                                                \
    return true;                                                                                     \
  }
#define BMI_MF_SWEEP(X, FTT, R)                                                                       \
  if (ma.mode == 0 && xc == X && fc == X && fp32 == std::is_same<FTT, float>::value && rout == R &&    \
      rin == R) {                                                                                      \
    launch_mfma_sweep<X, FTT, R>(ma, grid.y, st);                                                      \
    return true;                                                                                       \
  }
#define BMI_MF_BLK(X, R) BMI_MF_SWEEP(X, double, R) BMI_MF_SWEEP(X, float, R)
#define BMI_MF_TREE(X, A, B) BMI_MF(X, false, double, A, B) BMI_MF(X, false, double, B, A)
  BMI_MF_BLK(false, 16)
  BMI_MF_BLK(false, 25)
  BMI_MF_BLK(false, 36)
  BMI_MF_BLK(true, 16)
  BMI_MF_BLK(true, 25)
  BMI_MF_BLK(true, 32)
  BMI_MF_BLK(true, 36)
  BMI_MF(true, false, double, 16, 16)
  BMI_MF(true, false, double, 25, 25)
  BMI_MF(false, false, double, 16, 16)
  BMI_MF(false, false, double, 25, 25)
  BMI_MF_TREE(false, 16, 36)
  BMI_MF_TREE(false, 25, 16)
  BMI_MF_TREE(false, 25, 36)
  BMI_MF_TREE(true, 16, 36)
  BMI_MF_TREE(true, 25, 16)
  BMI_MF_TREE(true, 25, 36)
  BMI_MF_TREE(true, 32, 16)
  BMI_MF_TREE(true, 32, 36)
#undef BMI_MF_TREE
#undef BMI_MF_BLK
#undef BMI_MF_SWEEP
#undef BMI_MF
  return false;
}

// FP32 blocks on the FP32 matrix cores (block sums FP32, sums over blocks FP64)
static bool launch_mfma32(bool cplx, int rows, const MultiArgs& ma, dim3 grid, hipStream_t st) {
#define BMI_MF32(CC, R)                                                             \
  if (cplx == CC && rows == R) {                                                  \
    hipLaunchKernelGGL((k_multi_mfma32<CC, R, R>), grid, dim3(256), 0, st, ma);   \
    BMI_CHECK_HIP(hipGetLastError());                                             \
    return true;                                                                  \
  }
  BMI_MF32(false, 16)
  BMI_MF32(false, 25)
  BMI_MF32(false, 36)
  BMI_MF32(true, 16)
  BMI_MF32(true, 25)
  BMI_MF32(true, 32)
  BMI_MF32(true, 36)
#undef BMI_MF32
  return false;
}

// FP32 blocks widened to FP64 on the FP64 matrix cores (default: the accuracy of the single-RHS
// reduced products, 1e-8, and the FP64 Krylov step count), or multiplied in FP32 on the FP32
// matrix cores (BMI_MULTI_MATH32=1: 1.3x faster products at 1e-7, which cost restarted GMRES
// about half as many steps again on the 64-RHS Helmholtz M = 5 problem)
static bool multi_math32() {
  static const bool on = [] {
    const char* v = std::getenv("BMI_MULTI_MATH32");
    return v && v[0] == '1';
  }();
  return on;
}

// block products of the RHS-fastest sweeps: 1 = matrix cores, 0 = vector units (BMI_MULTI_VECTOR=1)
static int multi_engine() {
  static const int e = [] {
    const char* v = std::getenv("BMI_MULTI_VECTOR");
    return (v && v[0] == '1') ? 0 : 1;
  }();
  return e;
}

// the LDS copy moves whole 8-byte units: blocks must start and end on them and fit the tile
static bool multi_lds_fits(bool fc, bool fp32, int rout, int rin, int ld, int64_t fstride, int64_t fcomp) {
  const int64_t es = (fc ? 2 : 1) * (fp32 ? 4 : 8);
  const int ldmax = (rout + 3) / 4 * 4;
  return ld >= rout && ld <= ldmax && (es * fstride) % 8 == 0 && (es * fcomp) % 8 == 0 &&
         (es * ld * rin) % 8 == 0;
}

static MultiArgs tree_args(int nown, int nrhs, int mode, const double* F, int64_t fstride, int ld, const double* x,
                           int64_t xoff, int64_t xcs, double* y, int64_t yoff, int64_t ycs, int accumulate) {
  MultiArgs ma{};
  ma.nown = nown;
  ma.nrhs = nrhs;
  ma.F = F;
  ma.fstride = fstride;
  ma.ldf = ld;
  ma.x = x;
  ma.xoff = xoff;
  ma.xcs = xcs;
  ma.xks = 1;
  ma.xrs = nrhs;
  ma.y = y;
  ma.yoff = yoff;
  ma.ycs = ycs;
  ma.yks = 1;
  ma.yrs = nrhs;
  ma.accumulate = accumulate;
  ma.mode = mode;
  return ma;
}

static void tree_step(bool cplx, int rout, int rin, const MultiArgs& ma, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(ma.nown), static_cast<unsigned>((ma.nrhs + 63) / 64), 1);
  const bool ok = multi_engine() == 1 ? launch_mfma(cplx, false, false, rout, rin, ma, grid, st)
                                      : launch_lds(cplx, false, false, rout, rin, ma, grid, st);
  BMI_REQUIRE(ok, BMI_UNSUPPORTED, "tree step without an RHS-fastest instantiation");
}

void launch_forward_t(bool cplx, int npatch, int L, int rows, int np2, int dd, int nrhs, const double* mom,
                      const double* T, const double* xs_t, int64_t xseg, double* fw_t, const int64_t* lvl_off,
                      hipStream_t st) {
  const int64_t R = nrhs;
  // leaf moments: fw_L[c] = Mom (rows x dd) xs[c]
  tree_step(cplx, rows, dd,
            tree_args(npatch << (2 * L), nrhs, 3, mom, 0, rows, xs_t, xseg * R, dd * R, fw_t, lvl_off[L] * R,
                      rows * R, 0),
            st);
  // parents from children, per interpolation component: fw_l[c] = sum_q T_q fw_{l+1}[4c + q]
  for (int l = L - 1; l >= 0; --l)
    for (int comp = 0; comp * np2 < rows; ++comp)
      tree_step(cplx, np2, np2,
                tree_args(npatch << (2 * l), nrhs, 1, T, static_cast<int64_t>(np2) * np2, np2, fw_t,
                          (lvl_off[l + 1] + comp * np2) * R, rows * R, fw_t, (lvl_off[l] + comp * np2) * R,
                          rows * R, 0),
                st);
}

void launch_backward_t(bool cplx, int npatch, int L, int rows, int np2, int dd, int nrhs, const double* momt,
                       const double* Tt, double* bw_t, const int64_t* lvl_off, double* yf_t, int64_t yseg,
                       hipStream_t st) {
  const int64_t R = nrhs;
  // children += T_q^T parent
  for (int l = 1; l <= L; ++l)
    for (int comp = 0; comp * np2 < rows; ++comp)
      tree_step(cplx, np2, np2,
                tree_args(npatch << (2 * l), nrhs, 2, Tt, static_cast<int64_t>(np2) * np2, np2, bw_t,
                          (lvl_off[l - 1] + comp * np2) * R, rows * R, bw_t, (lvl_off[l] + comp * np2) * R,
                          rows * R, 1),
                st);
  // leaf rows: yf[c] = Mom^T (dd x rows) bw_L[c]
  tree_step(cplx, dd, rows,
            tree_args(npatch << (2 * L), nrhs, 3, momt, 0, dd, bw_t, lvl_off[L] * R, rows * R, yf_t, yseg * R,
                      dd * R, 0),
            st);
}

bool multi_t_supported(bool cplx, int dd, int cd) {
  return (dd == 16 || dd == 36) && (cd == 16 || cd == 25 || (cplx && cd == 32));
}

bool launch_multi_near_t(bool cplx, bool fp32, int ncl, int nrhs, int dd, const int* rp, const int* src,
                         const void* F, int64_t fstride, int64_t fcomp, const double* xs_t, int64_t xseg,
                         double* ys_t, int64_t yseg, int accumulate, hipStream_t st) {
  const MultiArgs ma{ncl, nrhs, nullptr, nullptr, rp, src, F, fstride, fcomp, dd,
                     xs_t, xseg * nrhs, static_cast<int64_t>(dd) * nrhs, 1, nrhs,
                     ys_t, yseg * nrhs, static_cast<int64_t>(dd) * nrhs, 1, nrhs, accumulate, 0};
  TimedScope ts("matvec_nearfield", st);
  const dim3 grid(static_cast<unsigned>(ncl), static_cast<unsigned>((nrhs + 63) / 64), 1);
  if (multi_engine() == 1 && fp32 && multi_math32()) return launch_mfma32(cplx, dd, ma, grid, st);
  if (multi_engine() == 1) return launch_mfma(cplx, cplx, fp32, dd, dd, ma, grid, st);
  if (!multi_lds_fits(cplx, fp32, dd, dd, dd, fstride, fcomp)) return false;
  return launch_lds(cplx, cplx, fp32, dd, dd, ma, grid, st);
}

bool launch_multi_cpl_t(bool cplx, bool fp32, int ntgt, int nrhs, int cd, int ld, const int2* tgt, const int* rp,
                        const int* src, const void* F, int64_t fstride, int64_t fcomp, const int64_t* lvl_off,
                        const double* fw_t, double* bw_t, int accumulate, hipStream_t st) {
  const MultiArgs ma{ntgt, nrhs, tgt, lvl_off, rp, src, F, fstride, fcomp, ld,
                     fw_t, 0, static_cast<int64_t>(cd) * nrhs, 1, nrhs,
                     bw_t, 0, static_cast<int64_t>(cd) * nrhs, 1, nrhs, accumulate, 0};
  TimedScope ts("coupling_apply", st);
  const dim3 grid(static_cast<unsigned>(ntgt), static_cast<unsigned>((nrhs + 63) / 64), 1);
  if (multi_engine() == 1 && ld >= cd && ld <= (cd + 3) / 4 * 4) {
    if (fp32 && multi_math32()) return launch_mfma32(cplx, cd, ma, grid, st);
    return launch_mfma(cplx, cplx, fp32, cd, cd, ma, grid, st);
  }
  if (!multi_lds_fits(cplx, fp32, cd, cd, ld, fstride, fcomp)) return false;
  return launch_lds(cplx, cplx, fp32, cd, cd, ma, grid, st);
}

int fp32_coupling_ld(bool cplx, int cd) {
  const int rpl = cplx ? 2 : 4;
  return (cd + rpl - 1) / rpl * rpl;
}

void launch_mx_prep(int64_t ne, int nrhs, int np2, int cd, const double* fw0, const double* fw1, const double* tan,
                    double* Z, hipStream_t st) {
  const int64_t n = ne * nrhs * np2;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mx_prep, dim3(nblk(n)), dim3(256), 0, st, ne, nrhs, np2, cd, fw0, fw1, tan, Z);
  BMI_CHECK_HIP(hipGetLastError());
}

// One block-row sweep of 4 nrhs columns over the kernel values.  Against a workgroup per target and
// right-hand side with a row of K per thread (3.25 TB/s; product of 1,536 elements, P 2, 9x9 nodes, one
// column): 872 -> 662 us.
void launch_mx_coupling(bool fp32, int ntgt_all, int nrhs, int np2, int cd, const int* order, const int2* tgt_all,
                        const int* rp_all, const int* src, const void* K, const int64_t* lvl_off, const double* Z,
                        double* w0, double* w1, const PairSweep* pairs, hipStream_t st) {
  if (ntgt_all <= 0 || nrhs <= 0) return;
  if (np2 > 256) throw Error(BMI_UNSUPPORTED, "Maxwell far field with more than 16x16 Chebyshev nodes");
  TimedScope ts("coupling_apply", st);
  // x: 4 nrhs columns per cluster; y: cd rows per cluster and right-hand side, twice np2 of either half
  RowsArgs a{ntgt_all, 4 * nrhs, np2, np2, 1, tgt_all, lvl_off, rp_all, src, K, static_cast<int64_t>(np2) * np2, Z, 0,
             static_cast<int64_t>(4) * nrhs * np2, np2, 1, w0, 0, static_cast<int64_t>(nrhs) * cd, np2, 1, 0, 1, 1};
  a.xl = 2 * nrhs, a.yl = nrhs;
  a.order = order;
  a.y1 = w1, a.ysplit = 2 * nrhs;
  if (pairs)
    launch_pair_rows(true, fp32, a, *pairs, st);
  else
    launch_block_rows(true, fp32, a, st);
}

void launch_mx_finish(int64_t ne, int nrhs, int np2, int cd, const double* tan, double* w0, double* w1, double qre,
                      double qim, hipStream_t st) {
  const int64_t n = ne * nrhs * np2;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mx_finish, dim3(nblk(n)), dim3(256), 0, st, ne, nrhs, np2, cd, tan, w0, w1, qre, qim);
  BMI_CHECK_HIP(hipGetLastError());
}

void convert_blocks_to_fp32(const double* src, float* dst, int64_t nb, int cd, int ld, bool cplx, hipStream_t st) {
  const int64_t n = nb * ld * cd * (cplx ? 2 : 1);
  if (n <= 0) return;
  hipLaunchKernelGGL(k_to_fp32_blocks, dim3(nblk(n)), dim3(256), 0, st, src, dst, nb, cd, ld, cplx ? 2 : 1);
  BMI_CHECK_HIP(hipGetLastError());
}

void convert_to_bf16(const double* src, unsigned short* dst, int64_t n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_to_bf16, dim3(nblk(n)), dim3(256), 0, st, src, dst, n);
  BMI_CHECK_HIP(hipGetLastError());
}

}  // namespace bmi
