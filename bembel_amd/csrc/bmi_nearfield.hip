// Near-field Galerkin quadrature on the GPU: one workgroup per element pair.
//
// Restates DuffyTrick::integrate0..4 (DuffyTrick/integrate0.hpp:22-38, integrate1.hpp:25-48,
// integrate2.hpp:27-67, integrate3.hpp:27-80, integrate4.hpp:27-64) for the Laplace and
// Helmholtz single-layer integrands (Laplace/SingleLayerOperator.hpp:44-85,
// Helmholtz/SingleLayerOperator.hpp:44-85), the Maxwell single layer (EFIE,
// Maxwell/SingleLayerOperator.hpp:44-88) and the test operator
// (LinearOperator/Dummy/DummyOperator.hpp:53-59).
//
// Design: all lanes of a workgroup work on the same element pair, so the elements' polynomials
// (k_element_poly) are wave-uniform and are read through the scalar cache.  The scalar operators run
// factorised rules: a lane fixes an outer point, sums kernel x basis over inner points, and the outer
// products of the sums go to the block -- on the matrix cores where a block per lane would cost the
// second wave per SIMD (identical and edge rules), in registers else.  Maxwell blocks (four
// (P+1)^2 x (P+1)^2 complex component blocks; blockIdx.y = 2*row component + column component) are
// accumulated per evaluation.  Bound: FP64 VALU.
//
// Measured, 24,576 elements of the sphere, P 2, 13 points per direction for touching pairs, against
// points in Bernstein form, blocks in registers and the library's sine and cosine: Laplace identical 58.0
// -> 22.7 ms, edge 97.0 -> 41.3, vertex 18.6 -> 17.6, regular 16.6 -> 15.9; Helmholtz identical 82.5 ->
// 29.3, edge 149.5 -> 69.2, vertex 54.7 -> 46.4, regular 35.7 -> 30.8 (VALU busy: Laplace identical 0.77, edge
// 0.71, vertex 0.69, regular 0.60).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "bmi_internal.h"
#include "bmi_device.h"

namespace bmi {

struct NFParams {
  const double* poly;  // element polynomials, 4 PD^2 doubles per element (k_element_poly)
  int poly_stride;
  double h;        // element width in the parameter domain
  double rh, rh2;  // 1 / h, 1 / h^2 (powers of two)
  // powers of two with the size l of the geometry in them, about l^-4 and (l / h)^2: squared measures of line
  // points times ms are of order one at any unit of length, and mr takes the factor back
  double ms, mr;
  double kre, kim;  // wavenumber
  int dummy_fn;
  const double* ffield;  // far-field table, FF_STRIDE doubles per point
  int nff;               // points per element in the table
  int ffs;               // doubles per point in the table
  double* out;
  int64_t rs, cs;  // row / column stride of a block in the output (in scalars)
  int64_t comp_rs, comp_cs;  // offsets of the vector components (Maxwell)
  double qre, qim;           // -1 / (kappa^2 h^2): divergence-part factor (Maxwell)
};

// far-field table record: x0 x1 x2 kappa w s0 s1 pad [ds0 ds1 ds2 dt0 dt1 dt2 pad pad]

// 1 / x, x != 0: the hardware estimate (v_rcp_f64) refined by two steps of Newton's iteration
// for the reciprocal, y <- y + y (1 - x y) (residual by an FMA); within an ulp or two of the
// rounded quotient, for half the instructions of a division
__device__ __forceinline__ double rcp_newton(double x) {
  double y = __builtin_amdgcn_rcp(x);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const double e = fma(-x, y, 1.0);
    y = fma(y, e, y);
  }
  return y;
}

// evaluation point of the integrand: physical point, weight (kappa*w or w), local coords;
// Maxwell also keeps the two tangent vectors
template <int KIND>
struct Pt {
  double x0, x1, x2, W, s0, s1;
};
template <>
struct Pt<BMI_MAXWELL_SL> {
  double x0, x1, x2, W, s0, s1;
  double t[6];  // d/ds x, d/dt x
};

// Surface points.  A patch is a rational polynomial of degree PD - 1 in either parameter; on one element
// its four homogeneous coordinates are kept in powers of the centred local coordinates u - 1/2,
// v - 1/2 (G[(a * PD + b) * 4 + k], k_element_poly): values and derivatives take half the operations
// of the Bernstein form (no basis to evaluate), and |u - 1/2| <= 1/2 keeps the sums as well
// conditioned.  With x = p / w the tangents are (p_u - x w_u) / w, (p_v - x w_v) / w; derivatives
// in the patch parameters are 1 / h times those in u, v.
// The coordinates are those about the element's centre, rounded to single precision (the table's last entries;
// zero for the test operator, whose values depend on the place): what all points of an element share, the
// rounding of its coefficients, is then small against the element and not against the body, and the distances
// of touching elements keep it.  Blocks of edge neighbours of 6,144 elements, P 2, against extended precision:
// coefficients summed in doubles about the origin 1.5e-15 (points in Bernstein form, each rounded for itself,
// 5.2e-16), so 4.5e-16, 1.7e-16 with the sums of add_products.
// element polynomials, written by an earlier kernel only: in the constant address space, so that
// wave-uniform loads go through the scalar cache wherever they stand (as plain global memory the
// compiler gave that up in the longer rules)
typedef const __attribute__((address_space(4))) double* PolyPtr;

// a point of one element about the centre of the other; the centres are read where they are used, as the
// coefficients
struct Shift {
  PolyPtr o1, o2;
  template <class PT>
  __device__ __forceinline__ static PT moved(PT p, PolyPtr from, PolyPtr to) {
    asm volatile("" : "+s"(from), "+s"(to));
    p.x0 += from[0] - to[0], p.x1 += from[1] - to[1], p.x2 += from[2] - to[2];
    return p;
  }
  template <class PT>
  __device__ __forceinline__ PT to_second(const PT& p) const { return moved(p, o1, o2); }
  template <class PT>
  __device__ __forceinline__ PT to_first(const PT& p) const { return moved(p, o2, o1); }
};

// Sums over wave-uniform coefficients (scalar registers) take powers of the coordinate: of the operands
// of a multiply-add one may be scalar, and a Horner chain starts with two (moves into vector registers
// were half the instructions of a contraction).
template <int PD>
struct Powers {
  double f[PD], d[PD];  // t^a, a t^(a - 1)
  __device__ explicit Powers(double t) {
    f[0] = 1.0, d[0] = 0.0;
#pragma unroll
    for (int a = 1; a < PD; ++a) f[a] = f[a - 1] * t, d[a] = a * f[a - 1];
  }
  // r = sum g(a) t^a, rd its derivative
  template <class Coef>
  __device__ void sum(Coef g, double& r, double& rd) const {
    r = g(PD - 1) * f[PD - 1], rd = g(PD - 1) * d[PD - 1];
#pragma unroll
    for (int a = PD - 2; a >= 1; --a) r = fma(g(a), f[a], r);
#pragma unroll
    for (int a = PD - 2; a >= 2; --a) rd = fma(g(a), d[a], rd);
    r += g(0);
    if constexpr (PD > 2) rd += g(1);
  }
};

template <int PD>
__device__ __forceinline__ void poly_point(PolyPtr G, double u, double v, double X[3], double Eu[3],
                                           double Ev[3], double& bot) {
  // G is uniform: the coefficients are loaded at every point (kept across a loop they would fill the
  // vector registers)
  asm volatile("" : "+s"(G));
  v -= 0.5;
  Powers<PD> q(u - 0.5);
  double p[4] = {0, 0, 0, 0}, pu[4] = {0, 0, 0, 0}, pv[4] = {0, 0, 0, 0};
#pragma unroll
  for (int b = PD - 1; b >= 0; --b) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double r, ru;
      q.sum([&](int a) { return G[(a * PD + b) * 4 + k]; }, r, ru);
      pv[k] = fma(pv[k], v, p[k]);
      p[k] = fma(p[k], v, r);
      pu[k] = fma(pu[k], v, ru);
    }
  }
  bot = rcp_newton(p[3]);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    X[k] = p[k] * bot;
    Eu[k] = fma(-X[k], pu[3], pu[k]);
    Ev[k] = fma(-X[k], pv[3], pv[k]);
  }
}

// |a x b|^2
__device__ __forceinline__ double cross_square(const double a[3], const double b[3]) {
  const double c0 = a[1] * b[2] - a[2] * b[1];
  const double c1 = a[2] * b[0] - a[0] * b[2];
  const double c2 = a[0] * b[1] - a[1] * b[0];
  return c0 * c0 + c1 * c1 + c2 * c2;
}

template <int PD, int KIND>
__device__ __forceinline__ Pt<KIND> make_point(PolyPtr G, const NFParams& prm, double u, double v,
                                               double w) {
  double X[3], Eu[3], Ev[3], bot;
  poly_point<PD>(G, u, v, X, Eu, Ev, bot);
  Pt<KIND> p;
  p.x0 = X[0], p.x1 = X[1], p.x2 = X[2];
  p.s0 = u, p.s1 = v;
  if constexpr (KIND == BMI_MAXWELL_SL) {
    // the vector basis carries no surface measure: the Piola factor cancels
    // (Maxwell/SingleLayerOperator.hpp:71-85)
    p.W = w;
    const double f = bot * prm.rh;
#pragma unroll
    for (int k = 0; k < 3; ++k) p.t[k] = Eu[k] * f, p.t[3 + k] = Ev[k] * f;
  } else if (KIND == BMI_DUMMY) {
    p.W = w;
  } else {
    p.W = sqrt(cross_square(Eu, Ev)) * (bot * bot) * (prm.rh2 * w);
  }
  return p;
}

// test functions of the reference Duffy unit tests (tests/DuffyTrick/test_testFunctions.hpp)
template <class PA, class PB>
__device__ __forceinline__ double dummy_value(int fn, const PA& a, const PB& b) {
  if (fn == 0)
    return sin(M_PI * a.x0) * sin(2 * M_PI * b.x0) * exp(-a.x1) * exp(b.x1);
  if (fn == 1) {
    const double c = a.x1 - b.x0;
    return exp(-a.x0 - 2 * b.x1) * (1. / (1e-3 + c * c));
  }
  return 1.0;
}

// Block accumulation split over groups of G lanes.  Each lane evaluates its own integrand point
// (surface points, kernel, Bernstein values); the G lanes of a group exchange those values and
// each adds all G evaluations to its part of the block: for complex operators the lane role
// (lane mod G) picks real or imaginary parts (role & 1) and, with G = 4, a half of the rows
// (role >> 1).  Per lane this divides the accumulator registers by G at the same number of
// multiply-adds; real blocks (G = 1) stay whole in every lane.  Complex blocks use G = 2 (a
// four-way split halves the accumulators again but doubles the exchanges, which measured
// slower for P = 2).
template <int P, int KIND>
struct BlockAcc {
  static constexpr int I = P + 1;
  static constexpr int I2 = I * I;
  static constexpr bool CPLX = KIND == BMI_HELMHOLTZ_SL || KIND == BMI_MAXWELL_SL;
  static constexpr bool MAXW = KIND == BMI_MAXWELL_SL;
  // lanes per group: two lanes hold a block, real blocks split into two halves of their rows,
  // complex ones into their real and imaginary parts (splitting complex blocks into four lanes
  // as well measured slower: Helmholtz edge rule 182 -> 303 ms, more sums exchanged per pass)
  static constexpr int G = 2;
  static constexpr int RH = CPLX ? G / 2 : G;         // row halves
  static constexpr int NR = (I2 + RH - 1) / RH;       // rows held per lane
  static constexpr int ID = MAXW ? I : 1;
  static constexpr int TOT = CPLX ? 2 * I2 * I2 : I2 * I2;
  double acc[NR * I2];

  // what the block update needs from one evaluation
  struct Eval {
    double vr, vi;  // kernel x weights (x tangent product for Maxwell)
    double qr, qi;  // Maxwell divergence factor
    double X[I], Y[I], U[I], V[I];
    double DX[ID], DY[ID], DU[ID], DV[ID];
  };

  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int k = 0; k < NR * I2; ++k) acc[k] = 0.0;
  }

  // one evaluation of the integrand; a lane without work (valid = false) contributes zero
  __device__ __forceinline__ Eval eval(const Pt<KIND>& a, const Pt<KIND>& b, const NFParams& prm, int rc, int cc,
                                       bool valid) const {
    Eval e;
    const double d0 = a.x0 - b.x0, d1 = a.x1 - b.x1, d2 = a.x2 - b.x2;
    const double s = d0 * d0 + d1 * d1 + d2 * d2;
    const double ri = rsqrt_newton(s);  // 1 / r
    const double r = s * ri;
    e.vi = 0.0, e.qr = 0.0, e.qi = 0.0;
    if constexpr (KIND == BMI_LAPLACE_SL) {
      e.vr = (a.W * b.W) * (0.25 * M_1_PI) * ri;
    } else if constexpr (CPLX) {
      // exp(-i kappa r) / (4 pi r), kappa = kre + i kim (Helmholtz/SingleLayerOperator.hpp:115-120)
      double sn, cs;
      sincos_phase(prm.kre * r, &sn, &cs);
      const double damp = prm.kim != 0.0 ? exp(prm.kim * r) : 1.0;
      const double mag = damp * (a.W * b.W) * (0.25 * M_1_PI) * ri;
      const double kr = mag * cs, ki = -mag * sn;
      if constexpr (MAXW) {
        // vector part K w w (t_rc(a) . t_cc(b)), divergence part -K w w / (kappa^2 h^2)
        // (Maxwell/SingleLayerOperator.hpp:44-88)
        const double* ta = a.t + 3 * rc;
        const double* tb = b.t + 3 * cc;
        const double dt = ta[0] * tb[0] + ta[1] * tb[1] + ta[2] * tb[2];
        e.vr = kr * dt, e.vi = ki * dt;
        e.qr = kr * prm.qre - ki * prm.qim, e.qi = kr * prm.qim + ki * prm.qre;
      } else {
        e.vr = kr, e.vi = ki;
      }
    } else {
      e.vr = dummy_value(prm.dummy_fn, a, b) * a.W * b.W;
    }
    if (!valid) e.vr = 0.0, e.vi = 0.0, e.qr = 0.0, e.qi = 0.0;
    if constexpr (MAXW) {
      bernstein_basis_der<P>(a.s0, e.X, e.DX);
      bernstein_basis_der<P>(a.s1, e.Y, e.DY);
      bernstein_basis_der<P>(b.s0, e.U, e.DU);
      bernstein_basis_der<P>(b.s1, e.V, e.DV);
    } else {
      bernstein_basis<P>(a.s0, e.X);
      bernstein_basis<P>(a.s1, e.Y);
      bernstein_basis<P>(b.s0, e.U);
      bernstein_basis<P>(b.s1, e.V);
    }
    return e;
  }

  // the evaluation held by lane `src` of the wave
  __device__ __forceinline__ static Eval fetch(const Eval& e, int src) {
    Eval o;
    o.vr = __shfl(e.vr, src, 64);
    if constexpr (CPLX) o.vi = __shfl(e.vi, src, 64);
    if constexpr (MAXW) o.qr = __shfl(e.qr, src, 64), o.qi = __shfl(e.qi, src, 64);
#pragma unroll
    for (int k = 0; k < I; ++k) {
      o.X[k] = __shfl(e.X[k], src, 64), o.Y[k] = __shfl(e.Y[k], src, 64);
      o.U[k] = __shfl(e.U[k], src, 64), o.V[k] = __shfl(e.V[k], src, 64);
      if constexpr (MAXW) {
        o.DX[k] = __shfl(e.DX[k], src, 64), o.DY[k] = __shfl(e.DY[k], src, 64);
        o.DU[k] = __shfl(e.DU[k], src, 64), o.DV[k] = __shfl(e.DV[k], src, 64);
      }
    }
    return o;
  }

  // add one evaluation to this lane's part of the block
  __device__ __forceinline__ void accumulate(const Eval& e, int role, int rc, int cc) {
    const int part = CPLX ? (role & 1) : 0;
    const int half = CPLX ? (role >> 1) : role;
    double bv[I2], bd[MAXW ? I2 : 1], av[I2], ad[MAXW ? I2 : 1];
#pragma unroll
    for (int jy = 0; jy < I; ++jy)
#pragma unroll
      for (int jx = 0; jx < I; ++jx) {
        bv[jy * I + jx] = e.U[jx] * e.V[jy];
        if constexpr (MAXW) bd[jy * I + jx] = cc == 0 ? e.DU[jx] * e.V[jy] : e.U[jx] * e.DV[jy];
      }
#pragma unroll
    for (int iy = 0; iy < I; ++iy)
#pragma unroll
      for (int ix = 0; ix < I; ++ix) {
        av[iy * I + ix] = e.X[ix] * e.Y[iy];
        if constexpr (MAXW) ad[iy * I + ix] = rc == 0 ? e.DX[ix] * e.Y[iy] : e.X[ix] * e.DY[iy];
      }
    const double s = part ? e.vi : e.vr;
    const double q = part ? e.qi : e.qr;
#pragma unroll
    for (int ii = 0; ii < NR; ++ii) {
      // row ii of this lane's half (rows past the end hold zero)
      constexpr int dummy = 0;
      (void)dummy;
      double ar = av[ii], dr = MAXW ? ad[ii < (MAXW ? I2 : 1) ? ii : 0] : 0.0;
      if constexpr (RH == 2) {
        const bool in = NR + ii < I2;
        const double ah = in ? av[in ? NR + ii : 0] : 0.0;
        ar = half ? ah : ar;
        if constexpr (MAXW) {
          const double dh = in ? ad[in ? NR + ii : 0] : 0.0;
          dr = half ? dh : dr;
        }
      }
      const double as = s * ar;
      const double aq = MAXW ? q * dr : 0.0;
#pragma unroll
      for (int j = 0; j < I2; ++j) {
        if constexpr (MAXW)
          acc[ii * I2 + j] += as * bv[j] + aq * bd[j];
        else
          acc[ii * I2 + j] += as * bv[j];
      }
    }
  }

  // the lane's own evaluation and those of the other lanes of its group, in role order (all
  // lanes of the wave must call this together)
  __device__ __forceinline__ void add(const Pt<KIND>& a, const Pt<KIND>& b, const NFParams& prm, int rc, int cc,
                                      bool valid, int lane) {
    const Eval e = eval(a, b, prm, rc, cc, valid);
    if constexpr (G == 1) {
      accumulate(e, 0, rc, cc);
    } else {
      const int role = lane & (G - 1), base = lane & ~(G - 1);
#pragma unroll 1
      for (int r = 0; r < G; ++r) accumulate(fetch(e, base + r), role, rc, cc);
    }
  }

  // output slot of accumulator k of a lane with this role (complex blocks store all real parts,
  // then all imaginary parts); -1 if unused
  __device__ __forceinline__ static int slot(int role, int k) {
    const int part = CPLX ? (role & 1) : 0;
    const int half = CPLX ? (role >> 1) : role;
    const int row = half * NR + k / I2;
    return row < I2 ? part * I2 * I2 + row * I2 + k % I2 : -1;
  }
};

// Duffy rules reuse surface points: some points of the edge rule depend on the outer index i and
// one coordinate of the inner index j only, and the inner points of the vertex rule on the outer
// first coordinate and j only.  Those points are tabulated in LDS for a chunk of outer indices and
// the (i, j) work of the chunk is spread over the workgroup.  The chunk is the smallest number of
// outer indices that keeps at least 90 % of the lanes busy (or the best one that fits).
__host__ __device__ constexpr int pick_chunk(int items_per_unit, int nt, int max_units) {
  int best = 1;
  int best_num = 0, best_den = 1;
  for (int c = 1; c <= max_units; ++c) {
    const int items = c * items_per_unit;
    const int slots = ((items + nt - 1) / nt) * nt;
    if (10 * items >= 9 * slots) return c;
    if (items * best_den > best_num * slots) best = c, best_num = items, best_den = slots;
  }
  return best;
}
// LDS for the point tables (bytes), shared by the launch and the kernel
constexpr int DUFFY_TABLE_BYTES = 48 * 1024;
template <class PtK>
__host__ __device__ constexpr int edge_chunk(int n, int nt) {
  const int cap = DUFFY_TABLE_BYTES / (8 * n * static_cast<int>(sizeof(PtK)));
  const int mx = cap < n * n ? cap : n * n;
  return pick_chunk(n * n, nt, mx > 0 ? mx : 1);
}
template <class PtK>
__host__ __device__ constexpr int vertex_chunk(int n, int nt) {
  const int cap = DUFFY_TABLE_BYTES / (2 * n * n * static_cast<int>(sizeof(PtK)));
  const int mx = cap < n ? cap : n;
  return pick_chunk(n * n * n, nt, mx > 0 ? mx : 1);
}

// Coordinate lines of an element (edge and identical rules, scalar operators): with one coordinate
// fixed the four homogeneous coordinates and their derivatives across the line are polynomials of
// degree PD - 1 in the other: L[4 a + k] and L[4 PD + 4 a + k], a the power of the moving coordinate.
template <int PD>
__device__ __forceinline__ void line_contract(PolyPtr G, bool fix_u, double f, double* L) {
  const Powers<PD> q(f - 0.5);
#pragma unroll
  for (int a = 0; a < PD; ++a)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      q.sum([&](int b) { return fix_u ? G[(b * PD + a) * 4 + k] : G[(a * PD + b) * 4 + k]; }, L[4 * a + k],
            L[4 * PD + 4 * a + k]);
}

// A point of a contracted line.  The surface measure stays split as sqrt(cc) m, m with the weight: the
// kernel takes sqrt(cc / |x - y|^2) by one reciprocal square root of the product.  cc is scaled by
// NFParams::ms: the product of two of them and |x - y|^2 would else leave the range of a double
// where lengths do by the power of ten.
struct LinePt {
  double x0, x1, x2, cc, m, s0, s1;
};

// the smallest cc |x - y|^2 whose root is taken: a vanishing measure of either point (an element without
// area) then gives cc times a finite number, zero, and not 0 / 0
constexpr double MIN_CCS = 1e-300;

template <int PD, int KIND>
__device__ __forceinline__ LinePt line_point(const double* L, const NFParams& prm, bool fix_u, double u, double v,
                                             double w) {
  const double t = (fix_u ? v : u) - 0.5;
  double p[4], d1[4], d2[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    p[k] = L[4 * (PD - 1) + k], d1[k] = L[4 * PD + 4 * (PD - 1) + k], d2[k] = p[k];
#pragma unroll
    for (int a = PD - 2; a >= 0; --a) {
      if (a < PD - 2) d2[k] = fma(d2[k], t, p[k]);     // along the line
      p[k] = fma(p[k], t, L[4 * a + k]);
      d1[k] = fma(d1[k], t, L[4 * PD + 4 * a + k]);  // across the line (the fixed direction)
    }
  }
  const double bot = rcp_newton(p[3]);
  double X[3], E1[3], E2[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    X[k] = p[k] * bot;
    E1[k] = fma(-X[k], d1[3], d1[k]);
    E2[k] = fma(-X[k], d2[3], d2[k]);
  }
  LinePt q;
  q.x0 = X[0], q.x1 = X[1], q.x2 = X[2];
  q.s0 = u, q.s1 = v;
  if constexpr (KIND == BMI_DUMMY) {
    q.cc = 1.0, q.m = w;
  } else {
    q.cc = cross_square(E1, E2) * prm.ms, q.m = (bot * bot) * (prm.mr * w);
  }
  return q;
}

// N points of one line in LDS at moving coordinates t (weights one, local coordinates unset), each
// coefficient read once
template <int PD, int KIND, int N>
__device__ __forceinline__ void line_points(const double* L, const NFParams& prm, const double* t, LinePt* q) {
  double p[N][4], d1[N][4], d2[N][4];
#pragma unroll
  for (int k = 3; k >= 0; --k) {
    const double c = L[4 * (PD - 1) + k], d = L[4 * PD + 4 * (PD - 1) + k];
#pragma unroll
    for (int m = 0; m < N; ++m) p[m][k] = c, d1[m][k] = d, d2[m][k] = c;
#pragma unroll
    for (int a = PD - 2; a >= 0; --a) {
      const double ca = L[4 * a + k], da = L[4 * PD + 4 * a + k];
#pragma unroll
      for (int m = 0; m < N; ++m) {
        if (a < PD - 2) d2[m][k] = fma(d2[m][k], t[m] - 0.5, p[m][k]);
        p[m][k] = fma(p[m][k], t[m] - 0.5, ca);
        d1[m][k] = fma(d1[m][k], t[m] - 0.5, da);
      }
    }
    // keeps the coefficients of at most two coordinates in registers
    if (k == 2) __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int m = 0; m < N; ++m) {
    const double bot = rcp_newton(p[m][3]);
    double X[3], E1[3], E2[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      X[k] = p[m][k] * bot;
      E1[k] = fma(-X[k], d1[m][3], d1[m][k]);
      E2[k] = fma(-X[k], d2[m][3], d2[m][k]);
    }
    q[m].x0 = X[0], q[m].x1 = X[1], q[m].x2 = X[2];
    q[m].cc = cross_square(E1, E2) * prm.ms, q[m].m = (bot * bot) * prm.mr;
    // computed here: moved behind the branches of the phases, the points would keep both lines'
    // coefficients in registers
    asm volatile("" : "+v"(q[m].x0), "+v"(q[m].x1), "+v"(q[m].x2), "+v"(q[m].cc), "+v"(q[m].m));
  }
}

// Factorised vertex rule (scalar operators): a lane fixes one outer point and sums
// kernel x basis vector of the varying point over (its share of) the inner index, then adds the
// outer product with the fixed point's basis vector to its block: (P+1)^2 multiply-adds per
// evaluation instead of (P+1)^4.  A shape is the chunk of outer indices staged per LDS table
// and the number of lanes that split one outer point's inner range (even for complex
// operators, whose lane pairs hold the real and imaginary parts of the block).  The score
// trades busy lanes against the outer products, which every lane of an outer point repeats.
struct FactorShape {
  int chunk, lanes;
};
__host__ __device__ constexpr FactorShape factor_shape(int outer_per_chunk, int max_chunk, int nt, int g,
                                                       int eval_cost) {
  FactorShape best{1, g};
  long best_score = -1;
  for (int c = 1; c <= max_chunk; ++c) {
    const int units = c * outer_per_chunk;
    int S = nt / units;
    S -= S % g;  // whole lane groups per unit
    if (S < g) break;
    const long score = static_cast<long>(units) * S * 1000 / (eval_cost + S);
    if (score > best_score) best_score = score, best = FactorShape{c, S};
  }
  return best;
}
// vertex rule: chunks of first outer coordinates (n outer points each), inner range n^2
__host__ __device__ constexpr FactorShape vertex_shape(int n, int nt, int ptsize, int g) {
  const int cap = DUFFY_TABLE_BYTES / (2 * n * n * ptsize);
  return factor_shape(n, cap < n ? (cap > 0 ? cap : 1) : n, nt, g, 90);
}
// doubles between lines in LDS (16 bytes beyond a whole number of 64-byte rows: lanes on neighbouring
// lines read different banks)
__host__ __device__ constexpr int line_stride(int pd) { return 8 * pd + 2; }
// edge rule, factorised: chunks of outer indices i (n units (i, j0) each, S lanes per unit sharing the n
// inner indices).  A lane's work per chunk, in instructions counted from the compiled code: 3,260 per unit
// (contracted lines, fixed points, vectors, tables) and 630 per inner index
__host__ __device__ constexpr FactorShape edge_shape(int n, int nt, int ptsize) {
  const int cap = DUFFY_TABLE_BYTES / (2 * n * ptsize);
  FactorShape best{1, 1};
  long best_cost = -1;
  for (int S = 1; S <= n; ++S) {
    int c = nt / (S * n);
    if (c > cap) c = cap;
    if (c > n * n) c = n * n;
    if (c < 1) break;
    const long cost = static_cast<long>((n * n + c - 1) / c) * (3260 + static_cast<long>((n + S - 1) / S) * 630);
    if (best_cost < 0 || cost < best_cost) best_cost = cost, best = FactorShape{c, S};
  }
  return best;
}

// kernel times both point weights, (kr, ki): the scalar integrands of eval() without the basis
template <int KIND>
__device__ __forceinline__ void kernel_ww(const Pt<KIND>& a, const Pt<KIND>& b, const NFParams& prm, double& kr,
                                          double& ki) {
  const double d0 = a.x0 - b.x0, d1 = a.x1 - b.x1, d2 = a.x2 - b.x2;
  const double s = d0 * d0 + d1 * d1 + d2 * d2;
  const double ri = rsqrt_newton(s);  // 1 / r
  if constexpr (KIND == BMI_LAPLACE_SL) {
    kr = (a.W * b.W) * (0.25 * M_1_PI) * ri, ki = 0.0;
  } else if constexpr (KIND == BMI_HELMHOLTZ_SL) {
    const double r = s * ri;
    double sn, cs;
    sincos_phase(prm.kre * r, &sn, &cs);
    const double damp = prm.kim != 0.0 ? exp(prm.kim * r) : 1.0;
    const double mag = damp * (a.W * b.W) * (0.25 * M_1_PI) * ri;
    kr = mag * cs, ki = -mag * sn;
  } else {
    kr = dummy_value(prm.dummy_fn, a, b) * a.W * b.W, ki = 0.0;
  }
}

// the same with the second point (or both) on a contracted line
template <int KIND>
__device__ __forceinline__ void kernel_scaled(double d0, double d1, double d2, double cc, double f, const NFParams& prm,
                                              double& kr, double& ki) {
  // f sqrt(cc) exp(-i kappa r) / (4 pi r)
  const double s = d0 * d0 + d1 * d1 + d2 * d2;
  const double mag = (f * (0.25 * M_1_PI)) * (cc * rsqrt_newton(fmax(cc * s, MIN_CCS)));
  if constexpr (KIND == BMI_LAPLACE_SL) {
    kr = mag, ki = 0.0;
  } else {
    const double r = s * rsqrt_newton(s);
    double sn, cs;
    sincos_phase(prm.kre * r, &sn, &cs);
    const double a = prm.kim != 0.0 ? mag * exp(prm.kim * r) : mag;
    kr = a * cs, ki = -a * sn;
  }
}
template <int KIND>
__device__ __forceinline__ void kernel_ww(const Pt<KIND>& a, const LinePt& b, const NFParams& prm, double& kr,
                                          double& ki) {
  if constexpr (KIND == BMI_DUMMY)
    kr = dummy_value(prm.dummy_fn, a, b) * a.W * b.m, ki = 0.0;
  else
    kernel_scaled<KIND>(a.x0 - b.x0, a.x1 - b.x1, a.x2 - b.x2, b.cc, a.W * b.m, prm, kr, ki);
}
template <int KIND>
__device__ __forceinline__ void kernel_ww(const LinePt& a, const Pt<KIND>& b, const NFParams& prm, double& kr,
                                          double& ki) {
  if constexpr (KIND == BMI_DUMMY)
    kr = dummy_value(prm.dummy_fn, a, b) * a.m * b.W, ki = 0.0;
  else
    kernel_scaled<KIND>(a.x0 - b.x0, a.x1 - b.x1, a.x2 - b.x2, a.cc, a.m * b.W, prm, kr, ki);
}
template <int KIND>
__device__ __forceinline__ void kernel_ww(const LinePt& a, const LinePt& b, const NFParams& prm, double& kr,
                                          double& ki) {
  if constexpr (KIND == BMI_DUMMY)
    kr = dummy_value(prm.dummy_fn, a, b) * a.m * b.m, ki = 0.0;
  else
    kernel_scaled<KIND>(a.x0 - b.x0, a.x1 - b.x1, a.x2 - b.x2, a.cc * b.cc, a.m * b.m, prm, kr, ki);
}

// the value of the lane's neighbour (lane ^ 1)
__device__ __forceinline__ double neighbour(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);  // quad permute 1, 0, 3, 2
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// lane-private sum of (kernel x basis vector) over inner points
template <int P, bool CPLX>
struct VecSum {
  static constexpr int I = P + 1, I2 = I * I;
  double r[I2], i[CPLX ? I2 : 1];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int k = 0; k < I2; ++k) {
      r[k] = 0.0;
      if constexpr (CPLX) i[k] = 0.0;
    }
  }
  // += (kr + i ki) * basis(s0, s1)
  __device__ __forceinline__ void add(double kr, double ki, double s0, double s1) {
    double X[I], Y[I];
    bernstein_basis<P>(s0, X);
    bernstein_basis<P>(s1, Y);
#pragma unroll
    for (int iy = 0; iy < I; ++iy)
#pragma unroll
      for (int ix = 0; ix < I; ++ix) {
        const double b = X[ix] * Y[iy];
        r[iy * I + ix] += kr * b;
        if constexpr (CPLX) i[iy * I + ix] += ki * b;
      }
  }
  // the vector summed over the two lanes of this lane's group (each holds a share of the inner
  // range): real parts, or for complex vectors the part of this lane's role (0 real, 1 imaginary);
  // all lanes must call this together
  __device__ __forceinline__ void total(int role, double* w) const {
#pragma unroll
    for (int k = 0; k < I2; ++k) {
      if constexpr (CPLX) {
        // hand the neighbour the part it keeps
        const double give = (role & 1) ? r[k] : i[k], keep = (role & 1) ? i[k] : r[k];
        w[k] = keep + neighbour(give);
      } else {
        w[k] = r[k] + neighbour(r[k]);
      }
    }
  }
};

// D(i, j) of v_mfma_f64_16x16x4f64 on lane j + 16 (i mod 4), element i / 4
typedef double nf_d4 __attribute__((ext_vector_type(4)));

// Sums of outer products on the matrix cores: every lane pair of a wave contributes row vector x column
// vector, (P+1)^2 entries each; the pairs put them in the wave's own part of LDS (three arrays of 32
// vectors: fixed, real, imaginary) and eight 16x16x4 steps add the 32 products to the wave's block.  The
// block takes 8 registers (16 complex) instead of a share of it per lane (90 and 162 for P = 2), which
// kept the rules at one wave per SIMD.  The 32 products have a sum of their own (one part of a complex block
// after the other: the registers of one): thousands of terms in one running sum rounded the blocks to 4.5e-16
// where the points leave 1.6e-16 (identical rule, 6,144 elements, P 2).
template <int I2>
__host__ __device__ constexpr int stage_doubles(bool cplx) {
  return 32 * (cplx ? 3 : 2) * I2;
}
// LDS operations of a wave are in order; the fences keep the compiler's order as well
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int I2, bool CPLX, bool COLS>
__device__ __forceinline__ void add_products(const double* stage, int lane, nf_d4& dr, nf_d4& di) {
  const int li = lane & 15, lk = lane >> 4, row = li < I2 ? li : I2 - 1;  // entries past the block are not read back
#pragma unroll
  for (int part = 0; part < (CPLX ? 2 : 1); ++part) {
    nf_d4 d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const int m = (4 * st + lk) * I2 + row;
      const double f = stage[m], v = stage[(part + 1) * 32 * I2 + m];
      d = __builtin_amdgcn_mfma_f64_16x16x4f64(COLS ? f : v, COLS ? v : f, d, 0, 0, 0);
    }
    if (part == 0)
      dr += d;
    else
      di += d;
  }
}

// One sub-region of the edge rule: the fixed point F against the inner points inner(j) for j = sub,
// sub + S, ... < count, which differ in one local coordinate only (FIX0: s0 is the same for all), so
// the sum over them needs the P + 1 basis values of the moving coordinate and the other direction's
// values multiply the sum.  COLS: F supplies the rows (element 1) and the inner points the columns;
// otherwise the inner points supply the rows.  Adds the outer product of F's basis with the summed
// vector to the wave's block.  All lanes of the wave must call this together.
template <int P, int KIND, bool COLS, bool FIX0, class PtF, class Inner>
__device__ __forceinline__ void line_pass(nf_d4& dr, nf_d4& di, double* stage, const PtF& F, int lane, bool act,
                                          int sub, int S, int count, const NFParams& prm, double fixed, Inner inner) {
  constexpr int I = P + 1, I2 = I * I;
  constexpr bool CPLX = KIND == BMI_HELMHOLTZ_SL;
  double ur[I], ui[I];
#pragma unroll
  for (int k = 0; k < I; ++k) ur[k] = 0.0, ui[k] = 0.0;
  if (act) {
#pragma unroll 1
    for (int j = sub; j < count; j += S) {
      const auto b = inner(j);
      double kr, ki, B[I];
      if constexpr (COLS)
        kernel_ww<KIND>(F, b, prm, kr, ki);
      else
        kernel_ww<KIND>(b, F, prm, kr, ki);
      bernstein_basis<P>(FIX0 ? b.s1 : b.s0, B);
#pragma unroll
      for (int k = 0; k < I; ++k) {
        ur[k] += kr * B[k];
        if constexpr (CPLX) ui[k] += ki * B[k];
      }
    }
  }
  double Bf[I], X[I], Y[I];
  bernstein_basis<P>(fixed, Bf);
  bernstein_basis<P>(F.s0, X);
  bernstein_basis<P>(F.s1, Y);
  // 32 lanes' vectors at a time (inactive lanes contribute zero)
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if ((lane >> 5) == half) {
      const int m = (lane & 31) * I2;
#pragma unroll
      for (int k = 0; k < I2; ++k) {
        const double g = Bf[FIX0 ? k % I : k / I];
        const int o = FIX0 ? k / I : k % I;
        stage[m + k] = act ? X[k % I] * Y[k / I] : 0.0;
        stage[32 * I2 + m + k] = act ? g * ur[o] : 0.0;
        if constexpr (CPLX) stage[64 * I2 + m + k] = act ? g * ui[o] : 0.0;
      }
    }
    wave_fence();
    add_products<I2, CPLX, COLS>(stage, lane, dr, di);
    wave_fence();
  }
}

// One factorised sub-region: the fixed point F against the inner points inner(j) for j = sub,
// sub + S, ... < count.  COLS: F supplies the rows (element 1) and the inner points the columns;
// otherwise the inner points supply the rows.  Adds the outer product of F's basis with the
// summed vector to this lane's part of the block.  All lanes of the wave must call this
// together (the lane pairs of complex operators exchange their sums).
template <int P, int KIND, bool COLS, class Acc, class PtK, class Inner>
__device__ __forceinline__ void factor_pass(Acc& acc, const PtK& F, int role, bool act, int sub, int S, int count,
                                            const NFParams& prm, Inner inner) {
  constexpr int I = P + 1, I2 = I * I;
  VecSum<P, Acc::CPLX> u;
  u.zero();
  if (act) {
#pragma unroll 1
    for (int j = sub; j < count; j += S) {
      const PtK b = inner(j);
      double kr, ki;
      if constexpr (COLS)
        kernel_ww<KIND>(F, b, prm, kr, ki);
      else
        kernel_ww<KIND>(b, F, prm, kr, ki);
      u.add(kr, ki, b.s0, b.s1);
    }
  }
  double w[I2];
  u.total(role, w);
  if (!act) return;
  double X[I], Y[I];
  bernstein_basis<P>(F.s0, X);
  bernstein_basis<P>(F.s1, Y);
  double f[I2];
#pragma unroll
  for (int iy = 0; iy < I; ++iy)
#pragma unroll
    for (int ix = 0; ix < I; ++ix) f[iy * I + ix] = X[ix] * Y[iy];
  // this lane's rows: half (role bit above the real/imaginary bit) x NR .. + NR
  const int half = Acc::RH == 2 ? (Acc::CPLX ? (role >> 1) : role) : 0;
#pragma unroll
  for (int ii = 0; ii < Acc::NR; ++ii) {
    const int row = half * Acc::NR + ii;
    const bool in = Acc::RH == 1 || row < I2;
    const int rr = in ? row : 0;
    // COLS: F's basis gives the rows; otherwise the summed vector does
    const double a = in ? (COLS ? f[rr] : w[rr]) : 0.0;
#pragma unroll
    for (int k = 0; k < I2; ++k) acc.acc[ii * I2 + k] += a * (COLS ? w[k] : f[k]);
  }
}

// f(std::integral_constant<int, r>()) for a rotation r that is uniform in the workgroup: the
// callee's tau and line evaluations then fold the rotation at compile time
template <class F>
__device__ __forceinline__ void with_rotation(int r, F&& f) {
  switch (r) {
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    default: f(std::integral_constant<int, 0>()); break;
  }
}

// DuffyTrick::tau (DuffyTrick/tau.hpp:26-42)
__device__ __forceinline__ void tau(double x, double y, int c, double& u, double& v) {
  switch (c) {
    case 1: u = 1 - y, v = x; return;
    case 2: u = 1 - x, v = 1 - y; return;
    case 3: u = y, v = 1 - x; return;
    default: u = x, v = y; return;
  }
}

// sum the per-lane partial blocks over the workgroup: lanes of equal role within each wave by
// shuffles, then the waves through LDS; the result is the full block in `sum` (Acc::TOT values)
template <int NT, class Acc>
__device__ __forceinline__ void reduce_block(Acc& acc, double* lds, int tid, double* sum) {
  constexpr int N = Acc::NR * Acc::I2;
  constexpr int TOT = Acc::TOT;
  constexpr int NW = NT / 64;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double v = acc.acc[k];
#pragma unroll
    for (int off = 32; off >= Acc::G; off >>= 1) v += __shfl_xor(v, off, 64);
    acc.acc[k] = v;
  }
  const int wave = tid >> 6, lane = tid & 63;
  if (lane < Acc::G) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int sl = Acc::slot(lane, k);
      if (sl >= 0) lds[wave * TOT + sl] = acc.acc[k];
    }
  }
  __syncthreads();
  for (int k = tid; k < TOT; k += NT) {
    double v = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += lds[w * TOT + k];
    sum[k] = v;
  }
  __syncthreads();
}

// the waves' blocks in LDS: entry (row, column) of part p (0 real, 1 imaginary) of wave w at
// lds[(w * parts + p) * I2^2 + row * I2 + column]; the caller has passed a barrier since lds was last used
template <int I2, bool CPLX>
__device__ __forceinline__ void spread_blocks(double* lds, int wave, int lane, const nf_d4& dr, const nf_d4& di) {
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int row = 4 * v + lk;
    if (row < I2 && li < I2) {
      lds[(wave * (CPLX ? 2 : 1)) * I2 * I2 + row * I2 + li] = dr[v];
      if constexpr (CPLX) lds[(wave * 2 + 1) * I2 * I2 + row * I2 + li] = di[v];
    }
  }
  __syncthreads();
}

// identical rule: outer coordinates xi0 whose lines are staged together: the chunk with the fewest
// rounds of 128 units, within LDS for two workgroups per CU
__host__ __device__ constexpr int identical_chunk(int n, int pd) {
  const int cap = 52 * 1024 / (4 * n * line_stride(pd) * 8);
  int best = 1, best_rounds = 1 << 30;
  for (int c = 1; c <= (cap < n ? cap : n); ++c) {
    const int rounds = n / c * ((c * n * n + 127) / 128) + (n % c * n * n + 127) / 128;
    if (rounds < best_rounds) best = c, best_rounds = rounds;
  }
  return best;
}

// waves per SIMD asked of the compiler: two for the scalar rules whose points lie on contracted lines
// (the latencies of one wave covered by the other; the Helmholtz vertex rule, whose lanes hold half a
// block each, spills at two waves: 48 -> 55 ms)
__host__ __device__ constexpr int nf_waves(int kind, int cls) {
  return (kind == BMI_LAPLACE_SL || kind == BMI_HELMHOLTZ_SL) && (cls == 2 || cls == 3) ? 2 : 1;
}

template <int P, int KIND, int PD, int CLS, int NT>
__global__ __launch_bounds__(NT, nf_waves(KIND, CLS)) void k_nearfield(const NFPair* __restrict__ pairs, NFParams prm) {
  extern __shared__ double lds[];
  using Acc = BlockAcc<P, KIND>;
  constexpr int I2 = Acc::I2;
  const NFPair pr = pairs[blockIdx.x];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const PolyPtr g1 = (PolyPtr)(prm.poly + static_cast<int64_t>(pr.e1) * prm.poly_stride);
  const PolyPtr g2 = (PolyPtr)(prm.poly + static_cast<int64_t>(pr.e2) * prm.poly_stride);
  // points are about the centre of their element; of two elements' points the one of the outer loop is moved
  const Shift sh{g1 + prm.poly_stride - 4, g2 + prm.poly_stride - 4};
  const double h = prm.h;
  const int n = pr.deg + 1;
  const int nq = n * n;
  const double* gx = c_gl_nodes + c_gl_offset[n - 1];
  const double* gw = c_gl_weights + c_gl_offset[n - 1];
  using PtK = Pt<KIND>;
  // Maxwell component block of this workgroup (0 for the scalar operators)
  const int rc = KIND == BMI_MAXWELL_SL ? static_cast<int>(blockIdx.y) >> 1 : 0;
  const int cc = KIND == BMI_MAXWELL_SL ? static_cast<int>(blockIdx.y) & 1 : 0;
  Acc acc;
  acc.zero();
  double aval = 0.0;  // the block entry a thread owns (factorised identical and regular rules)
  constexpr bool IDENT = KIND == BMI_LAPLACE_SL || KIND == BMI_HELMHOLTZ_SL;  // factorised identical rule
  nf_d4 dr{0.0, 0.0, 0.0, 0.0}, di{0.0, 0.0, 0.0, 0.0};  // sums over units on the matrix cores
  // every lane runs the same number of iterations (lane groups swap values); lanes past the end
  // evaluate a valid point with zero weight

  if constexpr (CLS == 0) {
    // integrate0: far-field tables of both elements
    const int nf = prm.nff, fs = prm.ffs;
    const double* f1 = prm.ffield + static_cast<int64_t>(pr.e1) * nf * fs;
    const double* f2 = prm.ffield + static_cast<int64_t>(pr.e2) * nf * fs;
    const int total = nf * nf;
    for (int base = 0; base < total; base += NT) {
      const bool valid = base + tid < total;
      const int idx = valid ? base + tid : total - 1;
      const int i = idx / nf, j = idx - (idx / nf) * nf;
      const double* a = f1 + i * fs;
      const double* b = f2 + j * fs;
      constexpr bool PLAIN_W = KIND == BMI_DUMMY || KIND == BMI_MAXWELL_SL;
      PtK pa, pb;
      pa.x0 = a[0], pa.x1 = a[1], pa.x2 = a[2], pa.W = PLAIN_W ? a[4] : a[3] * a[4], pa.s0 = a[5], pa.s1 = a[6];
      pb.x0 = b[0], pb.x1 = b[1], pb.x2 = b[2], pb.W = PLAIN_W ? b[4] : b[3] * b[4], pb.s0 = b[5], pb.s1 = b[6];
      if constexpr (KIND == BMI_MAXWELL_SL) {
#pragma unroll
        for (int k = 0; k < 6; ++k) pa.t[k] = a[8 + k], pb.t[k] = b[8 + k];
      }
      acc.add(pa, pb, prm, rc, cc, valid, lane);
    }
  } else if constexpr (CLS == 1 && !Acc::MAXW) {
    // integrate1, factorised: surface points of both elements staged in LDS; S lanes share a
    // point of element 1 and each sums kernel x basis vector over its share of the points of
    // element 2.  The lanes' vectors and the outer points' basis values go to LDS, and every
    // thread adds the outer products into the one block entry it owns (no per-lane block, no
    // workgroup reduction).
    constexpr bool CPLX = Acc::CPLX;
    constexpr int I = P + 1;
    constexpr int VR = CPLX ? 2 * I2 : I2;  // doubles of one lane's vector
    constexpr int NE = Acc::TOT;
    static_assert(NE <= NT, "at most one block entry per thread");
    PtK* q1 = reinterpret_cast<PtK*>(lds);
    PtK* q2 = q1 + nq;
    double* rec = reinterpret_cast<double*>(q2 + nq);  // NT vectors
    double* bas = rec + NT * VR;                       // basis products of the round's outer points
    for (int k = tid; k < nq; k += NT) {
      const double u = gx[k / n], v = gx[k % n], w = h * (gw[k / n] * gw[k % n]);
      q1[k] = make_point<PD, KIND>(g1, prm, u, v, w);
      q2[k] = make_point<PD, KIND>(g2, prm, u, v, w);
    }
    __syncthreads();
    const int S = NT / nq > 1 ? NT / nq : 1;
    const int per_round = NT / S;
    const int epart = tid / (I2 * I2), erem = tid - epart * (I2 * I2);
    const int erow = erem / I2, ecol = erem - erow * I2;
    for (int u0 = 0; u0 < nq; u0 += per_round) {
      const int unit = u0 + tid / S, sub = tid - (tid / S) * S;
      const bool act = tid / S < per_round && unit < nq;
      VecSum<P, CPLX> vs;
      vs.zero();
      if (act) {
        const PtK F = sh.to_second(q1[unit]);
#pragma unroll 1
        for (int j = sub; j < nq; j += S) {
          const PtK b = q2[j];
          double kr, ki;
          kernel_ww<KIND>(F, b, prm, kr, ki);
          vs.add(kr, ki, b.s0, b.s1);
        }
        if (sub == 0) {
          double X[I], Y[I];
          bernstein_basis<P>(F.s0, X);
          bernstein_basis<P>(F.s1, Y);
#pragma unroll
          for (int iy = 0; iy < I; ++iy)
#pragma unroll
            for (int ix = 0; ix < I; ++ix) bas[(tid / S) * I2 + iy * I + ix] = X[ix] * Y[iy];
        }
      }
      double* r = rec + tid * VR;
#pragma unroll
      for (int k = 0; k < I2; ++k) {
        r[k] = vs.r[k];
        if constexpr (CPLX) r[I2 + k] = vs.i[k];
      }
      __syncthreads();
      if (tid < NE) {
        const int nu = nq - u0 < per_round ? nq - u0 : per_round;
        const int o = epart * I2 + ecol;
#pragma unroll 1
        for (int m = 0; m < nu; ++m) {
          double v = 0.0;
          for (int s2 = 0; s2 < S; ++s2) v += rec[(m * S + s2) * VR + o];
          aval += bas[m * I2 + erow] * v;
        }
      }
      __syncthreads();
    }
  } else if constexpr (CLS == 1) {
    // integrate1: tensor Gauss rule; surface points of both elements staged in LDS
    PtK* q1 = reinterpret_cast<PtK*>(lds);
    PtK* q2 = q1 + nq;
    for (int k = tid; k < nq; k += NT) {
      const double u = gx[k / n], v = gx[k % n], w = h * (gw[k / n] * gw[k % n]);
      q1[k] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, w));
      q2[k] = make_point<PD, KIND>(g2, prm, u, v, w);
    }
    __syncthreads();
    const int total = nq * nq;
    for (int base = 0; base < total; base += NT) {
      const bool valid = base + tid < total;
      const int idx = valid ? base + tid : total - 1;
      const int i = idx / nq, j = idx - (idx / nq) * nq;
      acc.add(q1[i], q2[j], prm, rc, cc, valid, lane);
    }
    __syncthreads();
  } else if constexpr (CLS == 2 && IDENT) {
    // integrate2, factorised (symmetric kernels).  The sub-simplex pairs of the unfactorised form
    // below are, with t1 = xj0 (1 - xi0), t3 = t1 + xi0 (outer unit (i, j0)) and t2 = xj1 (1 - xi0 xi1),
    // t4 = t2 + xi0 xi1 (inner index j1): (t1,t2)-(t3,t4), (t1,t4)-(t3,t2), (t2,t1)-(t4,t3),
    // (t2,t3)-(t4,t1).  For one unit the eight points lie on four coordinate lines of the patch
    // (s = t1, s = t3, t = t1, t = t3), which depend on xi0 and j0 only: the lines of a chunk of xi0
    // values are contracted into LDS (one line per thread) and serve every xi1.  The tensor basis
    // splits the block: with B(x) the Bernstein values, A((ix,iy),(jx,jy)) += B_ix(t1) B_jx(t3)
    // U01(iy,jy) + B_iy(t1) B_jy(t3) U23(ix,jx), U01 = sum over j1 of K0 B(t2) B(t4)^T + K1 B(t4) B(t2)^T
    // and U23 likewise with K2, K3 (the fourth pair taken in the other order, which the symmetric
    // kernel allows).  The rule adds every pair in both orders, so the block is A + A^T, formed when
    // it is written.
    // A lane holds a unit; even waves sum U01 over the s-lines, odd waves U23 over the t-lines.  Two j1 are
    // evaluated together, so each line coefficient read from LDS serves four points (with two the
    // LDS reads bound the rule: 55 ms for 24,576 elements).  The sums over the units are outer products
    // of two (P+1)^2 vectors with the units as the inner index: each wave puts 32 units' vectors at a
    // time in its own part of LDS and multiplies them on the matrix cores (eight 16x16x4 steps), so a
    // round of units needs no barrier and no block in registers.  Bound: FP64 VALU.
    constexpr bool CPLX = Acc::CPLX;
    constexpr int I = P + 1;
    constexpr int LST = line_stride(PD);
    constexpr int UPR = NT / 2;  // units per round
    static_assert(NT == 256, "four waves: two of 64 units each per direction");
    const int C = identical_chunk(n, PD);
    const int wv = tid >> 6, ln = tid & 63;
    const bool tl = (wv & 1) != 0;
    const int myu = (wv >> 1) * 64 + ln;
    double* stage = lds + C * 4 * n * LST + wv * stage_doubles<I2>(CPLX);
    for (int c0 = 0; c0 < n; c0 += C) {
      const int cn = n - c0 < C ? n - c0 : C;
      __syncthreads();  // the previous chunk's lines are no longer read
      for (int l = tid; l < cn * n * 4; l += NT) {
        // line q of (ci, j0) at (q * cn + ci) * n + j0: lanes on consecutive j0 read neighbouring lines
        const int q = l / (cn * n), r = l - q * (cn * n), ci = r / n, j0 = r - ci * n;
        const double xi0 = gx[c0 + ci];
        const double t1 = gx[j0] * (1 - xi0);
        double L[8 * PD];
        line_contract<PD>(g1, q < 2, (q & 1) ? t1 + xi0 : t1, L);
#pragma unroll
        for (int k = 0; k < 8 * PD; ++k) lds[l * LST + k] = L[k];
      }
      __syncthreads();
      const int units = cn * nq;
      for (int u0 = 0; u0 < units; u0 += UPR) {
        if (u0 + (wv >> 1) * 64 >= units) continue;  // no unit for this wave
        const bool act = u0 + myu < units;
        const int uc = act ? u0 + myu : 0;
        const int ci = uc / nq, rem = uc - ci * nq, i1 = rem / n, j0 = rem - i1 * n;
        const double xi0 = gx[c0 + ci], xi1 = gx[i1], x01 = xi0 * xi1;
        const double t1 = gx[j0] * (1 - xi0), t3 = t1 + xi0;
        double ur[I2], ui[CPLX ? I2 : 1];
#pragma unroll
        for (int k = 0; k < I2; ++k) {
          ur[k] = 0.0;
          if constexpr (CPLX) ui[k] = 0.0;
        }
        // s-lines: (t1,t2)-(t3,t4) and (t1,t4)-(t3,t2); t-lines: (t2,t1)-(t4,t3) and (t4,t1)-(t2,t3)
        // (the second pair in the other order); either way the first line holds the points at
        // (t2, t4) of the first member, the second line those of the second at (t4, t2)
        const double* L0 = lds + ((tl ? 2 * cn * n : 0) + ci * n + j0) * LST;
        const int L1 = cn * n * LST;
#pragma unroll 1
        for (int j1 = 0; j1 < n; j1 += 2) {
          const bool two = j1 + 1 < n;  // an odd rule ends with a repeated point of weight zero
          const double g0 = gx[j1], g1_ = gx[two ? j1 + 1 : j1], w0 = gw[j1], w1 = two ? gw[j1 + 1] : 0.0;
          const double t[4] = {g0 * (1 - x01), g0 * (1 - x01) + x01, g1_ * (1 - x01), g1_ * (1 - x01) + x01};
          // the lines are read again in every iteration, one at a time (an opaque offset keeps
          // the compiler from holding them in registers across the loop)
          int off = 0;
          asm volatile("" : "+v"(off));
          const double* Lq = L0 + off;
          LinePt a[4], b[4];
          line_points<PD, KIND, 4>(Lq, prm, t, a);
          __builtin_amdgcn_sched_barrier(0);
          line_points<PD, KIND, 4>(Lq + L1, prm, t, b);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            double B2[I], B4[I];
            bernstein_basis<P>(t[2 * h], B2);
            bernstein_basis<P>(t[2 * h + 1], B4);
            const double wj = h ? w1 : w0;
            // K0 B(t2) B(t4)^T, then K1 B(t4) B(t2)^T (one kernel evaluation's registers at a time)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
              double kr, ki;
              kernel_ww<KIND>(a[2 * h + m], b[2 * h + 1 - m], prm, kr, ki);
              kr *= wj, ki *= wj;
#pragma unroll
              for (int p = 0; p < I; ++p) {
                const double f = kr * (m ? B4[p] : B2[p]), fi = CPLX ? ki * (m ? B4[p] : B2[p]) : 0.0;
#pragma unroll
                for (int q = 0; q < I; ++q) {
                  ur[p * I + q] += f * (m ? B2[q] : B4[q]);
                  if constexpr (CPLX) ui[p * I + q] += fi * (m ? B2[q] : B4[q]);
                }
              }
              if constexpr (CPLX) __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
        double B1[I], B3[I];
        bernstein_basis<P>(t1, B1);
        bernstein_basis<P>(t3, B3);
        const double sc = act ? h * h * (gw[c0 + ci] * gw[i1]) * xi0 * (1 - xi0) * (1 - x01) * gw[j0] : 0.0;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          if ((ln >> 5) == half) {
            const int m = (ln & 31) * I2;
#pragma unroll
            for (int k = 0; k < I2; ++k) {
              stage[m + k] = sc * B1[k / I] * B3[k % I];
              stage[32 * I2 + m + k] = ur[k];
              if constexpr (CPLX) stage[64 * I2 + m + k] = ui[k];
            }
          }
          wave_fence();
          add_products<I2, CPLX, true>(stage, ln, dr, di);
          wave_fence();
        }
      }
    }
    __syncthreads();
    spread_blocks<I2, CPLX>(lds, wv, ln, dr, di);
    if (tid < Acc::TOT) {
      const int part = tid / (I2 * I2), rem = tid - part * (I2 * I2);
      const int ei = rem / I2, ej = rem - ei * I2;
      const int iy = ei / I, ix = ei - iy * I, jy = ej / I, jx = ej - jy * I;
      const int o01 = (ix * I + jx) * I2 + iy * I + jy, o23 = (iy * I + jy) * I2 + ix * I + jx;
      auto at = [&](int w, int o) { return lds[(w * (CPLX ? 2 : 1) + part) * I2 * I2 + o]; };
      aval = (at(0, o01) + at(2, o01)) + (at(1, o23) + at(3, o23));
    }
    __syncthreads();
  } else if constexpr (CLS == 2) {
    // integrate2: identical elements, 8 Duffy sub-simplices, symmetrised
    const int total = nq * nq;
    for (int base = 0; base < total; base += NT) {
      const bool valid = base + tid < total;
      const int idx = valid ? base + tid : total - 1;
      const int i = idx / nq, j = idx - (idx / nq) * nq;
      const double xi0 = gx[i / n], xi1 = gx[i % n], wi = gw[i / n] * gw[i % n];
      const double xj0 = gx[j / n], xj1 = gx[j % n], wj = gw[j / n] * gw[j % n];
      const double w = h * h * wi * xi0 * (1 - xi0) * (1 - xi0 * xi1);
      const double t1 = xj0 * (1 - xi0);
      const double t2 = xj1 * (1 - xi0 * xi1);
      const double t3 = t1 + xi0;
      const double t4 = t2 + xi0 * xi1;
      // point pairs (t1,t2)-(t3,t4), (t1,t4)-(t3,t2), (t2,t1)-(t4,t3), (t2,t3)-(t4,t1), written as
      // selects; the loop is unrolled only when the block accumulator leaves registers to spare
      constexpr int UNR2 = Acc::G == 1 ? 4 : 1;
#pragma unroll UNR2
      for (int k = 0; k < 4; ++k) {
        const bool sw = k >= 2, odd = k & 1;
        const double pu = sw ? t2 : t1, qu = sw ? t4 : t3;
        const double r = sw ? t1 : t2, sv = sw ? t3 : t4;
        const PtK a = make_point<PD, KIND>(g1, prm, pu, odd ? sv : r, w);
        const PtK b = make_point<PD, KIND>(g1, prm, qu, odd ? r : sv, wj);
        acc.add(a, b, prm, rc, cc, valid, lane);
        acc.add(b, a, prm, rc, cc, valid, lane);
      }
    }
  } else if constexpr (CLS == 3 && !Acc::MAXW) {
    // integrate3, factorised: the sub-regions and points of the unfactorised form below.  Unit (i, j0), inner
    // index j1.  g = 0: rows (t1, e0), columns (t2, e1); g = 1: rows (t3, xi1), columns on element 2 at
    // tau(t4 or 1 - t4, e1; r2); g = 2: rows on element 1 at tau(t4 or 1 - t4, e1; r1), columns (t3, xi1).
    // The weight products are split into the unit's factor (w and the j0 part of the inner weights)
    // and gw[j1].  What a unit needs of each point:
    // * (t4, e1) runs along a coordinate line over j1: one contraction per unit, held in registers, and
    //   a one-dimensional evaluation per j1;
    // * (t3, xi1) lies on the line of xi1: 2 n lines per element pair, contracted into LDS once;
    // * (t1, e0) once per unit, and (t2, e1) from a table per chunk of i, shared by the j0.
    // In every sub-region the inner points have one coordinate in common, so their sum is over P + 1
    // basis values (line_pass).  Bound: FP64 VALU, two waves per SIMD.
    const int r1 = pr.rot1, r2 = pr.rot2;
    constexpr bool CPLX = Acc::CPLX;
    constexpr int LST = line_stride(PD);
    const FactorShape shp = edge_shape(n, NT, static_cast<int>(sizeof(PtK)));
    const int CI = shp.chunk, S = shp.lanes;
    PtK* tab = reinterpret_cast<PtK*>(lds);  // (odd, ci, j1)
    double* lines = lds + (2 * CI * n * static_cast<int>(sizeof(PtK)) >> 3);  // (element, i1)
    double* stage = lines + 2 * n * LST + (tid >> 6) * stage_doubles<I2>(CPLX);
    // tau(x, y; r) with y fixed: the fixed and the moving local coordinate
    auto held = [](int r, double y) { return (r == 0 || r == 3) ? y : 1 - y; };
    auto moved = [](int r, double x) { return r < 2 ? x : 1 - x; };
    for (int l = tid; l < 2 * n; l += NT) {
      const int el = l / n, r = el ? r2 : r1;
      double L[8 * PD];
      line_contract<PD>(el ? g2 : g1, r & 1, held(r, gx[l - el * n]), L);
#pragma unroll
      for (int k = 0; k < 8 * PD; ++k) lines[l * LST + k] = L[k];
    }
    for (int i0 = 0; i0 < nq; i0 += CI) {
      const int cn = nq - i0 < CI ? nq - i0 : CI;
      const int per = cn * n;
      __syncthreads();
      for (int e = tid; e < 2 * per; e += NT) {
        const bool odd = e >= per;
        const int rem = odd ? e - per : e, ci = rem / n, jx = rem - ci * n, i = i0 + ci;
        const double xi0 = gx[i / n], xi1 = gx[i % n];
        const double t2 = (1 - xi0) * (1 - xi1);
        double u, v;
        tau(odd ? 1 - t2 : t2, xi1 * gx[jx], r2, u, v);
        tab[e] = make_point<PD, KIND>(g2, prm, u, v, gw[jx]);
      }
      __syncthreads();
      const int unit = tid / S, sub = tid - (tid / S) * S;
      const bool act = unit < per;
      const int uu = act ? unit : 0;
      const int ci = uu / n, j0 = uu - (uu / n) * n;
      const int i = i0 + ci, i1 = i % n;
      const double xi0 = gx[i / n], xi1 = gx[i1], wi = gw[i / n] * gw[i1];
      const double w = h * h * wi * xi1 * xi1;
      const double e0 = xi1 * gx[j0];
      const double t1 = xi0 * (1 - xi1), t2 = (1 - xi0) * (1 - xi1), t3 = xi0 * (1 - e0), t4 = (1 - xi0) * (1 - e0);
      const double fa = w * (gw[j0] * (1 - xi1)), fb = w * (gw[j0] * (1 - e0));
      const PtK* colt = tab + ci * n;
      // the point (t3 or 1 - t3, xi1) of element 1 or 2
      auto on_line = [&](int el, double x) {
        const int r = el ? r2 : r1;
        const bool fu = r & 1;
        const double f = held(r, xi1), m = moved(r, x);
        return line_point<PD, KIND>(lines + (el * n + i1) * LST, prm, fu, fu ? f : m, fu ? m : f, fb);
      };
#pragma unroll 1
      for (int odd = 0; odd < 2; ++odd) {
        {
          double u, v;
          tau(odd ? 1 - t1 : t1, e0, r1, u, v);
          const PtK F = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, fa));
          const double xc = moved(r2, odd ? 1 - t2 : t2);
          auto col = [&](int j1) { return colt[odd * per + j1]; };
          if (r2 & 1)
            line_pass<P, KIND, true, false>(dr, di, stage, F, lane, act, sub, S, n, prm, xc, col);
          else
            line_pass<P, KIND, true, true>(dr, di, stage, F, lane, act, sub, S, n, prm, xc, col);
        }
        const double x = odd ? 1 - t4 : t4;
        // g = 1, 2: the rotation, uniform in the workgroup, fixed at compile time (tau and the line
        // evaluation without selects)
        const LinePt F1 = sh.to_second(on_line(0, odd ? 1 - t3 : t3));
        with_rotation(r2, [&](auto R) {
          constexpr int RC = decltype(R)::value;
          constexpr bool FS = (RC & 1) == 0;
          double L[8 * PD];
          const double xf = RC < 2 ? x : 1 - x;
          line_contract<PD>(g2, FS, xf, L);
          line_pass<P, KIND, true, FS>(dr, di, stage, F1, lane, act, sub, S, n, prm, xf, [&](int j1) {
            double u, v;
            tau(x, xi1 * gx[j1], RC, u, v);
            return line_point<PD, KIND>(L, prm, FS, u, v, gw[j1]);
          });
        });
        const LinePt F2 = sh.to_first(on_line(1, odd ? 1 - t3 : t3));
        with_rotation(r1, [&](auto R) {
          constexpr int RC = decltype(R)::value;
          constexpr bool FS = (RC & 1) == 0;
          double L[8 * PD];
          const double xf = RC < 2 ? x : 1 - x;
          line_contract<PD>(g1, FS, xf, L);
          line_pass<P, KIND, false, FS>(dr, di, stage, F2, lane, act, sub, S, n, prm, xf, [&](int j1) {
            double u, v;
            tau(x, xi1 * gx[j1], RC, u, v);
            return line_point<PD, KIND>(L, prm, FS, u, v, gw[j1]);
          });
        });
      }
    }
    __syncthreads();
  } else if constexpr (CLS == 4 && !Acc::MAXW) {
    // integrate4, factorised: the four outer points per i as below; per chunk of first outer
    // coordinates the inner points p5 (element 2) and p6 (element 1) are tabulated, and a lane
    // fixed to one outer index i sums over its share of j: p5 gives columns for the rows of
    // q0, q1, p6 gives rows for the columns of q2, q3.
    const int r1 = pr.rot1, r2 = pr.rot2;
    constexpr bool CPLX = Acc::CPLX;
    PtK* q = reinterpret_cast<PtK*>(lds);  // 4 * nq
    PtK* tin = q + 4 * nq;
    for (int i = tid; i < nq; i += NT) {
      const double xi0 = gx[i / n], wi = gw[i / n] * gw[i % n];
      const double xi1 = gx[i % n] * xi0;
      const double w = h * h * wi * (xi0 * xi0 * xi0);
      double u, v;
      tau(xi0, xi1, r1, u, v);
      q[4 * i + 0] = make_point<PD, KIND>(g1, prm, u, v, w);
      tau(xi1, xi0, r1, u, v);
      q[4 * i + 1] = make_point<PD, KIND>(g1, prm, u, v, w);
      tau(xi0, xi1, r2, u, v);
      q[4 * i + 2] = make_point<PD, KIND>(g2, prm, u, v, w);
      tau(xi1, xi0, r2, u, v);
      q[4 * i + 3] = make_point<PD, KIND>(g2, prm, u, v, w);
    }
    const FactorShape shp = vertex_shape(n, NT, static_cast<int>(sizeof(PtK)), Acc::G);
    const int C0 = shp.chunk, S = shp.lanes;
    const int role = lane & (Acc::G - 1);
    for (int a0 = 0; a0 < n; a0 += C0) {
      const int cn = n - a0 < C0 ? n - a0 : C0;
      __syncthreads();
      for (int e = tid; e < 2 * cn * nq; e += NT) {
        const int which = e / (cn * nq), rem = e - which * (cn * nq);
        const int c0 = rem / nq, j = rem - c0 * nq;
        const double xi0 = gx[a0 + c0];
        const double e0 = xi0 * gx[j / n], e1 = xi0 * gx[j % n];
        const double wj = gw[j / n] * gw[j % n];
        double u, v;
        if (which == 0) {
          tau(e0, e1, r2, u, v);
          tin[e] = make_point<PD, KIND>(g2, prm, u, v, wj);
        } else {
          tau(e0, e1, r1, u, v);
          tin[e] = make_point<PD, KIND>(g1, prm, u, v, wj);
        }
      }
      __syncthreads();
      const int units = cn * n;
      const int unit = tid / S, sub = tid - (tid / S) * S;
      const bool act = unit < units;
      const int uu = act ? unit : 0;
      const int c0 = uu / n, i1 = uu - (uu / n) * n;
      const int i = (a0 + c0) * n + i1;
      const PtK* p5 = tin + c0 * nq;
      const PtK* p6 = tin + (cn + c0) * nq;
#pragma unroll 1
      for (int k = 0; k < 2; ++k)  // rows q0, q1 (element 1), columns p5 (element 2)
        factor_pass<P, KIND, true>(acc, sh.to_second(q[4 * i + k]), role, act, sub, S, nq, prm, [&](int j) { return p5[j]; });
#pragma unroll 1
      for (int k = 2; k < 4; ++k)  // rows p6 (element 1), columns q2, q3 (element 2)
        factor_pass<P, KIND, false>(acc, sh.to_first(q[4 * i + k]), role, act, sub, S, nq, prm, [&](int j) { return p6[j]; });
    }
    __syncthreads();
  } else if constexpr (CLS == 3) {
    // integrate3: common edge, 6 Duffy sub-regions.  With t1 = xi0 (1 - xi1), t2 = (1 - xi0)(1 - xi1),
    // e0 = xi1 xj0, e1 = xi1 xj1, t3 = xi0 (1 - e0), t4 = (1 - xi0)(1 - e0), sub-region k = 2g + odd
    // pairs a = tau(a0 or 1 - a0, a1; r1) on element 1 (weight w) with b = tau(b0 or 1 - b0, b1; r2)
    // on element 2 (weight wa for g = 0, else wb), where (a0, a1) = (t1, e0), (t3, xi1), (t4, e1)
    // and (b0, b1) = (t2, e1), (t4, e1), (t3, xi1).  The points of g = 0 (a: i, xj0; b: i, xj1), the
    // a points of g = 1 and the b points of g = 2 (i, xj0) come from per-chunk tables (W holds the
    // surface measure; the weight is applied where the point is used, as make_point does).
    const int r1 = pr.rot1, r2 = pr.rot2;
    const int CI = edge_chunk<PtK>(n, NT);
    PtK* tab = reinterpret_cast<PtK*>(lds);
    for (int i0 = 0; i0 < nq; i0 += CI) {
      const int cn = nq - i0 < CI ? nq - i0 : CI;
      const int per = cn * n;  // entries of one table kind
      __syncthreads();
      for (int e = tid; e < 8 * per; e += NT) {
        const int kind = e / per, rem = e - kind * per;
        const int ci = rem / n, jx = rem - ci * n;
        const int i = i0 + ci;
        const double xi0 = gx[i / n], xi1 = gx[i % n], xj = gx[jx];
        const bool odd = kind & 1;
        double u, v;
        if (kind < 2) {  // g = 0, a: (t1, e0) on element 1
          const double t1 = xi0 * (1 - xi1);
          tau(odd ? 1 - t1 : t1, xi1 * xj, r1, u, v);
          tab[e] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, 1.0));
        } else if (kind < 4) {  // g = 1, a: (t3, xi1) on element 1
          const double t3 = xi0 * (1 - xi1 * xj);
          tau(odd ? 1 - t3 : t3, xi1, r1, u, v);
          tab[e] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, 1.0));
        } else if (kind < 6) {  // g = 2, b: (t3, xi1) on element 2
          const double t3 = xi0 * (1 - xi1 * xj);
          tau(odd ? 1 - t3 : t3, xi1, r2, u, v);
          tab[e] = make_point<PD, KIND>(g2, prm, u, v, 1.0);
        } else {  // g = 0, b: (t2, e1) on element 2 (xj = xj1)
          const double t2 = (1 - xi0) * (1 - xi1);
          tau(odd ? 1 - t2 : t2, xi1 * xj, r2, u, v);
          tab[e] = make_point<PD, KIND>(g2, prm, u, v, 1.0);
        }
      }
      __syncthreads();
      const int total = cn * nq;
      for (int base = 0; base < total; base += NT) {
        const bool valid = base + tid < total;
        const int idx = valid ? base + tid : total - 1;
        const int ci = idx / nq, j = idx - (idx / nq) * nq;
        const int i = i0 + ci;
        const int j0 = j / n, j1 = j - (j / n) * n;
        const double xi0 = gx[i / n], xi1 = gx[i % n], wi = gw[i / n] * gw[i % n];
        const double xj0 = gx[j0], xj1 = gx[j1], wj = gw[j0] * gw[j1];
        const double w = h * h * wi * xi1 * xi1;
        const double e0 = xi1 * xj0, e1 = xi1 * xj1;
        const double t4 = (1 - xi0) * (1 - e0);
        const double wa = wj * (1 - xi1), wb = wj * (1 - e0);
        const int ta = ci * n + j0, tb = ci * n + j1;
#pragma unroll 1
        for (int k = 0; k < 6; ++k) {
          const int g = k >> 1;
          const bool odd = k & 1;
          PtK a, b;
          if (g == 0) {
            a = tab[(0 + odd) * per + ta];
            b = tab[(6 + odd) * per + tb];
          } else if (g == 1) {
            double u, v;
            a = tab[(2 + odd) * per + ta];
            tau(odd ? 1 - t4 : t4, e1, r2, u, v);
            b = make_point<PD, KIND>(g2, prm, u, v, 1.0);
          } else {
            double u, v;
            tau(odd ? 1 - t4 : t4, e1, r1, u, v);
            a = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, 1.0));
            b = tab[(4 + odd) * per + ta];
          }
          a.W *= w;
          b.W *= g == 0 ? wa : wb;
          acc.add(a, b, prm, rc, cc, valid, lane);
        }
      }
    }
    __syncthreads();
  } else {
    // integrate4: common vertex.  The four outer points per i are staged in LDS; the two inner
    // points p5 = tau(e0, e1; r2) on element 2 and p6 = tau(e0, e1; r1) on element 1, e = xi0 xj,
    // depend on the first outer coordinate and j only and are tabulated per chunk of xi0 values
    const int r1 = pr.rot1, r2 = pr.rot2;
    PtK* q = reinterpret_cast<PtK*>(lds);  // 4 * nq
    PtK* tin = q + 4 * nq;                 // 2 * nq per xi0 of the chunk
    for (int i = tid; i < nq; i += NT) {
      const double xi0 = gx[i / n], wi = gw[i / n] * gw[i % n];
      const double xi1 = gx[i % n] * xi0;
      const double w = h * h * wi * (xi0 * xi0 * xi0);
      double u, v;
      tau(xi0, xi1, r1, u, v);
      q[4 * i + 0] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, w));
      tau(xi1, xi0, r1, u, v);
      q[4 * i + 1] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, w));
      tau(xi0, xi1, r2, u, v);
      q[4 * i + 2] = make_point<PD, KIND>(g2, prm, u, v, w);
      tau(xi1, xi0, r2, u, v);
      q[4 * i + 3] = make_point<PD, KIND>(g2, prm, u, v, w);
    }
    const int C0 = vertex_chunk<PtK>(n, NT);
    for (int a0 = 0; a0 < n; a0 += C0) {
      const int cn = n - a0 < C0 ? n - a0 : C0;
      __syncthreads();
      for (int e = tid; e < 2 * cn * nq; e += NT) {
        const int which = e / (cn * nq), rem = e - which * (cn * nq);
        const int c0 = rem / nq, j = rem - c0 * nq;
        const double xi0 = gx[a0 + c0];
        const double e0 = xi0 * gx[j / n], e1 = xi0 * gx[j % n];
        double u, v;
        if (which == 0) {
          tau(e0, e1, r2, u, v);
          tin[e] = make_point<PD, KIND>(g2, prm, u, v, 1.0);
        } else {
          tau(e0, e1, r1, u, v);
          tin[e] = sh.to_second(make_point<PD, KIND>(g1, prm, u, v, 1.0));
        }
      }
      __syncthreads();
      const int total = cn * n * nq;  // (xi0 of the chunk, xi1, j)
      for (int base = 0; base < total; base += NT) {
        const bool valid = base + tid < total;
        const int idx = valid ? base + tid : total - 1;
        const int c0 = idx / (n * nq), rem = idx - c0 * (n * nq);
        const int i1 = rem / nq, j = rem - i1 * nq;
        const int i = (a0 + c0) * n + i1;
        const double wj = gw[j / n] * gw[j % n];
        PtK p5 = tin[c0 * nq + j], p6 = tin[(cn + c0) * nq + j];
        p5.W *= wj;
        p6.W *= wj;
        acc.add(q[4 * i + 0], p5, prm, rc, cc, valid, lane);
        acc.add(q[4 * i + 1], p5, prm, rc, cc, valid, lane);
        acc.add(p6, q[4 * i + 2], prm, rc, cc, valid, lane);
        acc.add(p6, q[4 * i + 3], prm, rc, cc, valid, lane);
      }
    }
    __syncthreads();
  }

  // reduce the per-lane partial blocks and write the result
  double* red = lds;
  double* sum = lds + (NT / 64) * Acc::TOT;
  if constexpr ((CLS == 2 && IDENT) || (CLS == 1 && !Acc::MAXW)) {
    if (tid < Acc::TOT) sum[tid] = aval;  // each entry summed by its owner
    __syncthreads();
  } else if constexpr (CLS == 3 && !Acc::MAXW) {
    // the four waves' blocks (the rules above end with a barrier)
    spread_blocks<I2, Acc::CPLX>(lds, tid >> 6, lane, dr, di);
    for (int k = tid; k < Acc::TOT; k += NT) {
      double v = 0.0;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) v += lds[w * Acc::TOT + k];
      sum[k] = v;
    }
    __syncthreads();
  } else {
    reduce_block<NT>(acc, red, tid, sum);
  }
  double* o = prm.out;
  constexpr bool CPLX = Acc::CPLX;
  const int64_t base = pr.off + rc * prm.comp_rs + cc * prm.comp_cs;
  // the factorised identical rule accumulated A; its block is A + A^T
  constexpr bool SYMW = CLS == 2 && IDENT;
  for (int k = tid; k < I2 * I2; k += NT) {
    const int i = k / I2, j = k - (k / I2) * I2;
    const int64_t idx = base + i * prm.rs + j * prm.cs;
    const int kt = j * I2 + i;
    if (CPLX) {
      o[2 * idx] = SYMW ? sum[k] + sum[kt] : sum[k];
      o[2 * idx + 1] = SYMW ? sum[I2 * I2 + k] + sum[I2 * I2 + kt] : sum[I2 * I2 + k];
    } else {
      o[idx] = SYMW ? sum[k] + sum[kt] : sum[k];
    }
  }
}

// far-field surface point table of all elements (DuffyTrick/farFieldQuadratureNodes.hpp:22-46)
template <int PD>
__global__ void k_ffield(const double* __restrict__ cp, int cp_stride, const int* __restrict__ elem_patch,
                         const double* __restrict__ elem_llc, int nel, int n, double h, int fs, double* out) {
  const int nq = n * n;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gid >= static_cast<int64_t>(nel) * nq) return;
  const int e = static_cast<int>(gid / nq), k = static_cast<int>(gid % nq);
  const double* gx = c_gl_nodes + c_gl_offset[n - 1];
  const double* gw = c_gl_weights + c_gl_offset[n - 1];
  const double u = gx[k / n], v = gx[k % n], w = h * (gw[k / n] * gw[k % n]);
  double X[3], Ds[3], Dt[3];
  const double* c = cp + static_cast<int64_t>(elem_patch[e]) * cp_stride;
  surface_point<PD>(c, elem_llc[2 * e] + h * u, elem_llc[2 * e + 1] + h * v, X, Ds, Dt);
  const double c0 = Ds[1] * Dt[2] - Ds[2] * Dt[1];
  const double c1 = Ds[2] * Dt[0] - Ds[0] * Dt[2];
  const double c2 = Ds[0] * Dt[1] - Ds[1] * Dt[0];
  double* o = out + gid * fs;
  o[0] = X[0], o[1] = X[1], o[2] = X[2];
  o[3] = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  o[4] = w, o[5] = u, o[6] = v, o[7] = 0.0;
  if (fs == FF_STRIDE_TAN) {
    o[8] = Ds[0], o[9] = Ds[1], o[10] = Ds[2];
    o[11] = Dt[0], o[12] = Dt[1], o[13] = Dt[2];
    o[14] = 0.0, o[15] = 0.0;
  }
}

void launch_ffield_table(const bmi_space* s, int n, int fs, double* out, hipStream_t st) {
  const int64_t total = static_cast<int64_t>(s->nel) * n * n;
  const int blocks = static_cast<int>((total + 255) / 256);
  const double h = 1.0 / s->n;
  const int stride = 4 * s->pd * s->pd;
  if (s->pd == 2)
    hipLaunchKernelGGL(k_ffield<2>, dim3(blocks), dim3(256), 0, st, s->d_cp.ptr, stride,
                       s->d_elem_patch.ptr, s->d_elem_llc.ptr, s->nel, n, h, fs, out);
  else if (s->pd == 5)
    hipLaunchKernelGGL(k_ffield<5>, dim3(blocks), dim3(256), 0, st, s->d_cp.ptr, stride,
                       s->d_elem_patch.ptr, s->d_elem_llc.ptr, s->nel, n, h, fs, out);
  else
    throw Error(BMI_UNSUPPORTED, "patch degree not supported on the device");
  BMI_CHECK_HIP(hipGetLastError());
}

// an unevaluated sum hi + lo: hi the rounded sum, lo the rounding errors of its additions and products
struct TwoSum {
  double hi = 0.0, lo = 0.0;
  __device__ __forceinline__ void add_product(double a, double b) {
#pragma clang fp contract(off)
    const double p = a * b, s = hi + p, t = s - hi;
    lo += fma(a, b, -p) + ((hi - (s - t)) + (p - t));
    hi = s;
  }
  __device__ __forceinline__ void add_product(double a, const double2& b) {  // a (hi, lo)
    add_product(a, b.x);
    lo = fma(a, b.y, lo);
  }
};

// the homogeneous coordinates of every element in powers of u - 1/2, v - 1/2 (poly_point): coefficient
// (a, b) is h^(a + b) / (a! b!) times the derivative at the element's centre, from differences of the
// control points in Bernstein form.  An error of a coefficient is one of all points of the element, of which a
// block's sum leaves the whole where it averages those of the points: each is rounded once.  The weights are
// exact (element corners are multiples of 2^-M, M <= 10: 44 bits), and the sums over the control points carry
// their rounding errors along.
// Bound: latency.  A workgroup holds an element, one direction after the other, a thread per sum of PD products
// (a thread per coefficient, with sums of PD^2 products and weights of its own in scratch memory: 24 elements
// 15.0 us, 3.3 so; 24,576 elements 83 -> 27 us).
constexpr int POLY_NT = 128;
template <int PD>
__global__ __launch_bounds__(POLY_NT) void k_element_poly(const double* __restrict__ cp, int cp_stride,
                                                          const int* __restrict__ elem_patch,
                                                          const double* __restrict__ elem_llc, double h, int centre,
                                                          int stride, double* __restrict__ out) {
  constexpr int p = PD - 1;
  static_assert(4 * PD * PD <= POLY_NT && 2 * PD <= POLY_NT, "a thread per sum");
  __shared__ double w[2][PD][PD];  // weights of the control points: direction, power, point
  __shared__ double2 r[PD][PD][4], v[PD][PD][4];  // sums (hi, lo)
  const int e = blockIdx.x, t = threadIdx.x;
  if (t < 2 * PD) {
    // the a-th power coefficient of one direction about the centre x: h^a binom(p, a) sum over q of
    // (-1)^(a - q) binom(a, q) B_(i - q) of degree p - a
    const int dir = t / PD, a = t % PD;
    const double x = elem_llc[2 * e + dir] + 0.5 * h;
    double B[PD], c[PD];
#pragma unroll
    for (int i = 0; i < PD; ++i) B[i] = i == 0 ? 1.0 : 0.0, c[i] = 0.0;
#pragma unroll
    for (int d = 1; d <= p; ++d)  // Bernstein recurrence up to degree p - a
      if (d <= p - a)
#pragma unroll
        for (int i = d; i >= 0; --i) B[i] = (i > 0 ? x * B[i > 0 ? i - 1 : 0] : 0.0) + (i < d ? (1 - x) * B[i] : 0.0);
    double f = 1.0;
    int bin = 1;
#pragma unroll
    for (int k = 0; k < p; ++k)
      if (k < a) bin = bin * (p - k) / (k + 1), f *= h;
    f *= bin;
    bin = 1;
#pragma unroll
    for (int q = 0; q <= p; ++q)
      if (q <= a) {
        const double g = ((a - q) & 1) ? -f * bin : f * bin;
#pragma unroll
        for (int i = 0; i + q <= p; ++i) c[i + q] += g * B[i];  // B is zero beyond degree p - a
        bin = bin * (a - q) / (q + 1);
      }
#pragma unroll
    for (int i = 0; i < PD; ++i) w[dir][a][i] = c[i];
  }
  __syncthreads();
  const int k = t & 3, j = (t >> 2) % PD, a = (t >> 2) / PD;
  const bool on = t < 4 * PD * PD;
  if (on) {
    const double* c = cp + static_cast<int64_t>(elem_patch[e]) * cp_stride + 4 * j + k;
    TwoSum s;
#pragma unroll
    for (int i = 0; i < PD; ++i) s.add_product(w[0][a][i], c[4 * PD * i]);
    r[a][j][k] = make_double2(s.hi, s.lo);
  }
  __syncthreads();
  TwoSum s;
  if (on) {
#pragma unroll
    for (int i = 0; i < PD; ++i) s.add_product(w[1][j][i], r[a][i][k]);
    v[a][j][k] = make_double2(s.hi, s.lo);
  }
  __syncthreads();
  if (!on) return;
  // about the centre: the weight times it taken off
  double* o = out + static_cast<int64_t>(e) * stride;
  const double O = centre && k < 3 ? static_cast<double>(static_cast<float>(v[0][0][k].x / v[0][0][3].x)) : 0.0;
  s.add_product(-O, v[a][j][3]);
  o[t] = s.hi + s.lo;
  if (t < 4) o[stride - 4 + t] = O;
}

// doubles of an element's polynomials and centre
static int poly_stride(const bmi_space* s) { return 4 * s->pd * s->pd + 4; }

static int64_t poly_doubles(const bmi_space* s) { return static_cast<int64_t>(s->nel) * poly_stride(s); }

static void element_polynomials(const bmi_space* s, bool centre, double* out, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(s->nel));
  const int stride = 4 * s->pd * s->pd;
  if (s->pd == 2)
    hipLaunchKernelGGL(k_element_poly<2>, grid, dim3(POLY_NT), 0, st, s->d_cp.ptr, stride, s->d_elem_patch.ptr,
                       s->d_elem_llc.ptr, 1.0 / s->n, centre ? 1 : 0, poly_stride(s), out);
  else if (s->pd == 5)
    hipLaunchKernelGGL(k_element_poly<5>, grid, dim3(POLY_NT), 0, st, s->d_cp.ptr, stride, s->d_elem_patch.ptr,
                       s->d_elem_llc.ptr, 1.0 / s->n, centre ? 1 : 0, poly_stride(s), out);
  else
    throw Error(BMI_UNSUPPORTED, "patch degree not supported on the device");
  BMI_CHECK_HIP(hipGetLastError());
}

// element widths, and the scaling of the line points' measures by the radius of the largest patch
static void set_lengths(const bmi_space* s, NFParams& prm) {
  double l = 0.0;
  for (const double r : s->crad[0]) l = std::max(l, r);
  const int k = l > 0.0 && std::isfinite(l) ? std::max(-250, std::min(250, std::ilogb(l))) : 0;
  prm.h = 1.0 / s->n;
  prm.rh = s->n;
  prm.rh2 = static_cast<double>(s->n) * s->n;
  prm.ms = std::ldexp(1.0, -4 * k);
  prm.mr = std::ldexp(prm.rh2, 2 * k);
}

// dynamic LDS of one workgroup of class CLS at quadrature degree deg (each workgroup sizes its
// point tables from its own pair's degree)
template <int P, int KIND, int PD, int CLS, int NT>
static size_t class_lds_bytes(int deg) {
  const int n = deg + 1, nq = n * n;
  size_t lds = sizeof(double) * ((NT / 64) + 1) * BlockAcc<P, KIND>::TOT;
  if (CLS == 1) lds = std::max(lds, 2 * nq * sizeof(Pt<KIND>));
  if (CLS == 1 && KIND != BMI_MAXWELL_SL)  // points, the lanes' vectors, the outer basis values
    lds = std::max(lds, 2 * nq * sizeof(Pt<KIND>) + static_cast<size_t>(NT) *
                                                        ((BlockAcc<P, KIND>::CPLX ? 3 : 2) * (P + 1) * (P + 1)) *
                                                        sizeof(double));
  constexpr bool FACT = KIND != BMI_MAXWELL_SL;  // factorised vertex rule
  constexpr int PS = static_cast<int>(sizeof(Pt<KIND>));
  const int cv = FACT ? vertex_shape(n, NT, PS, BlockAcc<P, KIND>::G).chunk : vertex_chunk<Pt<KIND>>(n, NT);
  // the waves' vectors behind the tables (factorised edge rule)
  const size_t stg = FACT ? (NT / 64) * stage_doubles<(P + 1) * (P + 1)>(BlockAcc<P, KIND>::CPLX) * sizeof(double) : 0;
  if (CLS == 3)
    lds = std::max(lds, FACT ? static_cast<size_t>(2 * n * edge_shape(n, NT, PS).chunk) * sizeof(Pt<KIND>) +
                                   static_cast<size_t>(2 * n * line_stride(PD)) * sizeof(double) + stg
                             : static_cast<size_t>(8 * n * edge_chunk<Pt<KIND>>(n, NT)) * sizeof(Pt<KIND>));
  if (CLS == 2 && (KIND == BMI_LAPLACE_SL || KIND == BMI_HELMHOLTZ_SL))  // lines, the waves' unit vectors
    lds = std::max(lds, (static_cast<size_t>(identical_chunk(n, PD)) * 4 * n * line_stride(PD) +
                         static_cast<size_t>(NT / 2) * (BlockAcc<P, KIND>::CPLX ? 3 : 2) * (P + 1) * (P + 1)) *
                            sizeof(double));
  if (CLS == 4) lds = std::max(lds, static_cast<size_t>(4 * nq + 2 * nq * cv) * sizeof(Pt<KIND>));
  return lds;
}

// one launch for the pairs [d_pairs, d_pairs + count) of class CLS; degs lists the distinct
// quadrature degrees among them, and the launch gets the largest LDS any of them needs (the
// table size is not monotone in the degree: the chunk sizes change with it)
template <int P, int KIND, int PD, int CLS>
static void launch_class(const NFPair* d_pairs, int count, const std::vector<int>& degs, NFParams prm,
                         hipStream_t st) {
  if (count == 0) return;
  constexpr int NT = (CLS == 0) ? 64 : 256;
  size_t lds = 0;
  for (int d : degs) lds = std::max(lds, class_lds_bytes<P, KIND, PD, CLS, NT>(d));
  BMI_REQUIRE(lds <= 160 * 1024, BMI_UNSUPPORTED, "quadrature degree too large for LDS staging");
  const char* name = CLS == 2 ? "nf_identical" : CLS == 3 ? "nf_edge" : CLS == 4 ? "nf_vertex" : "nf_regular";
  TimedScope ts(name, st);
  const int ncomp = KIND == BMI_MAXWELL_SL ? 4 : 1;
  hipLaunchKernelGGL((k_nearfield<P, KIND, PD, CLS, NT>), dim3(count, ncomp), dim3(NT), lds, st, d_pairs,
                     prm);
  BMI_CHECK_HIP(hipGetLastError());
}

template <int P, int KIND, int PD>
static void launch_all(const std::vector<NFPair>& pairs, const NFPair* d_pairs, NFParams prm,
                       hipStream_t st) {
  // pairs are sorted by class, then by falling degree: one launch per class holds every
  // quadrature degree of the class (each workgroup reads its pair's degree; LDS is sized for the
  // largest need among the degrees present), the most expensive pairs first so the tail of the
  // launch is short
  size_t a = 0;
  while (a < pairs.size()) {
    size_t b = a;
    std::vector<int> degs;
    while (b < pairs.size() && pairs[b].cls == pairs[a].cls) {
      if (degs.empty() || degs.back() != pairs[b].deg) degs.push_back(pairs[b].deg);
      ++b;
    }
    const int cnt = static_cast<int>(b - a);
    switch (pairs[a].cls) {
      case 0: launch_class<P, KIND, PD, 0>(d_pairs + a, cnt, degs, prm, st); break;
      case 1: launch_class<P, KIND, PD, 1>(d_pairs + a, cnt, degs, prm, st); break;
      case 2: launch_class<P, KIND, PD, 2>(d_pairs + a, cnt, degs, prm, st); break;
      case 3: launch_class<P, KIND, PD, 3>(d_pairs + a, cnt, degs, prm, st); break;
      default: launch_class<P, KIND, PD, 4>(d_pairs + a, cnt, degs, prm, st); break;
    }
    a = b;
  }
}

static void dispatch(const bmi_space* s, int kind, int P, const std::vector<NFPair>& pairs,
                     const NFPair* d_pairs, NFParams prm, hipStream_t st) {
  const int pd = s->pd;
#define BMI_NF_CASE(PP, KK, DD) \
  if (P == PP && kind == KK && pd == DD) return launch_all<PP, KK, DD>(pairs, d_pairs, prm, st);
  BMI_NF_CASE(1, BMI_LAPLACE_SL, 5)
  BMI_NF_CASE(2, BMI_LAPLACE_SL, 5)
  BMI_NF_CASE(1, BMI_HELMHOLTZ_SL, 5)
  BMI_NF_CASE(2, BMI_HELMHOLTZ_SL, 5)
  BMI_NF_CASE(1, BMI_LAPLACE_SL, 2)
  BMI_NF_CASE(2, BMI_LAPLACE_SL, 2)
  BMI_NF_CASE(1, BMI_HELMHOLTZ_SL, 2)
  BMI_NF_CASE(2, BMI_HELMHOLTZ_SL, 2)
  BMI_NF_CASE(1, BMI_MAXWELL_SL, 5)
  BMI_NF_CASE(2, BMI_MAXWELL_SL, 5)
  BMI_NF_CASE(1, BMI_MAXWELL_SL, 2)
  BMI_NF_CASE(2, BMI_MAXWELL_SL, 2)
  BMI_NF_CASE(0, BMI_DUMMY, 2)
#undef BMI_NF_CASE
  throw Error(BMI_UNSUPPORTED, "near-field kernel not instantiated for this operator/degree/patch order");
}

void launch_nearfield(const bmi_space* s, const bmi_op_desc& op, std::vector<NFPair>& pairs, double* out,
                      int64_t rs, int64_t cs, int64_t comp_rs, int64_t comp_cs, hipStream_t st) {
  ensure_device_space(s, st);
  const int ff = farfield_degree(op.kind, s->P);
  const FFTable* tab = ensure_ffield(s, ff, st, op.kind == BMI_MAXWELL_SL);
  {
    // stable counting sort by class, then by decreasing degree (degrees < 50): the launches take
    // one class each, its pairs with the largest rules first
    HostTimedScope hs("assembly_host_pair_sort");
    constexpr int ND = 50;
    std::vector<int64_t> start(5 * ND + 1, 0);
    for (const NFPair& p : pairs) {
      BMI_REQUIRE(p.cls >= 0 && p.cls < 5 && p.deg >= 0 && p.deg < ND, BMI_UNSUPPORTED,
                  "near-field pair class or quadrature degree out of range");
      start[p.cls * ND + (ND - 1 - p.deg) + 1]++;
    }
    for (int b = 0; b < 5 * ND; ++b) start[b + 1] += start[b];
    std::vector<NFPair> sorted(pairs.size());
    for (const NFPair& p : pairs) sorted[start[p.cls * ND + (ND - 1 - p.deg)]++] = p;
    pairs.swap(sorted);
  }
  // (two allocations: together they pass 2 MB from 1,536 elements on, where an allocation of the runtime
  // takes 0.3 ms more)
  DevBuf<NFPair> d_pairs;
  d_pairs.upload(pairs, st);
  DevBuf<double> d_poly;
  d_poly.alloc(static_cast<size_t>(poly_doubles(s)));
  element_polynomials(s, op.kind != BMI_DUMMY, d_poly.ptr, st);
  NFParams prm;
  prm.poly = d_poly.ptr;
  prm.poly_stride = poly_stride(s);
  set_lengths(s, prm);
  prm.kre = op.kappa_re;
  prm.kim = op.kappa_im;
  prm.dummy_fn = op.dummy_fn;
  prm.ffield = tab->buf.ptr;
  prm.nff = (ff + 1) * (ff + 1);
  prm.ffs = tab->fs;
  prm.out = out;
  prm.rs = rs;
  prm.cs = cs;
  prm.comp_rs = comp_rs;
  prm.comp_cs = comp_cs;
  prm.qre = prm.qim = 0.0;
  if (op.kind == BMI_MAXWELL_SL) {
    // -1 / (kappa^2 h^2) with h = 2^-M (Maxwell/SingleLayerOperator.hpp:71-76)
    const double k2r = op.kappa_re * op.kappa_re - op.kappa_im * op.kappa_im;
    const double k2i = 2 * op.kappa_re * op.kappa_im;
    const double h2 = prm.h * prm.h;
    const double den = (k2r * k2r + k2i * k2i) * h2;
    prm.qre = -k2r / den;
    prm.qim = k2i / den;
  }
  dispatch(s, op.kind, s->P, pairs, d_pairs.ptr, prm, st);
  BMI_CHECK_HIP(hipStreamSynchronize(st));
}

void launch_integrate_jobs(const bmi_space* s, const bmi_op_desc& op, const std::vector<int>& jobs,
                           int qdeg, double* out, hipStream_t st) {
  ensure_device_space(s, st);
  const FFTable* tab = ensure_ffield(s, qdeg, st, false);
  std::vector<NFPair> pairs;
  const int nj = static_cast<int>(jobs.size() / 5);
  for (int k = 0; k < nj; ++k) {
    NFPair p;
    p.cls = jobs[5 * k];
    p.e1 = jobs[5 * k + 1];
    p.rot1 = jobs[5 * k + 2];
    p.e2 = jobs[5 * k + 3];
    p.rot2 = jobs[5 * k + 4];
    p.deg = qdeg;
    p.off = k;
    pairs.push_back(p);
  }
  DevBuf<double> d_poly;
  d_poly.alloc(static_cast<size_t>(poly_doubles(s)));
  element_polynomials(s, op.kind != BMI_DUMMY, d_poly.ptr, st);
  NFParams prm;
  prm.poly = d_poly.ptr;
  prm.poly_stride = poly_stride(s);
  set_lengths(s, prm);
  prm.kre = op.kappa_re;
  prm.kim = op.kappa_im;
  prm.dummy_fn = op.dummy_fn;
  prm.ffield = tab->buf.ptr;
  prm.nff = (qdeg + 1) * (qdeg + 1);
  prm.ffs = tab->fs;
  prm.out = out;
  prm.rs = 0;
  prm.cs = 0;
  prm.comp_rs = prm.comp_cs = 0;
  prm.qre = prm.qim = 0.0;
  // jobs are launched one group per class, keeping their output slots
  std::vector<NFPair> sorted = pairs;
  std::stable_sort(sorted.begin(), sorted.end(), [](const NFPair& a, const NFPair& b) { return a.cls < b.cls; });
  DevBuf<NFPair> d_sorted;
  d_sorted.upload(sorted, st);
  dispatch(s, op.kind, s->P, sorted, d_sorted.ptr, prm, st);
  BMI_CHECK_HIP(hipStreamSynchronize(st));
}

}  // namespace bmi
