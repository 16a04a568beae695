// Tree transformations of products with column-major vectors (one to a few right-hand sides): moments
// and transfers up the cluster tree, transfers and leaf rows down it (H2Multipole.hpp:380-469).
//
// Both are tensor products: the Chebyshev grid of a cluster is a product grid, so a transfer matrix is
// E_a (x) E_b with the n x n matrices E_0, E_1 of the two halves of an interval, and a moment matrix is
// m1 (x) m2 with the n x c1 moments of one direction (c1 = 2^min_cluster_level (P + 1) basis
// functions).  Applied one direction at a time a parent costs 6 n^3 multiply-adds instead of 4 n^4 and
// a leaf c1 n (c1 + n) instead of c1^2 n^2, and all matrices fit in LDS.  Bound: latency (a few
// steps with a barrier each, few workgroups), so a step is spread over as many threads as it has
// results (a thread per row of results, its coefficients through the scalar cache, measured 1.1 to
// 1.8 times slower).  One column's T x is formed by the bottom launch on its way in.
//
// Measured against whole-matrix products (matrices in LDS for 16 and 25 rows, from the L2 beyond), us
// per launch: up, Laplace 24,576 elements 4x4 nodes 8.8 -> 6.4, Helmholtz 5x5 18.0 -> 9.0, 6,144
// elements 9x9 70.7 -> 12.9; down 9.3 -> 8.1, 16.8 -> 12, 42.3 -> 10.0; the Maxwell product of 1,536
// elements 1182 -> 872 us (one launch for both components).
//
// One workgroup owns one cluster at level `top` and its subtree down to level `bot`, all levels in LDS
// (matrices n x n, rows padded to an odd number of entries so that threads on consecutive rows read
// different banks); blockIdx.y is the right-hand side, blockIdx.z the vector component (Maxwell).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bmi_fmm.h"
#include "bmi_internal.h"

namespace bmi {

namespace {

template <bool C>
struct Num;
template <>
struct Num<false> {
  double r = 0.0;
  __device__ static Num get(const double* p, int64_t k) {
    Num v;
    v.r = p[k];
    return v;
  }
  __device__ void put(double* p, int64_t k) const { p[k] = r; }
  __device__ void fma(double a, const Num& x) { r += a * x.r; }
  __device__ void add(const Num& x) { r += x.r; }
};
template <>
struct Num<true> {
  double r = 0.0, i = 0.0;
  __device__ static Num get(const double* p, int64_t k) {
    const double2 d = *reinterpret_cast<const double2*>(p + 2 * k);
    Num v;
    v.r = d.x, v.i = d.y;
    return v;
  }
  __device__ void put(double* p, int64_t k) const { *reinterpret_cast<double2*>(p + 2 * k) = make_double2(r, i); }
  __device__ void fma(double a, const Num& x) { r += a * x.r, i += a * x.i; }
  __device__ void add(const Num& x) { r += x.r, i += x.i; }
};

// clusters of the levels above depth d of a subtree
__host__ __device__ constexpr int above(int d) { return ((1 << (2 * d)) - 1) / 3; }
// son (order (0,0), (1,0), (1,1), (0,1)) of the halves a of the first, b of the second direction
__device__ __forceinline__ int son_of(int a, int b) { return a ? (b ? 2 : 1) : (b ? 3 : 0); }
// (a, b) of son q
__device__ __forceinline__ int half1(int q) { return (q == 1 || q == 2) ? 1 : 0; }
__device__ __forceinline__ int half2(int q) { return q >= 2 ? 1 : 0; }
// element e of a leaf cluster (Morton order, mcl levels): its place in the two directions
__device__ __forceinline__ void leaf_place(int e, int mcl, int& is, int& it) {
  is = 0, it = 0;
  for (int l = mcl - 1; l >= 0; --l) {
    const int q = (e >> (2 * l)) & 3;
    is = 2 * is + half1(q), it = 2 * it + half2(q);
  }
}

template <int NP>
struct Grid {
  static constexpr int RS = NP | 1;    // entries between rows of a matrix
  static constexpr int MS = NP * RS;   // entries of a matrix
};

// LDS entries (scalars) of the up pass of depth D
__host__ __device__ constexpr int up_levels(int D, int nc, int ms) { return above(D + 1) * nc * ms; }
__host__ __device__ constexpr int max_int(int a, int b) { return a > b ? a : b; }
__host__ __device__ constexpr int up_scratch(int D, int nc, int np, int c1, bool moment) {
  const int rs = np | 1, ms = np * rs;
  const int u = D > 0 ? (1 << (2 * (D - 1))) * nc * 2 * ms : 0;
  return max_int(u, moment ? (1 << (2 * D)) * (c1 * (c1 | 1) + nc * c1 * rs) : 0);
}
__host__ __device__ constexpr int down_scratch(int D, int nc, int np, int c1) {
  const int rs = np | 1, ms = np * rs;
  const int w = D > 0 ? (1 << (2 * (D - 1))) * nc * 2 * ms : nc * ms;
  return max_int(w, (1 << (2 * D)) * nc * c1 * rs);
}

// Tables of one direction in LDS: E and the moments (of the component's two directions) as they are,
// and transposed copies for the steps whose threads walk the other index
template <int NP>
struct Tables {
  double *E, *Et, *m, *mt;
  // E(i, half h, polynomial j), moment of node i and basis function b; v: 1 the derivative's moments
  __device__ double e(int i, int h, int j) const { return E[i * 2 * NP + h * NP + j]; }
  __device__ double et(int i, int h, int j) const { return Et[(j * 2 + h) * NP + i]; }
};
__host__ __device__ constexpr int table_doubles(int np, int c1, int vd) { return 4 * np * np + 2 * vd * np * c1; }

template <int NP>
__device__ __forceinline__ Tables<NP> stage_tables(const TreeArgs& a, double* p) {
  const int nm = a.vd * NP * a.c1;
  Tables<NP> t{p, p + 2 * NP * NP, p + 4 * NP * NP, p + 4 * NP * NP + nm};
  for (int q = threadIdx.x; q < 2 * NP * NP; q += blockDim.x) {
    const int i = q / (2 * NP), h = q % (2 * NP) / NP, j = q % NP;
    const double v = a.E[q];
    t.E[q] = v;
    t.Et[(j * 2 + h) * NP + i] = v;
  }
  for (int q = threadIdx.x; q < nm; q += blockDim.x) {
    const int v = q / (NP * a.c1), r = q - v * (NP * a.c1), i = r / a.c1, b = r - i * a.c1;
    const double x = a.m[q];
    t.m[q] = x;
    t.mt[v * NP * a.c1 + b * NP + i] = x;
  }
  return t;
}

// Every step below is one entry of the result per thread (consecutive threads on consecutive entries
// of a row: consecutive LDS words of one operand, one broadcast of the other), its terms unrolled.
template <bool C, int NP>
__global__ __launch_bounds__(256) void k_tree_up(TreeArgs a, int top, int bot, int from_moment) {
  extern __shared__ double lds[];
  constexpr int S = C ? 2 : 1, RS = Grid<NP>::RS, MS = Grid<NP>::MS, N2 = NP * NP;
  using V = Num<C>;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int ctop = blockIdx.x, k = blockIdx.y, comp = blockIdx.z;
  const int nc = a.nc, c1 = a.c1, D = bot - top, rows = nc * N2;
  double* fw = comp ? a.v1 : a.v0;
  auto level = [&](int d) { return lds + S * nc * MS * above(d); };
  double* tmp = lds + S * up_levels(D, nc, MS);
  const Tables<NP> t = stage_tables<NP>(a, tmp + S * up_scratch(D, nc, NP, c1, from_moment != 0));
  // entry `row` of cluster cl of depth d in the multipole array
  auto place = [&](int d, int cl, int row) {
    const int64_t c = (static_cast<int64_t>(ctop) << (2 * d)) + cl;
    return a.lvl_off[top + d] * a.nrhs + (c * a.nrhs + k) * rows + row;
  };
  auto entry = [](int q) { return q / N2 * MS + q % N2 / NP * RS + q % NP; };  // row -> LDS
  const int nb = 1 << (2 * D);
  double* Lb = level(D);
  if (from_moment) {
    const int XS = c1 | 1, dd = c1 * c1, I2 = a.pp1 * a.pp1;
    double* X = tmp;
    double* Vb = tmp + S * nb * c1 * XS;
    const double* x = a.x + S * (static_cast<int64_t>(k) * a.ldx + comp * a.xseg + (static_cast<int64_t>(ctop) << (2 * D)) * dd);
    for (int idx = tid; idx < nb * dd; idx += nt) {
      const int cl = idx / dd, e = idx - cl * dd, el = e / I2, m = e - el * I2;
      int is, it;
      leaf_place(el, a.mcl, is, it);
      const int be = is * a.pp1 + m % a.pp1, al = it * a.pp1 + m / a.pp1;
      V v;
      if (a.trp) {
        // the super vector's row of T x, also written for the near-field sweep
        const int64_t row = (static_cast<int64_t>(ctop) << (2 * D)) * dd + idx;
        for (int p = a.trp[row]; p < a.trp[row + 1]; ++p) v.fma(a.tval[p], V::get(a.xin, a.tcol[p]));
        v.put(a.xs, row);
      } else {
        v = V::get(x, idx);
      }
      v.put(X, (cl * c1 + be) * XS + al);
    }
    __syncthreads();
    // V(beta, j) = sum over alpha of m2(j, alpha) x(beta, alpha)
    for (int idx = tid; idx < nc * nb * c1 * NP; idx += nt) {
      const int m = idx / NP, j = idx - m * NP, r = m / (nb * c1), b = m - r * (nb * c1);
      const double* m2 = t.mt + (r == 1 && comp == 1 ? NP * c1 : 0) + j;
      V acc;
#pragma unroll 6
      for (int al = 0; al < c1; ++al) acc.fma(m2[al * NP], V::get(X, b * XS + al));
      acc.put(Vb, m * RS + j);
    }
    __syncthreads();
    // moment(i, j) = sum over beta of m1(i, beta) V(beta, j)
    for (int idx = tid; idx < nb * rows; idx += nt) {
      const int cl = idx / rows, row = idx - cl * rows, r = row / N2, i = row % N2 / NP, j = row % NP;
      const double* m1 = t.m + (r == 1 && comp == 0 ? NP * c1 : 0) + i * c1;
      V acc;
#pragma unroll 6
      for (int be = 0; be < c1; ++be) acc.fma(m1[be], V::get(Vb, ((r * nb + cl) * c1 + be) * RS + j));
      acc.put(Lb, cl * nc * MS + entry(row));
      const int64_t g = place(D, cl, row);
      acc.put(fw, g);
      if (a.clear) V().put(a.clear, g);
    }
  } else {
    for (int idx = tid; idx < nb * rows; idx += nt) {
      const int cl = idx / rows, row = idx - cl * rows;
      V::get(fw, place(D, cl, row)).put(Lb, cl * nc * MS + entry(row));
    }
  }
  __syncthreads();
  for (int d = D - 1; d >= 0; --d) {
    const int n = (1 << (2 * d)) * nc;
    const double* Ch = level(d + 1);
    double* Pa = level(d);
    // U_a(i, jj) = sum over b, ii of E_b(ii, jj) child_ab(i, ii)
    for (int idx = tid; idx < n * 2 * N2; idx += nt) {
      const int m = idx / (2 * N2), ha = idx % (2 * N2) / N2, i = idx % N2 / NP, jj = idx % NP;
      const int cl = m / nc, r = m - cl * nc;
      V acc;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int o = ((4 * cl + son_of(ha, b)) * nc + r) * MS + i * RS;
#pragma unroll
        for (int ii = 0; ii < NP; ++ii) acc.fma(t.e(ii, b, jj), V::get(Ch, o + ii));
      }
      acc.put(tmp, (m * 2 + ha) * MS + i * RS + jj);
    }
    __syncthreads();
    // parent(j, jj) = sum over a, i of E_a(i, j) U_a(i, jj)
    for (int idx = tid; idx < n * N2; idx += nt) {
      const int m = idx / N2, j = idx % N2 / NP, jj = idx % NP;
      V acc;
#pragma unroll
      for (int ha = 0; ha < 2; ++ha)
#pragma unroll
        for (int i = 0; i < NP; ++i) acc.fma(t.e(i, ha, j), V::get(tmp, (m * 2 + ha) * MS + i * RS + jj));
      acc.put(Pa, m * MS + j * RS + jj);
      const int64_t g = place(d, m / nc, (m % nc) * N2 + j * NP + jj);
      acc.put(fw, g);
      if (a.clear) V().put(a.clear, g);
    }
    __syncthreads();
  }
}

template <bool C, int NP>
__global__ __launch_bounds__(256) void k_tree_down(TreeArgs a, int top, int bot) {
  extern __shared__ double lds[];
  constexpr int S = C ? 2 : 1, RS = Grid<NP>::RS, MS = Grid<NP>::MS, N2 = NP * NP;
  using V = Num<C>;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int ctop = blockIdx.x, k = blockIdx.y, comp = blockIdx.z;
  const int nc = a.nc, c1 = a.c1, D = bot - top, rows = nc * N2;
  const double* bw = comp ? a.v1 : a.v0;
  auto level = [&](int d) { return lds + S * nc * MS * above(d); };
  double* tmp = lds + S * up_levels(D, nc, MS);
  double* anc = tmp + S * down_scratch(D, nc, NP, c1);  // ancestors, level 0 .. top - 1
  const Tables<NP> t = stage_tables<NP>(a, anc + S * nc * MS * top);
  auto entry = [](int q) { return q / N2 * MS + q % N2 / NP * RS + q % NP; };
  // the coupling sums of the ancestors and of every level of the subtree
  for (int idx = tid; idx < (top + 1) * rows; idx += nt) {
    const int l = idx / rows, row = idx - l * rows;
    const int64_t c = static_cast<int64_t>(ctop) >> (2 * (top - l));
    double* to = l < top ? anc + S * nc * MS * l : level(0);
    V::get(bw, a.lvl_off[l] * a.nrhs + (c * a.nrhs + k) * rows + row).put(to, entry(row));
  }
  for (int d = 1; d <= D; ++d) {
    double* L = level(d);
    for (int idx = tid; idx < (rows << (2 * d)); idx += nt) {
      const int cl = idx / rows, row = idx - cl * rows;
      const int64_t c = (static_cast<int64_t>(ctop) << (2 * d)) + cl;
      V::get(bw, a.lvl_off[top + d] * a.nrhs + (c * a.nrhs + k) * rows + row).put(L, cl * nc * MS + entry(row));
    }
  }
  __syncthreads();
  // one cluster per level down to this workgroup's (every workgroup repeats this short chain instead of
  // waiting for a launch above it), then the subtree: W_b(j, ii) = sum over jj of E_b(ii, jj)
  // parent(j, jj), child_ab(i, ii) += sum over j of E_a(i, j) W_b(j, ii)
  for (int l = 1; l <= top; ++l) {
    const int q = (ctop >> (2 * (top - l))) & 3, ha = half1(q), hb = half2(q);
    const double* Pa = anc + S * nc * MS * (l - 1);
    double* Ch = l < top ? anc + S * nc * MS * l : level(0);
    for (int e = tid; e < rows; e += nt) {
      const int r = e / N2, j = e % N2 / NP, ii = e % NP;
      V acc;
#pragma unroll
      for (int jj = 0; jj < NP; ++jj) acc.fma(t.et(ii, hb, jj), V::get(Pa, r * MS + j * RS + jj));
      acc.put(tmp, r * MS + j * RS + ii);
    }
    __syncthreads();
    for (int e = tid; e < rows; e += nt) {
      const int r = e / N2, i = e % N2 / NP, ii = e % NP;
      V acc = V::get(Ch, r * MS + i * RS + ii);
#pragma unroll
      for (int j = 0; j < NP; ++j) acc.fma(t.e(i, ha, j), V::get(tmp, r * MS + j * RS + ii));
      acc.put(Ch, r * MS + i * RS + ii);
    }
    __syncthreads();
  }
  for (int d = 1; d <= D; ++d) {
    const int n = (1 << (2 * (d - 1))) * nc;
    const double* Pa = level(d - 1);
    double* Ch = level(d);
    for (int idx = tid; idx < n * 2 * N2; idx += nt) {
      const int m = idx / (2 * N2), b = idx % (2 * N2) / N2, j = idx % N2 / NP, ii = idx % NP;
      V acc;
#pragma unroll
      for (int jj = 0; jj < NP; ++jj) acc.fma(t.et(ii, b, jj), V::get(Pa, m * MS + j * RS + jj));
      acc.put(tmp, (m * 2 + b) * MS + j * RS + ii);
    }
    __syncthreads();
    for (int idx = tid; idx < n * 4 * N2; idx += nt) {
      const int m = idx / (4 * N2), q = idx % (4 * N2) / N2, i = idx % N2 / NP, ii = idx % NP;
      const int cl = m / nc, r = m - cl * nc, ha = half1(q), b = half2(q);
      const int o = ((4 * cl + q) * nc + r) * MS + i * RS + ii;
      V acc = V::get(Ch, o);
#pragma unroll
      for (int j = 0; j < NP; ++j) acc.fma(t.e(i, ha, j), V::get(tmp, (m * 2 + b) * MS + j * RS + ii));
      acc.put(Ch, o);
    }
    __syncthreads();
  }
  // leaf rows y(beta, alpha) = sum over components, i, j of m1(i, beta) m2(j, alpha) local(i, j)
  const int nb = 1 << (2 * D), dd = c1 * c1, I2 = a.pp1 * a.pp1;
  const double* L = level(D);
  for (int idx = tid; idx < nc * nb * c1 * NP; idx += nt) {
    const int m = idx / NP, j = idx - m * NP, r = m / (nb * c1), cl = m % (nb * c1) / c1, be = m % c1;
    const double* m1 = t.m + (r == 1 && comp == 0 ? NP * c1 : 0) + be;
    V acc;
#pragma unroll
    for (int i = 0; i < NP; ++i) acc.fma(m1[i * c1], V::get(L, (cl * nc + r) * MS + i * RS + j));
    acc.put(tmp, m * RS + j);
  }
  __syncthreads();
  double* y = a.y + S * (static_cast<int64_t>(k) * a.ldx + comp * a.xseg + (static_cast<int64_t>(ctop) << (2 * D)) * dd);
  for (int idx = tid; idx < nb * dd; idx += nt) {
    const int cl = idx / dd, e = idx - cl * dd, el = e / I2, m = e - el * I2;
    int is, it;
    leaf_place(el, a.mcl, is, it);
    const int be = is * a.pp1 + m % a.pp1, al = it * a.pp1 + m / a.pp1;
    V acc;
    for (int r = 0; r < nc; ++r) {
      const double* m2 = t.m + (r == 1 && comp == 1 ? NP * c1 : 0) + al;
#pragma unroll
      for (int j = 0; j < NP; ++j) acc.fma(m2[j * c1], V::get(tmp, ((r * nb + cl) * c1 + be) * RS + j));
    }
    acc.put(y, idx);
  }
}

constexpr size_t TREE_LDS = 128 * 1024;

size_t up_bytes(const TreeArgs& a, int np, int D, bool moment) {
  return sizeof(double) * ((a.cplx ? 2 : 1) * (up_levels(D, a.nc, np * (np | 1)) + up_scratch(D, a.nc, np, a.c1, moment)) +
                           table_doubles(np, a.c1, a.vd));
}
size_t down_bytes(const TreeArgs& a, int np, int D) {
  const int ms = np * (np | 1);
  return sizeof(double) * ((a.cplx ? 2 : 1) * (up_levels(D, a.nc, ms) + down_scratch(D, a.nc, np, a.c1) + a.nc * ms * (a.L - D)) +
                           table_doubles(np, a.c1, a.vd));
}

template <bool C, int NP>
void up(const TreeArgs& a, hipStream_t st) {
  int bot = a.L;
  bool first = true;
  while (true) {
    // leaf level: two levels in one launch where that leaves a workgroup per compute unit, else one
    // (the levels above take a launch in either case); the levels above: three
    const int64_t wg = (static_cast<int64_t>(a.npatch) << (2 * std::max(0, bot - 2))) * a.nrhs * a.vd;
    int D = std::min(bot, first ? (bot <= 2 || wg >= 256 ? 2 : 1) : 3);
    while (D > (first ? 0 : 1) && up_bytes(a, NP, D, first) > TREE_LDS) --D;
    const size_t lds = up_bytes(a, NP, D, first);
    BMI_REQUIRE(lds <= TREE_LDS, BMI_UNSUPPORTED, "leaf clusters too large for the tree kernels");
    const int top = bot - D;
    hipLaunchKernelGGL((k_tree_up<C, NP>), dim3(static_cast<unsigned>(a.npatch << (2 * top)), static_cast<unsigned>(a.nrhs),
                                                static_cast<unsigned>(a.vd)),
                       dim3(256), lds, st, a, top, bot, first ? 1 : 0);
    BMI_CHECK_HIP(hipGetLastError());
    first = false;
    bot = top;
    if (top == 0) break;
  }
}

template <bool C, int NP>
void down(const TreeArgs& a, hipStream_t st) {
  // one launch whatever the depth; one level below a workgroup's cluster (two measured no faster with
  // 384 workgroups left, 24,576 elements, and slower with fewer)
  int D = std::min(a.L, 1);
  while (D > 0 && down_bytes(a, NP, D) > TREE_LDS) --D;
  const size_t lds = down_bytes(a, NP, D);
  BMI_REQUIRE(lds <= TREE_LDS, BMI_UNSUPPORTED, "leaf clusters too large for the tree kernels");
  const int top = a.L - D;
  hipLaunchKernelGGL((k_tree_down<C, NP>), dim3(static_cast<unsigned>(a.npatch << (2 * top)), static_cast<unsigned>(a.nrhs),
                                                static_cast<unsigned>(a.vd)),
                     dim3(256), lds, st, a, top, a.L);
  BMI_CHECK_HIP(hipGetLastError());
}

template <int NP>
void run(const TreeArgs& a, bool upward, hipStream_t st) {
  if (a.cplx)
    upward ? up<true, NP>(a, st) : down<true, NP>(a, st);
  else
    upward ? up<false, NP>(a, st) : down<false, NP>(a, st);
}

}  // namespace

void launch_tree(const TreeArgs& a, bool upward, hipStream_t st) {
  switch (a.np) {
    case 1: return run<1>(a, upward, st);
    case 2: return run<2>(a, upward, st);
    case 3: return run<3>(a, upward, st);
    case 4: return run<4>(a, upward, st);
    case 5: return run<5>(a, upward, st);
    case 6: return run<6>(a, upward, st);
    case 7: return run<7>(a, upward, st);
    case 8: return run<8>(a, upward, st);
    case 9: return run<9>(a, upward, st);
    case 10: return run<10>(a, upward, st);
    case 11: return run<11>(a, upward, st);
    case 12: return run<12>(a, upward, st);
    default: throw Error(BMI_UNSUPPORTED, "Chebyshev nodes out of range");
  }
}

}  // namespace bmi
