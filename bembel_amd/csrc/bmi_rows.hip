// Block-row sweeps of few right-hand sides, for blocks of any size: y_t (+)= sum_p F_p x_src(p) for
// the targets t of a CSR list, up to 64 columns, on the FP64 matrix cores.
//
// Bound: every block is read once from HBM.  v_mfma_f64_16x16x4f64 takes 64 block entries (512
// bytes) against up to 16 real columns in 64 cycles of a SIMD, 19.6 TB/s over the chip, so the
// matrix pipe stays ahead of memory however few of the 16 columns are used, and all columns of a
// tile cost one pass over the blocks.  Complex blocks use the 16 columns as [Re x | Im x] of 8
// right-hand sides: two products per tile (real and imaginary plane of F), combined at the end.
//
// Layout: a wave reads its block entries straight into the A operand (no LDS: each entry is used
// by one wave only): lane li + 16 lk holds row 16 m + li of column 4 s + lk, so the lanes of a load
// read four consecutive columns, 128 to 256 bytes each; real blocks load two rows per lane (16
// bytes), which the tiles 2g and 2g + 1 hold.  The next four column steps are loaded while the
// current ones are multiplied.  The waves of a workgroup share one target: they take its blocks in
// turn (or, with more than one column tile, different columns of the same blocks, so that these
// come from the caches), and their sums are added in wave order through LDS: the same bits on
// every run.
//
// Measured against one thread per row (generic sizes) and one wave per target (16 and 25 rows, two
// complex columns per pass): Laplace product, 6,144 elements, 9x9 nodes, one column 2160 -> 954 us;
// Helmholtz product, 1,536 elements, P 1, 9x9 nodes, five columns 2469 -> 735 us; Helmholtz GMRES
// of six columns, 384 elements, 5x5 nodes 157 -> 45 ms (coupling sweep 357 -> 20 us a product).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bmi_fmm.h"
#include "bmi_internal.h"

namespace bmi {

namespace {

typedef double rows_d4 __attribute__((ext_vector_type(4)));

// N neighbouring values, loaded together at the alignment of one (odd column strides)
template <typename FT, int N>
struct Entry {
  FT v[N];
  __device__ void load(const FT* p) { __builtin_memcpy(v, p, sizeof(v)); }
};

template <bool C, typename FT, int RV, int MT, int NT>
__global__ __launch_bounds__(512) void k_block_rows(RowsArgs a) {
  constexpr int S = C ? 2 : 1, PL = C ? 2 : 1;
  constexpr int CT = C ? 8 : 16;  // right-hand sides per column tile
  constexpr int KU = 4;           // column steps (of four columns) per chunk
  // RV: rows per load (two for real blocks; one for complex entries and blocks of a single row)
  static_assert(MT % RV == 0 && RV <= (C ? 1 : 2), "whole row groups");
  extern __shared__ double red[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int nw = static_cast<int>(blockDim.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int ncw = a.ncw, nbw = nw / ncw;
  const int cw = w % ncw, bw = w / ncw;
  const int n = a.n, ld = a.ld, vd = a.vd;
  const int k0 = (static_cast<int>(blockIdx.y) * ncw + cw) * (NT * CT);
  const int rc = static_cast<int>(blockIdx.z) / a.slabs;
  const int row0 = (static_cast<int>(blockIdx.z) - rc * a.slabs) * (16 * MT);
  const int own = a.order ? a.order[blockIdx.x] : static_cast<int>(blockIdx.x);
  int64_t lo = 0, ylo = 0;  // level offsets
  int cl = own;
  if (a.tgt) {
    const int2 T = a.tgt[own];
    cl = T.y;
    lo = a.lvl_off[T.x] * a.xl, ylo = a.lvl_off[T.x] * a.yl;
  }
  // first row of this lane in every row group, moved back where its load would pass the last row
  int rb[MT / RV];
  bool last[MT / RV];  // the pair was moved back by one: its first row is the load's second value
#pragma unroll
  for (int g = 0; g < MT / RV; ++g) {
    const int r = row0 + 16 * RV * g + RV * li;
    rb[g] = r < n - RV ? r : n - RV;
    last[g] = RV == 2 && r == n - 1;
  }
  // this lane's column of x in every column tile (columns past the last right-hand side repeat it)
  int64_t xcol[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) {
    const int j = k0 + u * CT + (C ? (li & 7) : li);
    xcol[u] = S * (lo + static_cast<int64_t>(j < a.nrhs ? j : a.nrhs - 1) * a.xks) + (C ? (li >> 3) : 0);
  }
  rows_d4 acc[PL][MT][NT];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int u = 0; u < NT; ++u) acc[p][m][u] = rows_d4{0.0, 0.0, 0.0, 0.0};
  // the wave's blocks: q = p * vd + (column component)
  const int q1 = a.rp[own + 1] * vd;
  int q = a.rp[own] * vd + bw;
  if (k0 >= a.nrhs) q = q1;
  struct Chunk {
    Entry<FT, C ? 2 : RV> f[MT / RV][KU];
    double x[NT][KU];
  };
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  // the sources in the constant address space: scalar loads, which do not take part in the count of the
  // vector loads below
  typedef const int __attribute__((address_space(4)))* SrcPtr;
  const SrcPtr src = (SrcPtr)(a.src);
  const FT* f = nullptr;  // the block being loaded and the source's values
  const double* xs = nullptr;
  auto take = [&](int q2) {
    const int p = vd == 1 ? q2 : q2 / vd, cc = q2 - p * vd;
    f = F + S * ((static_cast<int64_t>(p) * vd + rc) * vd + cc) * a.fblk;
    xs = a.x + S * (cc * a.xseg + static_cast<int64_t>(src[p]) * a.xcs);
  };
  auto load = [&](Chunk& c, int kb) {
#pragma unroll
    for (int s = 0; s < KU; ++s) {
      const int k = kb + 4 * s + lk;
      const int kk = k < n ? k : n - 1;
#pragma unroll
      for (int g = 0; g < MT / RV; ++g) c.f[g][s].load(f + S * (kk * ld + rb[g]));
#pragma unroll
      for (int u = 0; u < NT; ++u) c.x[u][s] = xs[xcol[u] + static_cast<int64_t>(kk) * (S * a.xrs)];
    }
  };
  auto multiply = [&](const Chunk& c, int kb) {
#pragma unroll
    for (int s = 0; s < KU; ++s) {
      if (kb + 4 * s >= n) break;
      const bool in = kb + 4 * s + lk < n;  // columns past the block count as zero
      double xv[NT];
#pragma unroll
      for (int u = 0; u < NT; ++u) xv[u] = in ? c.x[u][s] : 0.0;
#pragma unroll
      for (int g = 0; g < MT / RV; ++g) {
        const double v0 = in ? static_cast<double>(c.f[g][s].v[0]) : 0.0;
        double v1 = 0.0;
        if constexpr (C || RV == 2) v1 = in ? static_cast<double>(c.f[g][s].v[1]) : 0.0;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          if constexpr (C) {
            acc[0][g][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(v0, xv[u], acc[0][g][u], 0, 0, 0);
            acc[PL - 1][g][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, xv[u], acc[PL - 1][g][u], 0, 0, 0);
          } else {
            acc[0][RV * g][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(last[g] ? v1 : v0, xv[u], acc[0][RV * g][u], 0, 0, 0);
            if constexpr (RV == 2)
              acc[0][2 * g + 1][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(v1, xv[u], acc[0][2 * g + 1][u], 0, 0, 0);
          }
        }
      }
    }
  };
  if (q < q1) {
    // Two chunks in turn: the loads of one are in flight while the other is multiplied.  They are issued
    // without a condition (past the last chunk: its columns again, counted as zero), and each chunk is
    // waited for by the number of the loads after it: behind a branch, or with steps of a chunk left out,
    // the compiler's waits hold for every path and end up waiting for the loads just issued (Laplace
    // product, 6,144 elements, 9x9 nodes: 792 -> 753 us; the sweep reads 5.3 TB/s).
    constexpr int LOADS = KU * (MT / RV + NT);
    static_assert(LOADS < 64, "loads of a chunk within the counter");
    Chunk c0, c1;
    int kb = 0;  // first column of the chunk loaded last; n: past the end
    auto step = [&](const Chunk& now, Chunk& next) {
      const int kn = kb;
      kb += 4 * KU;
      if (kb >= n) {
        kb = n;
        if (q + nbw < q1) kb = 0, take(q += nbw);
      }
      load(next, kb);
      // vmcnt(LOADS), the other counters unbounded
      __builtin_amdgcn_s_waitcnt((LOADS & 15) | ((LOADS >> 4) << 14) | 0x0f70);
      multiply(now, kn);
    };
    const int chunks = (q1 - q + nbw - 1) / nbw * ((n + 4 * KU - 1) / (4 * KU));
    take(q);
    load(c0, 0);
    for (int t = 0; t < chunks; t += 2) {
      step(c0, c1);
      step(c1, c0);
    }
  }
  // sums over the waves of a column group, one row tile at a time: tile entry (row 4 v + lk, column
  // li) of plane p and column tile u of wave w at red[((w * PL + p) * NT + u) * 256 + row * 16 + li]
  for (int m = 0; m < MT; ++m) {
    __syncthreads();
#pragma unroll
    for (int mm = 0; mm < MT; ++mm)
      if (mm == m) {
#pragma unroll
        for (int p = 0; p < PL; ++p)
#pragma unroll
          for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              red[((w * PL + p) * NT + u) * 256 + (4 * v + lk) * 16 + li] = acc[p][mm][u][v];
      }
    __syncthreads();
    const int per = 16 * CT * NT;  // (row, right-hand side) of one column group
    for (int e = static_cast<int>(threadIdx.x); e < per * ncw; e += static_cast<int>(blockDim.x)) {
      const int g = e / per, r = e - g * per;
      const int i = r & 15, jl = r >> 4;
      const int u = jl / CT, jj = jl - u * CT;
      const int j = (static_cast<int>(blockIdx.y) * ncw + g) * (NT * CT) + jl;
      const int row = row0 + (RV == 1 ? 16 * m + i : 16 * RV * (m / RV) + RV * i + m % RV);
      if (j >= a.nrhs || row >= n) continue;
      double vr = 0.0, vi = 0.0;
      for (int b = 0; b < nbw; ++b) {
        const double* t = red + ((b * ncw + g) * PL * NT + u) * 256 + i * 16 + jj;
        if constexpr (C) {
          vr += t[0] - t[NT * 256 + 8];
          vi += t[8] + t[NT * 256];
        } else {
          vr += t[0];
        }
      }
      const bool second = a.y1 && j >= a.ysplit;
      double* y = (second ? a.y1 : a.y) + S * (ylo + rc * a.yseg + static_cast<int64_t>(cl) * a.ycs +
                                               static_cast<int64_t>(second ? j - a.ysplit : j) * a.yks +
                                               static_cast<int64_t>(row) * a.yrs);
      if (a.accumulate) {
        vr += y[0];
        if constexpr (C) vi += y[1];
      }
      y[0] = vr;
      if constexpr (C) y[1] = vi;
    }
  }
}

template <bool C, typename FT, int RV, int MT, int NT>
void launch_rows(const RowsArgs& a, dim3 grid, int nw, hipStream_t st) {
  const size_t lds = static_cast<size_t>(nw) * (C ? 2 : 1) * NT * 256 * sizeof(double);
  hipLaunchKernelGGL((k_block_rows<C, FT, RV, MT, NT>), grid, dim3(static_cast<unsigned>(64 * nw)), lds, st, a);
  BMI_CHECK_HIP(hipGetLastError());
}

}  // namespace

void launch_block_rows(bool cplx, bool fp32, RowsArgs a, hipStream_t st) {
  if (a.nown <= 0 || a.nrhs <= 0) return;
  if (a.xl == 0) a.xl = a.nrhs;
  if (a.yl == 0) a.yl = a.nrhs;
  const int tiles = (a.n + 15) / 16;
  const int ct = cplx ? 8 : 16;
  const int nt = a.nrhs > ct ? 2 : 1;
  // row tiles per workgroup: at most six real or three complex ones (registers: two waves per SIMD);
  // few targets get workgroups of fewer rows, so that more of the chip takes part
  const int rv = cplx || a.n < 2 ? 1 : 2;
  const int most = cplx ? 3 : 6, unit = rv;
  int slabs = (tiles + most - 1) / most;
  const int64_t owners = static_cast<int64_t>(a.nown) * a.vd;
  while (owners * slabs < 512 && slabs * unit < tiles) ++slabs;
  int mt = (tiles + slabs - 1) / slabs;
  mt = (mt + unit - 1) / unit * unit;
  a.slabs = (tiles + mt - 1) / mt;
  // column groups of a workgroup share its blocks through the caches; the rest of its waves take
  // blocks in turn
  const int groups = (a.nrhs + nt * ct - 1) / (nt * ct);
  a.ncw = groups >= 4 ? 4 : groups >= 2 ? 2 : 1;
  const int nw = owners * a.slabs < 2048 ? 8 : 4;
  const dim3 grid(static_cast<unsigned>(a.nown), static_cast<unsigned>((groups + a.ncw - 1) / a.ncw),
                  static_cast<unsigned>(a.slabs * a.vd));
#define BMI_ROWS(CC, FT, RVV, MTT)                                                        \
  if (cplx == CC && fp32 == std::is_same<FT, float>::value && rv == RVV && mt == MTT) { \
    if (nt == 1)                                                                        \
      launch_rows<CC, FT, RVV, MTT, 1>(a, grid, nw, st);                                \
    else                                                                                \
      launch_rows<CC, FT, RVV, MTT, 2>(a, grid, nw, st);                                \
    return;                                                                             \
  }
  BMI_ROWS(false, double, 1, 1)
  BMI_ROWS(false, float, 1, 1)
  BMI_ROWS(false, double, 2, 2)
  BMI_ROWS(false, double, 2, 4)
  BMI_ROWS(false, double, 2, 6)
  BMI_ROWS(false, float, 2, 2)
  BMI_ROWS(false, float, 2, 4)
  BMI_ROWS(false, float, 2, 6)
  BMI_ROWS(true, double, 1, 1)
  BMI_ROWS(true, double, 1, 2)
  BMI_ROWS(true, double, 1, 3)
  BMI_ROWS(true, float, 1, 1)
  BMI_ROWS(true, float, 1, 2)
  BMI_ROWS(true, float, 1, 3)
#undef BMI_ROWS
  throw Error(BMI_UNSUPPORTED, "no block-row sweep of this tile count");
}

}  // namespace bmi
