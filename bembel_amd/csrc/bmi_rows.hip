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
// Symmetric kernels (PAIR): the block (s, t) is the transpose of (t, s), so one block of each pair is
// read for both products, half the bytes.  A chunk's entries are also laid into LDS (a wave's own tiles)
// and read back with rows and columns exchanged, as the right operand of x_t^T F; the sums over this
// workgroup's rows are complete per chunk and go to the pair's place among the partial sums of s, which
// k_pair_gather adds in a fixed order.  Pairs are listed under either row by parity: under the smaller
// one the first rows have twice the mean and the last none (81 rows, 34,000 pairs: 779 us so, 681 us by
// parity, 886 us reading every block).  Products on an ellipsoid, 9x9 nodes: Helmholtz, 1,536 elements, five
// columns 566 -> 478 us; Maxwell, 1,536 elements, P 2 644 -> 519 us; Helmholtz, 6,144 elements, P 2 1.90 -> 1.31 ms.
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

// orders a wave's LDS writes before its own reads of them
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int PAIR_LD = 18;               // doubles per column of a staged tile: 16 rows, 16-byte reads without conflicts
constexpr int PAIR_TILE = 16 * PAIR_LD;  // one row tile of one plane

template <bool C, typename FT, int RV, int MT, int NT, bool PAIR>
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
  // PAIR: x of the target as the left operand of x_t^T F, lane = column li (complex: Re | Im) of row
  // 4 lk + s of every row tile; rows past the block count as zero
  double x1[PAIR ? MT : 1][4];
  rows_d4 acc2[PL];
  double* stage = red + w * (MT * PL * PAIR_TILE);
  if constexpr (PAIR) {
    const int j = C ? (li & 7) : li;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int i = 4 * lk + s;
        const int row = row0 + (RV == 1 ? 16 * m + i : 16 * RV * (m / RV) + RV * i + m % RV);
        x1[m][s] = row < n && j < a.nrhs ? a.x[xcol[0] + S * (static_cast<int64_t>(cl) * a.xcs + static_cast<int64_t>(row) * a.xrs)]
                                         : 0.0;
      }
  }
  // the wave's blocks: q = p * vd + (column component)
  const int q1 = a.rp[own + 1] * vd;
  int q = a.rp[own] * vd + bw;
  if (k0 >= a.nrhs) q = q1;
  struct Chunk {
    Entry<FT, C ? 2 : RV> f[MT / RV][KU];
    double x[NT][KU];
  };
  const FT* __restrict__ F = static_cast<const FT*>(a.F);
  // the lists in the constant address space: scalar loads, which do not take part in the count of the
  // vector loads below
  typedef const int __attribute__((address_space(4)))* ListPtr;
  const ListPtr src = (ListPtr)(a.src), blk = (ListPtr)(a.blk), slot = (ListPtr)(a.slot);
  const FT* f = nullptr;  // the block being loaded and the source's values
  const double* xs = nullptr;
  auto take = [&](int q2) {
    const int p = vd == 1 ? q2 : q2 / vd, cc = q2 - p * vd;
    f = F + S * ((static_cast<int64_t>(PAIR ? blk[p] : p) * vd + rc) * vd + cc) * a.fblk;
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
        if constexpr (PAIR) {
          double* t = stage + (4 * s + lk) * PAIR_LD + li;
          if constexpr (C || RV == 2) {
            t[2 * g * PAIR_TILE] = !C && last[g] ? v1 : v0;
            t[(2 * g + 1) * PAIR_TILE] = v1;
          } else {
            t[g * PAIR_TILE] = v0;
          }
        }
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
  // PAIR: the chunk's columns of x_t^T F over this slab's rows, complete: lane = column kb + li of
  // right-hand sides 4 v + lk
  auto transposed = [&]() {
    wave_lds_fence();
#pragma unroll
    for (int pl = 0; pl < PL; ++pl) acc2[pl] = rows_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int pl = 0; pl < PL; ++pl) {
        const double2* t = reinterpret_cast<const double2*>(stage + (m * PL + pl) * PAIR_TILE + li * PAIR_LD + 4 * lk);
        const double2 t0 = t[0], t1 = t[1];
        acc2[pl] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1[PAIR ? m : 0][0], t0.x, acc2[pl], 0, 0, 0);
        acc2[pl] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1[PAIR ? m : 0][1], t0.y, acc2[pl], 0, 0, 0);
        acc2[pl] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1[PAIR ? m : 0][2], t1.x, acc2[pl], 0, 0, 0);
        acc2[pl] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1[PAIR ? m : 0][3], t1.y, acc2[pl], 0, 0, 0);
      }
    wave_lds_fence();
  };
  auto store_partial = [&](int p, int kb) {
    const int col = kb + li;
    double* o = a.part + S * ((static_cast<int64_t>(slot[p]) * a.slabs + row0 / (16 * MT)) * a.nrhs * n + col);
#pragma unroll
    for (int v = 0; v < (C ? 2 : 4); ++v) {
      const int j = 4 * v + lk;
      if (4 * v >= a.nrhs) break;
      if (col < n && j < a.nrhs) {
        if constexpr (C)
          *reinterpret_cast<double2*>(o + static_cast<int64_t>(2) * j * n) =
              make_double2(acc2[0][v] - acc2[PL - 1][v + 2], acc2[0][v + 2] + acc2[PL - 1][v]);
        else
          o[static_cast<int64_t>(j) * n] = acc2[0][v];
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
    int kb = 0;              // first column of the chunk loaded last; n: past the end
    int done = -1, kdone = 0;  // PAIR: the chunk whose transposed product waits to be stored
    auto step = [&](const Chunk& now, Chunk& next) {
      const int kn = kb, qn = q;
      kb += 4 * KU;
      if (kb >= n) {
        kb = n;
        if (q + nbw < q1) kb = 0, take(q += nbw);
      }
      load(next, kb);
      // vmcnt(LOADS), the other counters unbounded
      __builtin_amdgcn_s_waitcnt((LOADS & 15) | ((LOADS >> 4) << 14) | 0x0f70);
      if constexpr (PAIR) {
        // stores of the chunk before: behind this wait, which would otherwise wait for them too
        if (done >= 0) store_partial(done, kdone);
      }
      multiply(now, kn);
      if constexpr (PAIR) {
        if (kn < n) transposed();
        done = kn < n ? qn : -1, kdone = kn;
      }
    };
    const int chunks = (q1 - q + nbw - 1) / nbw * ((n + 4 * KU - 1) / (4 * KU));
    take(q);
    load(c0, 0);
    for (int t = 0; t < chunks; t += 2) {
      step(c0, c1);
      step(c1, c0);
    }
    if constexpr (PAIR) {
      if (done >= 0) store_partial(done, kdone);
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

template <bool C, typename FT, int RV, int MT, int NT, bool PAIR>
void launch_rows(const RowsArgs& a, dim3 grid, int nw, hipStream_t st) {
  const int planes = C ? 2 : 1;
  const size_t lds = static_cast<size_t>(nw) * planes * std::max(NT * 256, PAIR ? MT * PAIR_TILE : 0) * sizeof(double);
  hipLaunchKernelGGL((k_block_rows<C, FT, RV, MT, NT, PAIR>), grid, dim3(static_cast<unsigned>(64 * nw)), lds, st, a);
  BMI_CHECK_HIP(hipGetLastError());
}

// thread per (target, column, row): the target's partial sums in slot order
template <bool C>
__global__ __launch_bounds__(256) void k_pair_gather(RowsArgs a, int ng, const int2* __restrict__ gtgt,
                                                     const int* __restrict__ grp) {
  constexpr int S = C ? 2 : 1;
  const int64_t gid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int per = a.nrhs * a.n;
  if (gid >= static_cast<int64_t>(ng) * per) return;
  const int g = static_cast<int>(gid / per), e = static_cast<int>(gid - static_cast<int64_t>(g) * per);
  const int j = e / a.n, row = e - j * a.n;
  const int64_t q0 = static_cast<int64_t>(grp[g]) * a.slabs, q1 = static_cast<int64_t>(grp[g + 1]) * a.slabs;
  const double* p = a.part + S * (q0 * per + e);
  double vr = 0.0, vi = 0.0;
#pragma unroll 4
  for (int64_t q = q0; q < q1; ++q, p += S * per) {
    if constexpr (C) {
      const double2 t = *reinterpret_cast<const double2*>(p);
      vr += t.x, vi += t.y;
    } else {
      vr += p[0];
    }
  }
  const int2 T = gtgt[g];
  const bool second = a.y1 && j >= a.ysplit;
  double* y = (second ? a.y1 : a.y) + S * (a.lvl_off[T.x] * a.yl + static_cast<int64_t>(T.y) * a.ycs +
                                           static_cast<int64_t>(second ? j - a.ysplit : j) * a.yks +
                                           static_cast<int64_t>(row) * a.yrs);
  y[0] += vr;
  if constexpr (C) y[1] += vi;
}

}  // namespace

// row tiles per workgroup: at most six real or three complex ones (registers: two waves per SIMD);
// few targets get workgroups of fewer rows, so that more of the chip takes part
static int rows_tiles(bool cplx, int n, int64_t owners) {
  const int tiles = (n + 15) / 16;
  const int most = cplx ? 3 : 6, unit = cplx || n < 2 ? 1 : 2;
  int slabs = (tiles + most - 1) / most;
  while (owners * slabs < 512 && slabs * unit < tiles) ++slabs;
  const int mt = (tiles + slabs - 1) / slabs;
  return (mt + unit - 1) / unit * unit;
}
int block_rows_slabs(bool cplx, int n, int64_t owners) {
  const int mt = rows_tiles(cplx, n, owners);
  return ((n + 15) / 16 + mt - 1) / mt;
}

void launch_block_rows(bool cplx, bool fp32, RowsArgs a, hipStream_t st) {
  if (a.nown <= 0 || a.nrhs <= 0) return;
  if (a.xl == 0) a.xl = a.nrhs;
  if (a.yl == 0) a.yl = a.nrhs;
  const int ct = block_rows_tile(cplx);
  const int nt = a.nrhs > ct ? 2 : 1;
  const bool pair = a.part != nullptr;
  BMI_REQUIRE(!pair || (nt == 1 && a.vd == 1 && a.tgt && a.n > 1), BMI_INVALID_ARG, "pairs of blocks: one column tile");
  const int64_t owners = static_cast<int64_t>(a.nown) * a.vd;
  const int rv = cplx || a.n < 2 ? 1 : 2;
  const int mt = rows_tiles(cplx, a.n, owners);
  a.slabs = block_rows_slabs(cplx, a.n, owners);
  // column groups of a workgroup share its blocks through the caches; the rest of its waves take
  // blocks in turn
  const int groups = (a.nrhs + nt * ct - 1) / (nt * ct);
  a.ncw = groups >= 4 ? 4 : groups >= 2 ? 2 : 1;
  // (eight waves where their staged tiles fit 64 KB)
  const int nw = owners * a.slabs < 2048 && (!pair || mt * (cplx ? 2 : 1) <= 3) ? 8 : 4;
  const dim3 grid(static_cast<unsigned>(a.nown), static_cast<unsigned>((groups + a.ncw - 1) / a.ncw),
                  static_cast<unsigned>(a.slabs * a.vd));
#define BMI_ROWS(CC, FT, RVV, MTT)                                                        \
  if (cplx == CC && fp32 == std::is_same<FT, float>::value && rv == RVV && mt == MTT) { \
    if (pair)                                                                           \
      launch_rows<CC, FT, RVV, MTT, 1, true>(a, grid, nw, st);                          \
    else if (nt == 1)                                                                   \
      launch_rows<CC, FT, RVV, MTT, 1, false>(a, grid, nw, st);                         \
    else                                                                                \
      launch_rows<CC, FT, RVV, MTT, 2, false>(a, grid, nw, st);                         \
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

void launch_pair_rows(bool cplx, bool fp32, RowsArgs a, const PairSweep& ps, hipStream_t st) {
  if (a.nown <= 0 || a.nrhs <= 0) return;
  a.rp = ps.rp, a.src = ps.src, a.blk = ps.blk, a.slot = ps.slot, a.part = ps.part;
  launch_block_rows(cplx, fp32, a, st);
  if (a.yl == 0) a.yl = a.nrhs;
  a.slabs = block_rows_slabs(cplx, a.n, a.nown);
  const int64_t nt = static_cast<int64_t>(ps.ngather) * a.nrhs * a.n;
  const dim3 grid(static_cast<unsigned>((nt + 255) / 256));
  if (cplx)
    hipLaunchKernelGGL(k_pair_gather<true>, grid, dim3(256), 0, st, a, ps.ngather, ps.gtgt, ps.grp);
  else
    hipLaunchKernelGGL(k_pair_gather<false>, grid, dim3(256), 0, st, a, ps.ngather, ps.gtgt, ps.grp);
  BMI_CHECK_HIP(hipGetLastError());
}

}  // namespace bmi
