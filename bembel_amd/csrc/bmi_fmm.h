// Launchers of the interpolation-FMM kernels (bmi_fmm.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

struct bmi_space;

namespace bmi {

// from this many right-hand sides on, block rows run one wave per owner and 64 columns
constexpr int MULTI_MIN_RHS = 8;

constexpr int CP_STRIDE = 12;  // doubles per cluster node: x(3) kappa ds(3) dt(3) pad(2)

// block rows of up to 64 columns, any block size (bmi_rows.hip): target own (cluster own of one level,
// or tgt[own] = (level, cluster)) takes the blocks rp[own] .. rp[own + 1], each n x n per component
// pair (column stride ld, fblk entries apart, vd x vd of them per entry).  Scalar (row r, column
// k) of cluster c and component m: x[level offset * nrhs + m * xseg + c * xcs + k * xks + r * xrs].
struct RowsArgs {
  int nown, nrhs, n, ld, vd;
  const int2* tgt;
  const int64_t* lvl_off;
  const int* rp;
  const int* src;
  const void* F;
  int64_t fblk;
  const double* x;
  int64_t xseg, xcs, xks, xrs;
  double* y;
  int64_t yseg, ycs, yks, yrs;
  int accumulate;
  int slabs, ncw;  // set by the launch: row slabs, column groups per workgroup
  int xl = 0, yl = 0;            // factors of the level offsets of x and y (0: nrhs)
  const int* order = nullptr;    // the order in which targets are taken (null: as listed)
  double* y1 = nullptr;          // columns from ysplit on go to y1, counted from there
  int ysplit = 0;
  // symmetric pairs (one of the blocks (t, s), (s, t) per entry, vd = 1, columns of one tile): the block
  // of every entry and the place of F^T x_t, which is due to s, among the partial sums
  const int* blk = nullptr;
  const int* slot = nullptr;
  double* part = nullptr;
};
// The lists of a symmetric far field (one block per pair, over every cluster; see RowsArgs) and the targets
// that receive partial sums.
struct PairSweep {
  const int* rp;
  const int* src;
  const int* blk;
  const int* slot;
  double* part;
  int ngather;
  const int2* gtgt;
  const int* grp;
};
// blocks of fewer rows are not paired: with 25 the partial sums of a few columns come near the size of the
// blocks, and four columns gain 3 %
constexpr int PAIR_MIN_ROWS = 36;
// row slabs of a launch: parts of the rows with partial sums of their own
int block_rows_slabs(bool cplx, int n, int64_t owners);
// columns of one tile
constexpr int block_rows_tile(bool cplx) { return cplx ? 8 : 16; }
// scalars of partial sums of one pair
inline int64_t pair_partial(bool cplx, int n, int64_t owners, int cols) {
  return static_cast<int64_t>(block_rows_slabs(cplx, n, owners)) * cols * n;
}
// whether a sweep of cols columns over npairs pairs (n rows, owners clusters) is the faster one: the bytes of the
// blocks that are not read, less three quarters of those of the partial sums, written and read (some stay in the
// caches), are 100 MB or more, the 20 us that the second pass through LDS and the gather take.  Over 191 cases of 36
// to 81 rows, 1 to 16 columns, 384 to 6,144 elements, FP64 and FP32 the pairs it takes are 0.97 to 1.49 times as
// fast as every block and the ones it leaves 0.84 to 1.04: 6,144 elements, 81 rows, one column 861 us by every block,
// 638 by pairs, 16 columns 1,079 and 970; 1,536 elements, 36 rows, 16 columns 166 and 193.
inline bool pairs_pay(bool cplx, bool fp32, int n, int64_t owners, int64_t npairs, int cols) {
  if (n < PAIR_MIN_ROWS || cols > block_rows_tile(cplx)) return false;
  const int64_t S = cplx ? 2 : 1;
  const int64_t blocks = S * n * n * (fp32 ? 4 : 8), partial = 2 * S * 8 * pair_partial(cplx, n, owners, cols);
  return npairs * (4 * blocks - 3 * partial) >= 400 * 1000 * 1000;
}
// the sweep of a's targets from their pairs: block rows, then the partial sums
void launch_pair_rows(bool cplx, bool fp32, RowsArgs a, const PairSweep& ps, hipStream_t st);
void launch_block_rows(bool cplx, bool fp32, RowsArgs a, hipStream_t st);

void launch_cluster_points(const bmi_space* s, int level, int np, const double* d_cheb, double* out,
                           hipStream_t st);
void launch_coupling_assemble(int kind, const int4* d_leaves, int nleaves, int np2,
                              const double* const* d_level_pts, double kre, double kim, double* out,
                              hipStream_t st);
// y = alpha A (x + x2) + beta y with A in CSR; x2 may be null; long_rows: 16 lanes per row
void launch_spmv(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* x,
                 int64_t ldx, double* y, int64_t ldy, const double* alpha, const double* beta, hipStream_t st,
                 const double* x2 = nullptr, bool long_rows = false);
// block sizes whose single columns run one wave per cluster, in two variants
bool wave_leaf_supported(int dd);
bool wave_coupling_supported(int cd);
// variant: 0 = one block per lane group per iteration, 1 = two (chosen by the autotuner)
// Fc/ncoarse: BF16 copies of the first ncoarse blocks (fp32 only); ld: column stride of F (0: cd)
void launch_coupling_apply(bool cplx, bool fp32, int variant, int ntgt, int nrhs, int cd, const int2* tgt,
                           const int* rp, const int* src, const void* F, int64_t fstride, const int64_t* lvl_off,
                           const double* fw, double* bw, hipStream_t st, const unsigned short* Fc = nullptr,
                           int ncoarse = 0, int ld = 0, const PairSweep* pairs = nullptr);
// many right-hand sides: internal vectors with the RHS index fastest (see bmi_fmm.hip)
void launch_spmv_tin(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* X,
                     int64_t ldx, double* Yt, hipStream_t st);
void launch_spmv_tout(bool cplx, int nrows, int nrhs, const int* rp, const int* ci, const double* v, const double* At,
                      const double* Bt, double* Y, int64_t ldy, const double* alpha, const double* beta,
                      hipStream_t st);
// lvl_off: host array of the level offsets
void launch_forward_t(bool cplx, int npatch, int L, int rows, int np2, int dd, int nrhs, const double* mom,
                      const double* T, const double* xs_t, int64_t xseg, double* fw_t, const int64_t* lvl_off,
                      hipStream_t st);
// momt: Mom^T (dd x rows, column-major); Tt: the four T_q transposed
void launch_backward_t(bool cplx, int npatch, int L, int rows, int np2, int dd, int nrhs, const double* momt,
                       const double* Tt, double* bw_t, const int64_t* lvl_off, double* yf_t, int64_t yseg,
                       hipStream_t st);
// block sizes the RHS-fastest sweeps are instantiated for
bool multi_t_supported(bool cplx, int dd, int cd);
bool launch_multi_near_t(bool cplx, bool fp32, int ncl, int nrhs, int dd, const int* rp, const int* src,
                         const void* F, int64_t fstride, int64_t fcomp, const double* xs_t, int64_t xseg,
                         double* ys_t, int64_t yseg, int accumulate, hipStream_t st);
// lvl_off: device array
bool launch_multi_cpl_t(bool cplx, bool fp32, int ntgt, int nrhs, int cd, int ld, const int2* tgt, const int* rp,
                        const int* src, const void* F, int64_t fstride, int64_t fcomp, const int64_t* lvl_off,
                        const double* fw_t, double* bw_t, int accumulate, hipStream_t st);
// column stride of the FP32 coupling copy: cd rounded up to whole 16-byte row vectors
int fp32_coupling_ld(bool cplx, int cd);
void convert_blocks_to_fp32(const double* src, float* dst, int64_t nb, int cd, int ld, bool cplx, hipStream_t st);
// Maxwell far field from the kernel values of each coupling leaf: the four columns (tangent-
// weighted value moments, summed derivative moments) of every cluster entry; one sweep over the
// kernel values, whose four columns of sums take the place of the moments; and both components'
// local expansions from these, in place
void launch_mx_prep(int64_t ne, int nrhs, int np2, int cd, const double* fw0, const double* fw1, const double* tan,
                    double* Z, hipStream_t st);
void launch_mx_coupling(bool fp32, int ntgt_all, int nrhs, int np2, int cd, const int* order, const int2* tgt_all,
                        const int* rp_all, const int* src, const void* K, const int64_t* lvl_off, const double* Z,
                        double* w0, double* w1, const PairSweep* pairs, hipStream_t st);
void launch_mx_finish(int64_t ne, int nrhs, int np2, int cd, const double* tan, double* w0, double* w1, double qre,
                      double qim, hipStream_t st);
void convert_to_bf16(const double* src, unsigned short* dst, int64_t n, hipStream_t st);
// tree transformations of column-major products (bmi_tree.hip).  upward: moments of x at level L and
// transfers up to level 0 into the multipole arrays v0, v1 (vd components of nc np^2 rows; clear: the
// array of local expansions set to zero, or null); downward: local expansions v0, v1 down the tree
// (read only) and the leaf rows y.
struct TreeArgs {
  bool cplx;
  int npatch, L, np, nc, vd, c1, mcl, pp1, nrhs;
  const double* E;  // np x 2 np: E[i * 2 np + h * np + j], polynomial j at node i of half h
  const double* m;  // np x c1 moments of one direction, then (vd 2) their derivative counterparts
  const int64_t* lvl_off;
  double *v0, *v1, *clear;
  const double* x;
  double* y;
  int64_t ldx, xseg;  // column and component strides of x or y
  // upward, one column, one component: x = T xin formed by the bottom launch and written to xs (T in
  // CSR; trp null: x is given)
  const int* trp = nullptr;
  const int* tcol = nullptr;
  const double* tval = nullptr;
  const double* xin = nullptr;
  double* xs = nullptr;
};
void launch_tree(const TreeArgs& a, bool upward, hipStream_t st);
void launch_leaf(bool cplx, int variant, int ncl, int nrhs, int dd, int vd, const int* rp, const int* src,
                 const double* F, const double* xs, int64_t ldxs, int64_t xseg, double* ys, int64_t ldys,
                 int64_t yseg, hipStream_t st);
// near-field sweep and coupling sweep of a single-RHS, single-component product in one launch
// (ys written, bw written); false when no fused kernel exists for these sizes
// near32: the near-field blocks dF are the FP32 copy (with FP32 coupling blocks)
// block sizes with symmetric single-RHS sweeps
bool sym_sweep_supported(bool cplx, int dd, int cd);
// upper half of the coupling blocks of a symmetric kernel, for single-RHS sweeps
struct SymList {
  int ntgt;  // targets with upper blocks, their CSR (sources) and the block index of each entry
  const int2* tgt;
  const int* rp;
  const int* src;
  const int* blk;
  double* part;      // B^T x_t of every entry (S * cd doubles), stored in gather order
  const int* slot;   // per entry: its slot in part
  int ngather;       // targets receiving partials and the ranges of their slots
  const int2* gtgt;
  const int* grp;
  // near-field lists (row clusters of the leaf level as targets of level 0; the diagonal leaf of a
  // cluster has slot -1): their level offsets are one zero
  const int64_t* lvl_off = nullptr;
};

// timing-scope name of the next single-RHS sweep launches on this thread (null: the sweep's own)
extern thread_local const char* tl_sweep_scope;
bool launch_sweep_fused(bool cplx, bool fp32, int leaf_variant, int cpl_variant, int ncl, int dd, const int* drp,
                        const int* dsrc, const void* dF, const double* xs, double* ys, int ntgt, int cd,
                        const int2* tgt, const int* crp, const int* csrc, const void* cF, const int64_t* lvl_off,
                        const double* fw, double* bw, hipStream_t st, const unsigned short* Fc = nullptr,
                        int ncoarse = 0, bool near32 = false, int ld = 0,
                        const SymList* sym = nullptr, const SymList* nsym = nullptr);
// FP32 node tables (offsets from each cluster's node 0, weights; node 0 in FP64) of one level
void launch_fly_points(const double* pts, int ncl, int np2, float4* out, double4* org, hipStream_t st);
// single-RHS sweep of the reduced operator: FP32 near-field blocks, coupling evaluated on the fly
// in FP32 (ys and bw written); false when no kernel exists for these sizes
// variant: near-field blocks loaded per iteration, 0 = one, 1 = two
bool launch_sweep_fly(bool cplx, int variant, int ncl, int dd, const int* drp, const int* dsrc, const float* dF32,
                      const double* xs, double* ys, int ntgt, int cd, const int2* tgt, const int* crp,
                      const int* csrc, const int64_t* lvl_off, const float4* pts, const double4* org,
                      double kre, double kim, const double* fw, double* bw, hipStream_t st);
}  // namespace bmi
