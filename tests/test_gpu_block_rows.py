"""Block-row sweeps (bmi_rows.hip) at the edges of their tiles: products with several columns, and
single columns of block sizes without a kernel of their own, against the oracle.

Block sizes: coupling blocks of n_cheb^2 rows (1, 4, 9, ..., 81: one row, below, at and past whole
16-row tiles and 4-column steps), near-field leaves of 4^min_cluster_level (P + 1)^2 rows.  Columns:
one, and below, at and past the 8 (complex) and 16 (real) columns of a tile and the column groups.
The products sum the same terms as the oracle in another order: 1e-12 relative, as the other
parity tests.
"""
import numpy as np
import pytest

import bembel_amd as B
import oracle_lib as O

pytestmark = pytest.mark.gpu


def _pair(op_name, M, P, n_cheb, mcl=1, precision=B.FP64):
    op = B.LaplaceSingleLayerOperator() if op_name == "laplace" else B.HelmholtzSingleLayerOperator()
    kappa = 0j if op_name == "laplace" else 2.5 - 0.3j
    op.set_wavenumber(kappa)
    ps = B.AnsatzSpace(B.Geometry(), M, P, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, min_cluster_level=mcl, precision=precision)
    kind = O.LAPLACE if op_name == "laplace" else O.HELMHOLTZ
    oh = O.H2(O.Space(O.Geometry(), M, P), kind, kappa, n_cheb, mcl=mcl)
    return H, oh, ps.number_of_dofs, op.scalar


def _columns(n, cols, scalar, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, cols))
    return x if scalar == np.float64 else x + 1j * rng.uniform(-1, 1, (n, cols))


def _check(H, oh, n, scalar, cols, tol=1e-12):
    X = _columns(n, max(cols), scalar, 5)
    ref = oh.matvec(X)
    for c in cols:
        Y = H @ X[:, :c]
        e = np.linalg.norm(Y - ref[:, :c]) / np.linalg.norm(ref[:, :c])
        assert e <= tol, (c, e)


@pytest.mark.parametrize("op", ["laplace", "helmholtz"])
@pytest.mark.parametrize("P,n_cheb", [(1, 1), (2, 2), (1, 3), (1, 4), (2, 5), (2, 6), (1, 7), (2, 9), (1, 11)])
def test_gpu_block_rows_sizes(gpu, op, P, n_cheb):
    H, oh, n, scalar = _pair(op, 3, P, n_cheb)
    _check(H, oh, n, scalar, (1, 2, 5))


@pytest.mark.parametrize("op", ["laplace", "helmholtz"])
@pytest.mark.parametrize("P,mcl", [(1, 0), (2, 0), (1, 2), (2, 2)])
def test_gpu_block_rows_leaf_sizes(gpu, op, P, mcl):
    H, oh, n, scalar = _pair(op, 3, P, 4, mcl)
    _check(H, oh, n, scalar, (1, 3))


@pytest.mark.parametrize("op", ["laplace", "helmholtz"])
@pytest.mark.parametrize("n_cheb", [4, 9])
def test_gpu_block_rows_columns(gpu, op, n_cheb):
    H, oh, n, scalar = _pair(op, 2, 2, n_cheb)
    _check(H, oh, n, scalar, (1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 65, 130))


@pytest.mark.parametrize("op", ["laplace", "helmholtz"])
def test_gpu_block_rows_fp32_blocks(gpu, op):
    # FP32 copies of the coupling blocks, columns padded to whole vectors: 1e-8 from the FP64 operator
    H, oh, n, scalar = _pair(op, 3, 1, 9, precision=B.MIXED)
    _check(H, oh, n, scalar, (1, 3, 20), tol=1e-6)


@pytest.mark.parametrize("precision", [B.FP64, B.MIXED])
@pytest.mark.parametrize("n_cheb", [2, 5, 9])
def test_gpu_block_rows_maxwell_columns(gpu, n_cheb, precision):
    # four columns of kernel sums per right-hand side, in two halves: the columns of a product are
    # those of single products (the same sums over the same blocks), against the oracle in test_gpu_maxwell
    op = B.MaxwellSingleLayerOperator()
    op.set_wavenumber(2.0 - 0.1j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), 3, 1, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, precision=precision)
    X = _columns(ps.number_of_dofs, 5, op.scalar, 7)
    one = np.stack([H @ X[:, k] for k in range(5)], 1)
    for c in (2, 3, 5):
        assert np.linalg.norm(H @ X[:, :c] - one[:, :c]) <= 1e-13 * np.linalg.norm(one[:, :c]), c


@pytest.mark.parametrize("precision", [B.FP64, B.MIXED])
@pytest.mark.parametrize("kind,P,n_cheb", [("laplace", 1, 6), ("laplace", 2, 7), ("helmholtz", 1, 6), ("helmholtz", 2, 9),
                                           ("maxwell", 1, 6), ("maxwell", 1, 9)])
def test_gpu_block_rows_pairs(gpu, kind, P, n_cheb, precision):
    # one block of each symmetric pair against every block: the same terms summed in another order, and
    # the two weights of a coupling entry multiplied in the other order (an ulp of the entry).  Columns up
    # to the tile and past it; the workspace first grown by a product that does not use pairs
    op = {"laplace": B.LaplaceSingleLayerOperator, "helmholtz": B.HelmholtzSingleLayerOperator,
          "maxwell": B.MaxwellSingleLayerOperator}[kind]()
    if kind != "laplace":
        op.set_wavenumber(2.0 - 0.1j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), 3, P, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, precision=precision)
    X = _columns(ps.number_of_dofs, 20, op.scalar, 11)
    for c in (20, 1, 2, 3, 7):
        H.set_sweep(None)
        got = H @ X[:, :c]
        again = H @ X[:, :c]
        H.set_sweep("full")
        want = H @ X[:, :c]
        assert np.array_equal(got, again), c
        tol = 1e-13 if precision == B.FP64 else 1e-6
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), c


# Row tiles of a workgroup by rows and clusters: real 2 (36 and 64 rows, 510 clusters), 4 (81 rows, 510; 36, 2,046) and 6
# (81 rows, 2,046), complex 1 (64 rows, 126), 2 (36 rows, 510) and 3 (81 rows, 510; 36 rows, 2,046); one to four row slabs
@pytest.mark.parametrize("kind,M,n_cheb,paired", [
    ("laplace", 4, 6, (1,)), ("laplace", 4, 8, (1, 8, 9)), ("laplace", 4, 9, (1, 3, 12)), ("laplace", 5, 6, (1, 8, 9, 15, 16)),
    ("laplace", 5, 9, (1, 9, 16)), ("helmholtz", 3, 8, (1,)), ("helmholtz", 4, 6, (1, 2, 3)),
    ("helmholtz", 4, 9, (1, 5, 7, 8)), ("helmholtz", 5, 6, (1, 7, 8)), ("maxwell", 4, 6, (1,)), ("maxwell", 4, 9, (1, 2))])
def test_gpu_block_rows_pair_tiles(gpu, kind, M, n_cheb, paired):
    # as above, the workspace growing from product to product; a product that reads every block gives the bits of
    # the forced one, and one column past the tile does
    op = {"laplace": B.LaplaceSingleLayerOperator, "helmholtz": B.HelmholtzSingleLayerOperator,
          "maxwell": B.MaxwellSingleLayerOperator}[kind]()
    if kind != "laplace":
        op.set_wavenumber(2.0 - 0.1j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), M, 1, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb)
    past = {"laplace": 17, "helmholtz": 9, "maxwell": 3}[kind]
    X = _columns(ps.number_of_dofs, past, op.scalar, 13)
    for c in paired + (past,):
        H.set_sweep(None)
        got = H @ X[:, :c]
        H.set_sweep("full")
        want = H @ X[:, :c]
        assert np.array_equal(got, want) == (c == past), c
        assert np.linalg.norm(got - want) <= 1e-13 * np.linalg.norm(want), c


@pytest.mark.parametrize("kind,M,n_cheb,precision,cols", [
    ("laplace", 3, 6, B.FP64, (1, 4, 16)), ("laplace", 4, 6, B.FP64, (12, 16)), ("laplace", 4, 6, B.MIXED, (2, 4, 16)),
    ("helmholtz", 4, 6, B.MIXED, (4, 8)), ("helmholtz", 3, 7, B.FP64, (2, 8)), ("maxwell", 3, 6, B.FP64, (1, 2))])
def test_gpu_block_rows_pairs_that_do_not_pay(gpu, kind, M, n_cheb, precision, cols):
    # few or small pairs, many columns, FP32 blocks: partial sums and gather cost more than the blocks saved
    op = {"laplace": B.LaplaceSingleLayerOperator, "helmholtz": B.HelmholtzSingleLayerOperator,
          "maxwell": B.MaxwellSingleLayerOperator}[kind]()
    if kind != "laplace":
        op.set_wavenumber(2.0 - 0.1j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), M, 1, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, precision=precision)
    X = _columns(ps.number_of_dofs, max(cols), op.scalar, 13)
    for c in cols:
        H.set_sweep(None)
        got = H @ X[:, :c]
        H.set_sweep("full")
        assert np.array_equal(got, H @ X[:, :c]), c


@pytest.mark.parametrize("kind,precision,n_cheb,cols,sums", [
    ("laplace", B.FP64, 9, (17, 12, 1), (0, 12, 12)), ("laplace", B.FP64, 9, (1, 12, 17), (1, 12, 12)),
    ("laplace", B.FP64, 6, (16, 1), (0, 1)), ("laplace", B.MIXED, 6, (1,), (0,)), ("helmholtz", B.MIXED, 9, (9, 4), (0, 4)),
    ("maxwell", B.FP64, 9, (3, 2), (0, 2))])
def test_gpu_partial_sums_held(gpu, kind, precision, n_cheb, cols, sums):
    # a handle holds partial sums for the largest product that used them, and none for others; the estimate
    # counts those of its product
    op = {"laplace": B.LaplaceSingleLayerOperator, "helmholtz": B.HelmholtzSingleLayerOperator,
          "maxwell": B.MaxwellSingleLayerOperator}[kind]()
    if kind != "laplace":
        op.set_wavenumber(2.0 - 0.1j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), 4, 1, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, precision=precision)
    S = 1 if kind == "laplace" else 2
    vd = 2 if kind == "maxwell" else 1
    clusters, pairs = 510, int((H.leaves()[:, 0] != 2).sum()) // 2

    def held():
        info = np.zeros(16, dtype=np.int64)
        B._check(B.library().bmi_h2_info(H._h, info.ctypes.data_as(B.C.POINTER(B.C.c_int64))))
        return int(info[8])

    def workspace(c):  # three super vectors, multipole and local coefficients, Maxwell's four columns
        coefficients = clusters * n_cheb ** 2 * vd
        return 8 * S * c * (3 * ps.number_of_super_dofs + (vd + 1) * coefficients + (2 * coefficients if vd == 2 else 0))

    base, most = held(), 0
    X = _columns(ps.number_of_dofs, max(cols), op.scalar, 3)
    for c, s in zip(cols, sums):
        H @ X[:, :c]
        most = max(most, c)
        partial = 8 * S * pairs * 2 * s * (4 if kind == "maxwell" else 1) * n_cheb ** 2  # two row slabs
        assert held() - base - workspace(most) == partial, (c, held() - base - workspace(most), partial)
        d = op.desc(n_cheb=n_cheb, eta=1.6, min_cluster_level=1, precision=precision)
        est = np.zeros(1, dtype=np.int64)
        B._check(B.library().bmi_h2_estimate_bytes(ps._h, B.C.byref(d), c,
                                                   est.ctypes.data_as(B.C.POINTER(B.C.c_int64))))
        if c == cols[0]:
            assert 1.0 <= est[0] / held() <= 1.05, c
