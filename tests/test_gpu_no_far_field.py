"""Products of operators without a far field: the six clusters of 24 elements have no admissible pair, so every
block is a near-field leaf.  All columns and precisions against the dense matrix assembled from the
same pairs (sums of 600 terms at most in another order, 1e-12 as the other parity tests; the FP32 leaves of the
reduced operator of a mixed handle within 2e-7)."""
import numpy as np
import pytest

import bembel_amd as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,P,n_cheb", [("laplace", 1, 4), ("laplace", 2, 9), ("helmholtz", 1, 4), ("helmholtz", 2, 5),
                                           ("maxwell", 1, 4)])
@pytest.mark.parametrize("precision", [B.FP64, B.MIXED, B.MIXED_BF16])
def test_gpu_products_without_far_field(gpu, kind, P, n_cheb, precision):
    op = {"laplace": B.LaplaceSingleLayerOperator, "helmholtz": B.HelmholtzSingleLayerOperator,
          "maxwell": B.MaxwellSingleLayerOperator}[kind]()
    if kind != "laplace":
        op.set_wavenumber(2.5 - 0.3j)
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), 1, P, op)
    H = B.H2Matrix(ps, op, n_cheb=n_cheb, precision=precision)
    assert (H.leaves()[:, 0] == 2).all()  # dense leaves only
    A = np.asarray(B.DenseMatrix(ps, op).matrix)
    rng = np.random.default_rng(1)
    X = rng.uniform(-1, 1, (len(A), 20))
    if kind != "laplace":
        X = X + 1j * rng.uniform(-1, 1, X.shape)
    for cols in (1, 2, 7, 8, 20):
        Y = H @ (X[:, 0] if cols == 1 else X[:, :cols])
        want = A @ (X[:, 0] if cols == 1 else X[:, :cols])
        e = np.linalg.norm(Y - want) / np.linalg.norm(want)
        assert e <= (1e-12 if precision == B.FP64 else 2e-7), (cols, e)
