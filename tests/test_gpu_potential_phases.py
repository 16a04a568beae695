"""Potentials where the phases kappa r leave the range of the two-part reduction, and where a target
meets a source or lies beyond the range of r^2.

The kernel chooses its sine and cosine for 256 targets and 256 sources at a time from |x| and |y|: a
target far away moves its neighbours in the call to the general form, with and without which they must
agree (both within 3e-16 per sine; the sums of up to 1,536 sources with signs within 1e-12 of the
largest value).  Values themselves are compared with the oracle in test_gpu_potential.py, their rounding
with extended precision here.
"""
import numpy as np
import pytest

import bembel_amd as B
import extended_lib as X
import oracle_lib as O

pytestmark = pytest.mark.gpu


def _potential(kind, kappa):
    op = B.MaxwellSingleLayerOperator() if kind == "maxwell" else B.LaplaceSingleLayerOperator()
    ps = B.AnsatzSpace(B.Geometry(scale=(1.0, 0.7, 0.5)), 2, 1, op)
    pot = {"laplace": B.LaplaceSingleLayerPotential, "helmholtz": B.HelmholtzSingleLayerPotential,
           "maxwell": B.MaxwellSingleLayerPotential}[kind]()
    pot.set_wavenumber(kappa)
    dp = B.DiscretePotential(pot, ps)
    rng = np.random.default_rng(3)
    n = ps.number_of_dofs
    rho = rng.uniform(-1, 1, n)
    dp.set_cauchy_data(rho if kind == "laplace" else rho + 1j * rng.uniform(-1, 1, n))
    return dp


@pytest.mark.parametrize("kind", ["helmholtz", "maxwell"])
@pytest.mark.parametrize("kappa", [3.0, 3.0 - 0.2j, -2.0])
def test_gpu_potential_far_target_leaves_its_neighbours(gpu, kind, kappa):
    dp = _potential(kind, complex(kappa))
    pts = np.random.default_rng(5).uniform(1.2, 2.0, (300, 3))  # two blocks of targets, the second ragged
    near = np.asarray(dp.evaluate(pts))
    for at in (0, 255, 299):
        p = pts.copy()
        p[at] = (0.0, 1e6, 0.0)
        got = np.asarray(dp.evaluate(p))
        keep = np.arange(300) != at
        assert np.isfinite(got).all() or np.imag(kappa) != 0
        assert np.abs(got[keep] - near[keep]).max() <= 1e-12 * np.abs(near).max(), at


def test_gpu_laplace_potential_beyond_the_range(gpu):
    dp = _potential("laplace", 0j)
    got = np.asarray(dp.evaluate(np.array([[1e200, 0.0, 0.0], [2.0, 0.0, 0.0]])))
    assert got[0] == 0.0 and np.isfinite(got[1]) and got[1] != 0.0  # r^2 overflows: 1 / r is 0


def _sphere_sum(T, pts, sup, elements, kappa, M):
    """The Helmholtz potential at pts of a P = 1 density (element functions' coefficients sup, four per
    element) with numpy in the type T, every operation rounded once: the 3 x 3 Gauss points of each element
    as sources."""
    x, w = X.gauss(3, T)
    Y, area = X.sphere_points(T, elements, M, x)
    b = X.linear(x)
    rho = np.einsum("eyx,ux,vy->euv", sup.reshape(-1, 2, 2), b, b)
    q = (rho * (area * w[:, None] * w[None, :])).reshape(-1)
    d = pts.astype(T)[:, None, :] - Y.reshape(1, -1, 3)
    r = np.sqrt((d ** 2).sum(-1))
    four_pi = 4 * (T(4) * np.arctan(T(1)))
    K = (np.cos(T(kappa) * r) - 1j * np.sin(T(kappa) * r)) / r / four_pi
    return (K * q).sum(-1)


@pytest.mark.parametrize("kappa", [8.0, 16.0])
def test_gpu_potential_rounds_as_its_operations(gpu, kappa):
    # few sources (864), where the phases carry most of the error: the distance to extended precision is that of
    # pairwise sums in doubles whose roots, sines and quotients are rounded once.  An eighth more is left for the
    # running sums over 64 sources (2 roundings of 2^-53 / sqrt(3) a source at the size of a partial sum, about
    # 2.5e-16 of the result here, beside 6.4e-16 and 25e-16 of the plain sums).  Roots within two ulps and
    # running sums over 256 sources were at 1.49 and 1.21 times the plain sums.
    if not X.HAS_EXTENDED:
        pytest.skip("no extended precision on this host")
    M = 2
    op = B.HelmholtzSingleLayerOperator()
    ps = B.AnsatzSpace(B.Geometry(), M, 1, op)
    rng = np.random.default_rng(11)
    rho = rng.uniform(-1, 1, ps.number_of_dofs) + 1j * rng.uniform(-1, 1, ps.number_of_dofs)
    d = rng.normal(size=(2000, 3))
    pts = d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(2, 4, (2000, 1))
    pot = B.HelmholtzSingleLayerPotential()
    pot.set_wavenumber(complex(kappa))
    dp = B.DiscretePotential(pot, ps)
    dp.set_cauchy_data(rho)
    got = np.asarray(dp.evaluate(pts))
    rp, col, val = O.Space(O.Geometry(), M, 1).T()
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))

    def total(T):
        sup = np.zeros(len(rp) - 1, dtype=np.result_type(T, np.complex128))
        np.add.at(sup, rows, val.astype(T) * rho[col])
        return _sphere_sum(T, pts, sup, ps.elements(), kappa, M)

    exact = total(np.longdouble)

    def error(y):
        return float(np.linalg.norm(y - exact) / np.linalg.norm(exact))

    print("error here", error(got), "of plain sums", error(total(np.float64)))
    assert error(got) <= 1.125 * error(total(np.float64))
