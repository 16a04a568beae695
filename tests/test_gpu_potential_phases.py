"""Potentials where the phases kappa r leave the range of the two-part reduction, and where a target
meets a source or lies beyond the range of r^2.

The kernel chooses its sine and cosine for 256 targets and 256 sources at a time from |x| and |y|: a
target far away moves its neighbours in the call to the general form, with and without which they must
agree (both within 3e-16 per sine; the sums of up to 1,536 sources with signs within 1e-12 of the
largest value).  Values themselves are compared with the oracle in test_gpu_potential.py.
"""
import numpy as np
import pytest

import bembel_amd as B

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
