"""Near-field rules over the quadrature degrees and rotations they meet: the chunks of outer coordinates,
lanes per unit and odd inner ranges of the factorised rules change with the number of points per
direction, and every rotation of the edge rule has its own code.

Every pair of the 24-element ellipsoid (all rotations, also across patches), and sampled touching and
near pairs of finer meshes (6 to 13 points per direction) equal the oracle to 1e-12 (the same
quadrature points, summed in another order).  A wavenumber whose phases lie beyond the range of the
two-part reduction takes the library's sine and cosine: phases of size t carry an error of t 2^-52 per
term, and the terms of a block with phases that vary by millions cancel to a small part of their
magnitudes (1/n^2 of n^4 independent phases, n 6 to 8), for which the bound allows a factor of 1000.
"""
import numpy as np
import pytest

import bembel_amd as B
import oracle_lib as O

pytestmark = pytest.mark.gpu
ELLIPSOID = (1.0, 0.7, 0.5)


def _compare(M, P, kappa, pairs, tol):
    op = B.LaplaceSingleLayerOperator() if kappa is None else B.HelmholtzSingleLayerOperator()
    kind, k = (O.LAPLACE, 0j) if kappa is None else (O.HELMHOLTZ, complex(kappa))
    op.set_wavenumber(k)
    ps = B.AnsatzSpace(B.Geometry(scale=ELLIPSOID), M, P, op)
    os_ = O.Space(O.Geometry(scale=ELLIPSOID), M, P)
    got = ps.pair_blocks(op, pairs)
    seen = set()
    for b, (i, j) in zip(got, pairs):
        want = os_.pair_block(kind, int(i), int(j), kappa=k)
        info, _ = os_.pair_info(int(i), int(j))
        seen.add((info[0], info[3]))
        e = np.linalg.norm(b - want) / np.linalg.norm(want)
        assert e <= tol, (M, P, kappa, i, j, info, e)
    return seen


@pytest.mark.parametrize("P", [1, 2])
@pytest.mark.parametrize("kappa", [None, 3 - 0.2j])
def test_gpu_rules_every_pair_of_a_coarse_mesh(gpu, P, kappa):
    pairs = [(i, j) for i in range(24) for j in range(24)]
    assert {0, 2, 3, 4} <= {c for c, _ in _compare(1, P, kappa, pairs, 1e-12)}


@pytest.mark.parametrize("M", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("P,kappa", [(1, None), (2, None), (1, 2.0), (2, 2.0)])
def test_gpu_rules_degrees(gpu, M, P, kappa):
    n = 6 * 4 ** M
    ps = B.AnsatzSpace(B.Geometry(scale=ELLIPSOID), M, P)
    vert = ps.elements()["vert"]
    rng = np.random.default_rng(M)
    pairs = []
    for e in rng.choice(n, 2, replace=False):
        touch = [f for f in range(n) if np.isin(vert[f], vert[e]).any()]
        pairs += [(e, f) for f in touch] + [(e, f) for f in rng.choice(n, 3)]
    _compare(M, P, kappa, pairs, 1e-12)


def test_gpu_rules_large_phases(gpu):
    kappa = 4.0e6  # phases up to 8e6 on this body, beyond 2^20
    pairs = [(0, 0), (0, 1), (0, 2), (0, 20), (3, 17)]
    _compare(1, 1, kappa, pairs, 8e6 * 2.0 ** -52 * 1e3)
