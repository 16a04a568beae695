"""Near-field rules over the quadrature degrees and rotations they meet: the chunks of outer coordinates,
lanes per unit and odd inner ranges of the factorised rules change with the number of points per
direction, and every rotation of the edge rule has its own code.

Every pair of the 24-element ellipsoid (all rotations, also across patches), and sampled touching and
near pairs of finer meshes (6 to 13 points per direction) equal the oracle to 1e-12 (the same
quadrature points, summed in another order).  A wavenumber whose phases lie beyond the range of the
two-part reduction takes the library's sine and cosine: phases of size t carry an error of t 2^-52 per
term, and the terms of a block with phases that vary by millions cancel to a small part of their
magnitudes (1/n^2 of n^4 independent phases, n 6 to 8), for which the bound allows a factor of 1000.

Elements without area give zero, with themselves and with their neighbours, and the unit of length only
scales a block.
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


# a unit square, and a patch on the line of its edge x = 1 (distinct corners, no area)
FLAT = """# two bilinear patches
#
#
#
2 3 2 0 0
PATCH 0
1 1
2 2
0 0 1 1
0 0 1 1
0 1 0 1
0 0 1 1
0 0 0 0
1 1 1 1
PATCH 1
1 1
2 2
0 0 1 1
0 0 1 1
1 1 1 1
0 -1 1 2
0 0 0 0
1 1 1 1
"""


@pytest.mark.parametrize("P", [1, 2])
@pytest.mark.parametrize("kappa", [None, 2.0, 2 - 0.5j])
def test_gpu_rules_elements_without_area(gpu, tmp_path, P, kappa):
    path = tmp_path / "flat.dat"
    path.write_text(FLAT)
    op = B.LaplaceSingleLayerOperator() if kappa is None else B.HelmholtzSingleLayerOperator()
    op.set_wavenumber(0j if kappa is None else complex(kappa))
    ps = B.AnsatzSpace(B.Geometry(str(path)), 1, P, op)
    patch, vert = ps.elements()["patch"], ps.elements()["vert"]
    touch = [(i, j) for i in range(8) for j in range(8) if len(set(vert[i]) & set(vert[j])) >= 2]
    got = ps.pair_blocks(op, touch)
    kinds = set()
    for b, (i, j) in zip(got, touch):
        assert np.isfinite(b).all(), (i, j)
        kinds.add((i == j, patch[i], patch[j]))
        assert (b == 0).all() == bool(patch[i] or patch[j]), (i, j)
    assert {(True, 1, 1), (False, 1, 1), (False, 0, 1), (True, 0, 0)} <= kinds


@pytest.mark.parametrize("unit", [2.0 ** -25, 2.0 ** 110])
def test_gpu_rules_unit_of_length(gpu, unit):
    # lengths in another unit, a power of two: Laplace blocks scale by its third power exactly
    pairs = [(0, 0), (0, 1), (5, 5), (1, 0), (7, 6)]
    op = B.LaplaceSingleLayerOperator()
    one, other = (B.AnsatzSpace(B.Geometry(scale=[u * a for a in ELLIPSOID]), 1, 2, op).pair_blocks(op, pairs)
                  for u in (1.0, unit))
    assert np.array_equal(other / unit ** 3, one)
