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
import extended_lib as X
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


def test_gpu_rules_round_points_once(gpu):
    # Regular pairs of near elements against extended precision.  A block's rounding averages out over its points
    # but for what all points of an element share, the coefficients of its polynomials: rounded once these leave
    # 1.0e-16 of the measure of either element (root mean square, computed on the sphere's elements), 1.5e-16 of
    # a block; the nodes and weights as doubles and the sums leave another 2.5e-16 (2.76e-16 with points in
    # Bernstein form, which share nothing): 2.9e-16.  Coefficients summed in doubles were at 3.2e-16.
    if not X.HAS_EXTENDED:
        pytest.skip("no extended precision on this host")
    M = 3
    op = B.LaplaceSingleLayerOperator()
    ps = B.AnsatzSpace(B.Geometry(), M, 1, op)
    os_ = O.Space(O.Geometry(), M, 1)
    el = ps.elements()
    rng = np.random.default_rng(4)
    pairs, degree = [], []
    for e in rng.permutation(ps.number_of_elements):
        near = [f for f in np.argsort(np.linalg.norm(el["mid"] - el["mid"][e], axis=1))[9:30]
                if os_.pair_info(int(e), int(f))[0][0] == 0]
        f = int(rng.choice(near))
        info, _ = os_.pair_info(int(e), f)
        if info[3] > 2:  # beyond the far-field rule, whose points come from a table
            pairs.append((int(e), f))
            degree.append(info[3])
        if len(pairs) == 60:
            break
    assert len(pairs) == 60
    got = ps.pair_blocks(op, pairs)
    errors = []
    T = np.longdouble
    for b, (e, f), deg in zip(got, pairs, degree):
        x, w = X.gauss(deg + 1, T)
        Y, area = X.sphere_points(T, {k: el[k][[e, f]] for k in ("llc", "patch")}, M, x)
        q = area * w[:, None] * w[None, :]
        basis = np.einsum("ux,vy->uvyx", X.linear(x), X.linear(x)).reshape(len(x) ** 2, 4)
        r = np.sqrt(((Y[0].reshape(-1, 1, 3) - Y[1].reshape(1, -1, 3)) ** 2).sum(-1))
        K = q[0].reshape(-1, 1) * q[1].reshape(1, -1) / r / (16 * np.arctan(T(1)))
        want = np.einsum("pi,pq,qj->ij", basis, K, basis)
        errors.append(float(min(np.linalg.norm(b - want), np.linalg.norm(b.T - want)) / np.linalg.norm(want)))
    rms = np.sqrt(np.mean(np.square(errors)))
    print("root mean square error", rms)
    assert rms <= 3.0e-16


@pytest.mark.parametrize("kappa", [None, 3.0])
def test_gpu_rules_round_touching_pairs(gpu, tmp_path, kappa):
    # A body whose control points have 21 bits, in its own unit and in a third of it: every length is exactly three
    # times the other, and what a block differs by from 27 times the other's is its rounding (either's, so by the
    # root of two).  Each of the 11^4 points of a rule is within a few ulps (2^-53) of its element's size, and their
    # errors average out: what is left is of the order of one ulp, 1.1e-16 to 3e-16 a block.  Coefficients rounded
    # against the body and sums of thousands of terms were at 2e-15.
    with open(B.SPHERE_DAT) as f:
        lines = f.read().splitlines()
    for p in range(6):
        for m in range(4):
            k = 5 + 9 * p + 5 + m
            lines[k] = " ".join("%.25g" % (round(float(v) * 2 ** 20) / 2 ** 20) for v in lines[k].split())
    path = tmp_path / "coarse.dat"
    path.write_text("\n".join(lines) + "\n")
    M = 5
    op = [B.LaplaceSingleLayerOperator() if kappa is None else B.HelmholtzSingleLayerOperator() for _ in range(2)]
    spaces = []
    for o, unit in zip(op, (1.0, 3.0)):
        o.set_wavenumber(0j if kappa is None else complex(3 * kappa / unit))
        spaces.append(B.AnsatzSpace(B.Geometry(str(path), scale=[unit * a for a in (1.0, 0.75, 0.5)]), M, 2, o))
    vert = spaces[0].elements()["vert"]
    rng = np.random.default_rng(2)
    pairs = {2: [], 3: [], 4: []}  # identical, edge, vertex: 1 per element, common vertices 4, 2, 1
    for e in rng.choice(len(vert), 12, replace=False):
        for f in np.nonzero(np.isin(vert, vert[e]).any(1))[0]:
            pairs[{4: 2, 2: 3, 1: 4}[int(np.isin(vert[f], vert[e]).sum())]].append((int(e), int(f)))
    for rule, todo in pairs.items():
        one, three = (s.pair_blocks(o, todo) for s, o in zip(spaces, op))
        norm = np.linalg.norm(one, axis=(1, 2))
        rms = np.sqrt(np.mean((np.linalg.norm(three / 27 - one, axis=(1, 2)) / norm) ** 2) / 2)
        print("rule", rule, len(todo), "root mean square error", rms)
        assert rms <= 4e-16, rule
