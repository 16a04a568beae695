"""Gauss points and the sphere's surface in a numpy type of choice: with np.longdouble the extended-precision
side of the rounding tests, with np.float64 a plain double evaluation, every operation rounded once."""
import numpy as np

import bembel_amd as B

HAS_EXTENDED = np.finfo(np.longdouble).eps < 2e-19


def gauss(n, T):
    """Nodes and weights of the n-point rule on [0, 1]."""
    x = np.polynomial.legendre.leggauss(n)[0].astype(np.longdouble)
    for _ in range(3):  # Newton's iteration on the Legendre polynomial
        p0, p1 = np.ones_like(x), x.copy()
        for k in range(2, n + 1):
            p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
        dp = n * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / dp
    return ((1 + x) / 2).astype(T), (1 / ((1 - x * x) * dp * dp)).astype(T)


def sphere_points(T, elements, M, x):
    """Points and h |d_s X x d_t X| at the local grid x (x) x of every element: (element, s, t[, 3])."""
    with open(B.SPHERE_DAT) as f:
        lines = f.read().splitlines()[5:]
    cp = np.array([[np.array(lines[9 * p + 5 + m].split(), dtype=float).reshape(5, 5).T for m in range(4)]
                   for p in range(6)]).transpose(0, 2, 3, 1).astype(T)  # (patch, s, t, xyzw)
    h = T(1) / 2 ** M
    binom = {3: (1, 3, 3, 1), 4: (1, 4, 6, 4, 1)}

    def bern(p, t):
        return np.stack([binom[p][k] * t ** k * (1 - t) ** (p - k) for k in range(p + 1)], -1)

    def der(t):
        b = bern(3, t)
        z = np.zeros_like(b[..., :1])
        return 4 * (np.concatenate([z, b], -1) - np.concatenate([b, z], -1))

    s, t = (elements["llc"].astype(T)[:, None, None, k] + h * (x[:, None] if k == 0 else x[None, :]) for k in (0, 1))
    s, t = np.broadcast_arrays(s, t)
    c = cp[elements["patch"]][:, None, None]

    def form(a, b):
        return ((a[..., :, None, None] * c).sum(-3) * b[..., :, None]).sum(-2)

    v, vs, vt = form(bern(4, s), bern(4, t)), form(der(s), bern(4, t)), form(bern(4, s), der(t))
    X = v[..., :3] / v[..., 3:]
    ds, dt = ((d[..., :3] - X * d[..., 3:]) / v[..., 3:] for d in (vs, vt))
    return X, h * np.sqrt((np.cross(ds, dt) ** 2).sum(-1))


def linear(x):
    """The two functions of degree 1."""
    return np.stack([1 - x, x], -1)
