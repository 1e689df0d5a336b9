"""GPU: the ellipsoid projection's shortcuts against the plain bisection, bit for bit.

The reference bisects g(t) (proximal_operators.py:42-139) with three divisions a
level.  The kernel answers most levels without evaluating g; the answers are the
same, so the results are the same 64 bits.  Axes thin in one direction, points
beside the surface and tight tolerances are where a level's answer is closest.
"""
import numpy as np
import pytest

from rainbow_amd import native

pytestmark = pytest.mark.gpu


def bisection(z, mu, xn, tol, expansion, max_it):
    """proximal_operators.py:42-139 over arrays; axes of different lengths."""
    ax = mu * xn[:, None]
    scale = 1.0 / np.maximum(1.0, np.maximum(ax.max(1), np.abs(z).max(1)))[:, None]
    sa, sz = scale * ax, scale * z
    aa, zz = sa * sa, sz * sz

    def g(t):
        q = (aa * zz) / ((aa + t[:, None]) * (aa + t[:, None]))
        return q[:, 0] + q[:, 1] + q[:, 2] - 1.0

    f = zz / aa
    inside = f[:, 0] + f[:, 1] + f[:, 2] - 1.0 < tol
    t0 = np.zeros(len(xn))
    t1 = sa.max(1) * np.sqrt(zz[:, 0] + zz[:, 1] + zz[:, 2])
    while (g(t1) > 0.0).any():
        t1 = np.where(g(t1) > 0.0, t1 * expansion, t1)
    tk, going = (t0 + t1) * 0.5, np.ones(len(xn), bool)
    for _ in range(max_it):
        gk = g(tk)
        going &= ~(np.abs(t1 - t0) < tol) & ~(np.abs(gk) < tol)
        t0, t1 = np.where(going & (gk > 0.0), tk, t0), np.where(going & ~(gk > 0.0), tk, t1)
        tk = np.where(going, (t0 + t1) * 0.5, tk)
    t = (tk / (scale[:, 0] * scale[:, 0]))[:, None]
    return np.where(inside[:, None], z, (ax * ax * z) / (ax * ax + t))


def inputs(seed, n):
    """Axes of 0.1 to 1 and a thin one of 1e-3 to 1e-7; points 1e-10 to 0.1 outside the surface, or well outside."""
    rng = np.random.default_rng(seed)
    thin, out, far = 10.0 ** rng.uniform(-7, -3, n), 1.0 + 10.0 ** rng.uniform(-10, -1, n), rng.uniform(size=n) < 0.1
    out[far] = rng.uniform(1.0, 3.0, far.sum())
    xn, phi = np.exp(rng.normal(0.0, 3.0, n)), rng.uniform(0.0, 2.0 * np.pi, n)
    mu = rng.uniform(0.1, 1.0, (n, 3))
    z = np.stack([np.cos(phi) * out, np.sin(phi) * out, 10.0 ** rng.uniform(-6, 0, n) * rng.choice([-1.0, 1.0], n)], 1)
    mu[:, 2] = thin
    z = z * mu * xn[:, None]
    turn = rng.integers(3, size=n)[:, None]                  # the thin axis in each place
    at = (np.arange(3)[None] + turn) % 3
    return np.take_along_axis(z, at, 1), np.take_along_axis(mu, at, 1), xn


@pytest.mark.parametrize("tol", [0.0, 1e-14, 1e-12, 1e-11, 1e-10, 2e-10, 1e-9, 1e-6])
def test_thin_axes_bitwise(tol):
    z, mu, xn = inputs(11, 60000)
    ctx = native.Context(0, "fp64")
    try:
        got = ctx.prox_ellipsoid(z, mu, xn, tol, 1.5, 100)
    finally:
        ctx.close()
    ref = bisection(z, mu, xn, tol, 1.5, 100)
    bad = (got.view(np.uint64) != ref.view(np.uint64)).any(1)
    assert not bad.any(), "%d of %d differ, by up to %g of xn" % (
        bad.sum(), len(xn), (np.abs(got - ref).max(1) / xn).max())
    assert (got != z).any()
