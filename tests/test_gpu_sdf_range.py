"""GPU: the signed-distance builds at the ends of what they accept."""
import numpy as np
import pytest

from rainbow_amd import mesh as MESH
from rainbow_amd import native

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = native.Context(0, "fp64")
    yield c
    c.close()


def sphere():
    V, T = MESH.create_sphere(0.5, 16, 16)
    return np.ascontiguousarray(V), np.ascontiguousarray(T, dtype=np.int32)


def bits(a):
    return a.view(np.uint64)


@pytest.mark.parametrize("exponent", [-300, -190, 190, 300])
def test_size_of_the_mesh(ctx, exponent):
    """A mesh scaled by a power of two has the signs of the mesh, and its scaled distances where no product of four
    lengths leaves the range of a double."""
    V, T = sphere()
    lo, hi = V.min(0) - 0.2, V.max(0) + 0.2
    s = 2.0 ** exponent
    base = ctx.sdf_build(V, T, lo, hi, 24, 24, 24)
    got = ctx.sdf_build(V * s, T, lo * s, hi * s, 24, 24, 24)
    assert np.array_equal(np.signbit(got), np.signbit(base))
    if abs(exponent) < 250:
        assert np.array_equal(bits(got), bits(base * s))
