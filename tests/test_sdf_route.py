"""Which signed-distance builds are pruned (no GPU): where that is the faster form."""
import os

import numpy as np
import pytest

from rainbow_amd import mesh as MESH
from rainbow_amd import native

pytestmark = pytest.mark.skipif(not os.path.exists(native.LIB_PATH), reason="librbh.so not built")


def pruned(V, T, n):
    lo, hi = V.min(0) - 0.2, V.max(0) + 0.2
    return native.sdf_is_pruned(V, T, lo, hi, n, n, n)


def sphere(t):
    V, T = MESH.create_sphere(0.5, t, t)
    return np.asarray(V), np.asarray(T)


def test_few_triangles_are_plain_at_any_size():
    V, T = (np.asarray(a) for a in MESH.create_box(1.0, 0.5, 0.25))
    assert not pruned(V, T, 64) and not pruned(V, T, 128)
    assert not pruned(*sphere(6), 128)                          # 48 triangles
    assert pruned(*sphere(7), 64) and not pruned(*sphere(7), 54)   # 70


@pytest.mark.parametrize("t,n", [(9, 54), (12, 48), (14, 64), (15, 64)])   # 126, 240, 336 and 390 triangles
def test_open_meshes_of_up_to_384_triangles(t, n):
    """Closed by its vertices, or with vertices at one position as one (of either zero), or open."""
    V, T = sphere(t)
    few = len(T) <= 384
    assert pruned(V, T, n)
    apart = V[T].reshape(-1, 3)
    apart[::2] = np.where(apart[::2] == 0.0, -0.0, apart[::2])
    order = np.arange(len(apart)).reshape(-1, 3)
    assert pruned(apart, order, n)
    assert pruned(V, T[1:], n) != few
    assert pruned(apart, order[1:], n) != few
    turned = T.copy()
    turned[0] = turned[0, ::-1]
    assert pruned(V, turned, n) != few
    assert pruned(V, np.concatenate([T, T[:1, [0, 0, 1]]]), n)     # a triangle without area


def test_open_meshes_on_small_grids_are_pruned():
    V, T = sphere(12)
    assert pruned(V, T[1:], 36) and not pruned(V, T[1:], 37)


def test_line_by_pairs():
    V, T = sphere(16)                                           # 448 triangles
    assert pruned(V, T, 10)
    V, T = sphere(11)                                           # 198: 1.1e7 pairs above 38.2^3 nodes
    assert not pruned(V, T, 38) and pruned(V, T, 39)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e61, 1e308])
def test_unbounded_coordinates_are_plain(value):
    V, T = sphere(16)
    V = V.copy()
    V[3, 1] = value
    assert not native.sdf_is_pruned(V, T, (-1.0,) * 3, (1.0,) * 3, 32, 32, 32)
