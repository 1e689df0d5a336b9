"""GPU: the pruned signed-distance build against the FP64 oracle (brute force).

Meshes beyond the plain build's sizes: closed ones, one with unwelded vertices
(every triangle its own), an open one and one with a doubled triangle (their
winding numbers are not constant off the surface), two nested closed surfaces,
grids whose nodes lie on the surface, and node counts off the 4 x 4 x 4 blocks.
The bound is the one of test_gpu_parity's plain build: both take the same
closest-point expressions in 64 bits.  Where a node lies on the surface only the
magnitude is compared (the sign there is rounding's).
"""
import numpy as np
import pytest

from oracle.grid import Grid, nodes_array
from oracle.sdf import signed_distance
from rainbow_amd import mesh as MESH
from rainbow_amd import native

pytestmark = pytest.mark.gpu


def meshes():
    V, T = MESH.create_sphere(0.5, 16, 16)
    T = np.asarray(T)
    yield "sphere", V, T, (0.2, 0.2, 0.2), (17, 13, 10)
    yield "unwelded", V[T].reshape(-1, 3), np.arange(3 * len(T)).reshape(-1, 3), (0.2, 0.2, 0.2), (9, 12, 11)
    yield "open", V, T[40:], (0.2, 0.2, 0.2), (12, 8, 9)
    yield "doubled", V, np.concatenate([T, T[:1]]), (0.3, 0.1, 0.2), (8, 8, 8)
    V2, T2 = MESH.create_sphere(0.25, 12, 12)
    yield "nested", np.concatenate([V, V2]), np.concatenate([T, np.asarray(T2) + len(V)]), (0.1, 0.1, 0.1), (16, 16, 16)
    B, F = MESH.create_box(1.0, 1.0, 1.0)
    for _ in range(3):   # faces quartered three times: 768 triangles, nodes of the grid on them
        n, tri = len(B), []
        mids = {}
        B = list(map(tuple, B))
        for a, b, c in np.asarray(F).tolist():
            m = []
            for e in ((a, b), (b, c), (c, a)):
                key = tuple(sorted(e))
                if key not in mids:
                    mids[key] = len(B)
                    B.append(tuple((np.array(B[e[0]]) + np.array(B[e[1]])) / 2.0))
                m.append(mids[key])
            tri += [(a, m[0], m[2]), (m[0], b, m[1]), (m[2], m[1], c), (m[0], m[1], m[2])]
        B, F = np.array(B), np.array(tri)
    yield "box", B, F, (0.25, 0.25, 0.25), (13, 13, 13)
    K, S = MESH.create_torus_knot(segments=40, sides=6)
    yield "knot", K, S, (0.2, 0.2, 0.2), (15, 14, 18)


@pytest.mark.parametrize("name,V,T,pad,res", list(meshes()), ids=lambda a: a if isinstance(a, str) else "")
def test_pruned_sdf_matches_oracle(name, V, T, pad, res):
    V = np.ascontiguousarray(V, dtype=np.float64)
    T = np.ascontiguousarray(T, dtype=np.int32)
    assert len(T) * 55000 > 1.1e7     # (below that the plain build runs)
    lo, hi = V.min(0) - pad, V.max(0) + pad
    ctx = native.Context(0, "fp32")
    try:
        got = ctx.sdf_build(V, T, lo, hi, *res)
        again = ctx.sdf_build(V, T, lo, hi, *res)
        small = ctx.sdf_build_noalloc(V, T, lo, hi, *res)
    finally:
        ctx.close()
    assert np.array_equal(got.view(np.uint64), again.view(np.uint64))
    assert np.array_equal(got.view(np.uint64), small.view(np.uint64))
    ref = signed_distance(nodes_array(Grid(lo, hi, *res)), V, T)
    assert np.abs(np.abs(got) - np.abs(ref)).max() < 1e-12
    off = np.abs(ref) > 1e-9
    assert np.array_equal(np.signbit(got[off]), np.signbit(ref[off]))
    assert (ref < 0).any() and (ref > 0).any()
