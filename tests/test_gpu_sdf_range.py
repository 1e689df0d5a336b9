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


def winding(P, V, T):
    """Sum of the solid angles over 4 pi, in the kernels' expressions (signed zeros too)."""
    with np.errstate(all="ignore"):
        a, b, c = (V[T[:, k]][None] - P[:, None] for k in range(3))
        (ax, ay, az), (bx, by, bz), (cx, cy, cz) = (np.moveaxis(x, 2, 0) for x in (a, b, c))
        la, lb, lc = (np.sqrt((x * x).sum(-1)) for x in (a, b, c))
        det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx)
        den = la * lb * lc + (a * b).sum(-1) * lc + (b * c).sum(-1) * la + (c * a).sum(-1) * lb
    return 2.0 * np.arctan2(det, den).sum(1) / (4.0 * np.pi)


def quartered_box(times):
    """A unit box, its faces quartered `times` times."""
    V, T = MESH.create_box(1.0, 1.0, 1.0)
    V, T = [tuple(v) for v in V], np.asarray(T).tolist()
    for _ in range(times):
        index, out = {v: i for i, v in enumerate(V)}, []

        def middle(i, j):
            v = tuple((np.array(V[i]) + np.array(V[j])) / 2.0)
            if v not in index:
                index[v] = len(V)
                V.append(v)
            return index[v]

        for a, b, c in T:
            m = middle(a, b), middle(b, c), middle(c, a)
            out += [(a, m[0], m[2]), (m[0], b, m[1]), (m[2], m[1], c), m]
        T = out
    return np.array(V), np.array(T, dtype=np.int32)


@pytest.mark.parametrize("seed", range(2))
@pytest.mark.parametrize("inwards", [False, True])
@pytest.mark.parametrize("times,n", [(2, 41), (3, 21)])      # 3 and 12 triangles a lane; a spacing of 1/32 and 1/16
def test_sign_on_the_surface(ctx, seed, inwards, times, n):
    """Nodes on a box's faces have a winding number of 0, 1/2 or 1, as the signed zeros of their triangles fall; away
    from 1/2 the sign must be the one of the sum of arctangents, whatever order the triangles come in."""
    V, T = quartered_box(times)
    T = T[np.random.default_rng(seed).permutation(len(T))]
    T = np.ascontiguousarray(T[:, ::-1] if inwards else T)
    lo, hi = np.full(3, -0.625), np.full(3, 0.625)          # nodes at +-1/2
    got = ctx.sdf_build(V, T, lo, hi, n, n, n)
    x = lo[0] + (hi[0] - lo[0]) / (n - 1) * np.arange(n)
    k, j, i = np.meshgrid(x, x, x, indexing="ij")
    P = np.stack([i.ravel(), j.ravel(), k.ravel()], 1)
    on = np.abs(P).max(1) == 0.5
    assert (got[on] == 0.0).all()
    w = np.abs(winding(P[on], V, T))
    sure = np.abs(w - 0.5) > 1e-6
    assert sure.any()
    assert np.array_equal(np.signbit(got[on])[sure], (w > 0.5)[sure])


@pytest.mark.parametrize("offset,size", [(0.0, None), (0.0, 1e-8), (1e4, None), (1e4, 1e-8), (1e4, 1e-10)])
def test_pruned_against_plain_bitwise(ctx, offset, size):
    """The pruned build and the plain one, bit for bit: over the whole mesh and in boxes of `size` around points of its
    surface, where every distance is small.  (128^3 nodes: the plain build fits the no-allocation array, the pruned
    one's workspace does not, so sdf_build_noalloc is the plain build.)"""
    V, T = sphere()
    q, _ = np.linalg.qr(np.random.default_rng(3).normal(size=(3, 3)))
    V = np.ascontiguousarray(V @ q + offset)
    rng = np.random.default_rng(4)
    for k in range(1 if size is None else 4):
        if size is None:
            lo, hi = V.min(0) - 0.2, V.max(0) + 0.2
        else:   # around a vertex, an edge and the inside of a triangle
            w = np.array([(1.0, 0.0, 0.0), (0.5, 0.5, 0.0), (0.2, 0.3, 0.5), (0.3, 0.7, 0.0)][k])
            c = w @ V[T[rng.integers(len(T))]]
            lo, hi = c - size, c + size * rng.uniform(0.5, 1.5, 3)
        pruned, plain = ctx.sdf_build(V, T, lo, hi, 128, 128, 128), ctx.sdf_build_noalloc(V, T, lo, hi, 128, 128, 128)
        bad = bits(pruned) != bits(plain)
        assert not bad.any(), "%d differ, by up to %g" % (bad.sum(), np.abs(pruned - plain).max())


def closest_sq(p, a, b, c):
    """Squared distance of p to a triangle, region after region (Ericson, "Real-Time Collision Detection" 5.1.5)."""
    ab, ac, ap, bp, cp = b - a, c - a, p - a, p - b, p - c
    d1, d2, d3, d4, d5, d6 = ab @ ap, ac @ ap, ab @ bp, ac @ bp, ab @ cp, ac @ cp
    if d1 <= 0.0 and d2 <= 0.0:
        return ap @ ap
    if d3 >= 0.0 and d4 <= d3:
        return bp @ bp
    vc, vb, va = d1 * d4 - d3 * d2, d5 * d2 - d1 * d6, d3 * d6 - d5 * d4
    if vc <= 0.0 and d1 >= 0.0 and d3 <= 0.0:
        q = a + d1 / (d1 - d3) * ab
    elif d6 >= 0.0 and d5 <= d6:
        return cp @ cp
    elif vb <= 0.0 and d2 >= 0.0 and d6 <= 0.0:
        q = a + d2 / (d2 - d6) * ac
    elif va <= 0.0 and d4 - d3 >= 0.0 and d5 - d6 >= 0.0:
        q = b + (d4 - d3) / ((d4 - d3) + (d5 - d6)) * (c - b)
    else:
        den = 1.0 / (va + vb + vc)
        q = a + ab * (vb * den) + ac * (vc * den)
    return (p - q) @ (p - q)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1.5e308])
@pytest.mark.parametrize("corner", [0, 1, 2])
def test_corner_out_of_range(ctx, value, corner):
    """A triangle with a corner at infinity has a distance where another corner is the closest point."""
    V = np.array([(0.1, 0.2, 0.0), (0.9, 0.1, 0.2), (0.3, 0.8, 0.1)])
    T = np.array([(0, 1, 2)], dtype=np.int32)
    V[corner, 0] = value
    lo, hi = (-1.0, -1.0, -1.0), (2.0, 2.0, 2.0)
    n = 6
    got = np.abs(ctx.sdf_build(V, T, lo, hi, n, n, n))
    assert np.array_equal(bits(got), bits(np.abs(ctx.sdf_build_noalloc(V, T, lo, hi, n, n, n))))
    x = lo[0] + (hi[0] - lo[0]) / (n - 1) * np.arange(n)
    with np.errstate(all="ignore"):
        ref = np.array([closest_sq(np.array((i, j, k)), *V) for k in x for j in x for i in x])
    known = ref < np.inf                          # (a NaN or an infinity leaves the minimum at infinity)
    assert np.abs(got[known] - np.sqrt(ref[known])).max(initial=0.0) < 1e-12
    assert (got[~known] == np.inf).all()


def test_plain_forms_bitwise(ctx):
    """Up to 65,536 nodes the plain build finds closest points by selects, above it by branches: the nodes that two
    grids on either side of the line share have the same bits."""
    V, T = quartered_box(1)
    q, _ = np.linalg.qr(np.random.default_rng(8).normal(size=(3, 3)))
    V = np.ascontiguousarray(V @ q)
    lo, h = np.full(3, -1.0), 1.0 / 32.0                     # exact spacing: shared nodes have the same coordinates
    out = [ctx.sdf_build(V, T, lo, lo + h * (np.array(n) - 1), *n).reshape(n[::-1]) for n in ((64, 32, 32), (66, 32, 32))]
    assert out[0].size == 65536
    assert np.array_equal(bits(out[0]), bits(np.ascontiguousarray(out[1][:, :, :64])))
    assert np.signbit(out[0]).any() and not np.signbit(out[0]).all()


@pytest.mark.parametrize("mesh", ["open511", "open512", "open513", "open719", "box"])   # (tiles of 256 triangles)
def test_many_roots_bitwise(ctx, mesh):
    """Open meshes, whose every node has its own winding number: from 163,840 nodes on a thread takes a node, below a
    wavefront does.  Two grids on either side of the line agree in the nodes they share, on the faces of a box (winding
    numbers near 1/2) too, and the larger one has the plain build's values."""
    if mesh == "box":
        V, T = quartered_box(3)
        T = T[1:]
    else:
        V, T = MESH.create_sphere(0.5, 20, 20)
        V, T = np.ascontiguousarray(V), np.ascontiguousarray(T, dtype=np.int32)
        T = T[-int(mesh[4:]):]
    lo, h = np.full(3, -0.625), 1.0 / 32.0                   # exact spacing: shared nodes have the same coordinates
    out = [ctx.sdf_build(V, T, lo, lo + h * (np.array(n) - 1), *n).reshape(n[::-1]) for n in ((63, 64, 40), (64, 64, 40))]
    assert out[1].size == 163840
    assert native.sdf_is_pruned(V, T, lo, lo + h * 62, 63, 64, 40)
    assert np.array_equal(bits(out[0]), bits(np.ascontiguousarray(out[1][:, :, :63])))
    hi = lo + h * 63
    many, plain = ctx.sdf_build(V, T, lo, hi, 128, 128, 128), ctx.sdf_build_noalloc(V, T, lo, hi, 128, 128, 128)
    assert np.array_equal(bits(many), bits(plain))
    assert np.signbit(plain).any()


def test_no_memory_for_the_grid():
    """A grid larger than the device (4,096^3 nodes, 550 GB) is refused as such, and the context goes on."""
    V, T = sphere()
    lo, hi = V.min(0) - 0.2, V.max(0) + 0.2
    ctx = native.Context(0, "fp64")
    try:
        before = ctx.sdf_build(V, T, lo, hi, 16, 16, 16)
        none = np.empty(1)                       # (nothing is written without a buffer on the device)
        rc = ctx.lib.rbh_sdf_build(ctx.h, native._ptr(V), len(V), native._ptr(T), len(T), native._ptr(lo), native._ptr(hi),
                                   4096, 4096, 4096, native._ptr(none))
        assert rc == -3 and ctx.lib.rbh_last_error(ctx.h) == b"SDF buffer"
        assert np.array_equal(bits(ctx.sdf_build(V, T, lo, hi, 16, 16, 16)), bits(before))
    finally:
        ctx.close()
