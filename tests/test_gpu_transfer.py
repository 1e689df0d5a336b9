"""GPU: scene states through the pinned transfer buffer, at the sizes where it wraps and grows."""
import numpy as np
import pytest

from rainbow_amd import math3 as Q
from rainbow_amd import mesh as MESH
from rainbow_amd import native, scenes
from rainbow_amd.stepper import engine_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("count,n", [(1, 0), (1, 1), (400, 60), (2, 18000)])
def test_state_round_trip(precision, count, n):
    """States written one after another, more than the transfer buffer's first megabyte together (400 scenes) and
    alone (18,000 bodies), come back as they were, also after a partial write; a step index read back too."""
    bank = scenes.ShapeBank(resolution=16)
    eng = scenes.new_engine(bank, dict(precision=precision))
    box = bank.get("box_shape", lambda: MESH.create_box(1.0, 1.0, 1.0))
    scenes.add_ground(eng, bank)
    for i in range(n):
        scenes.add_body(eng, "b%d" % i, box, np.array([3.0 * i, 5.0, 0.0]), q=Q.identity())
    ctx = native.Context(0, precision)
    try:
        desc, keep = engine_desc(eng, ctx)
        ids = [ctx.scene_create(desc) for _ in range(count)]
        rng = np.random.default_rng(n)
        want = [[rng.normal(size=(n + 1, d)).astype(np.float32).astype(np.float64) for d in (3, 4, 3, 3)] for _ in ids]
        for i, (sid, st) in enumerate(zip(ids, want)):
            ctx.set_state(sid, *st)
            ctx.set_step_index(sid, 7 + i)
        for sid, st in zip(ids, want):
            st[2] = st[2] + 1.0
            st[2] = st[2].astype(np.float32).astype(np.float64)
            ctx.set_state(sid, v=st[2])
        for i, (sid, st) in enumerate(zip(ids, want)):
            for a, b in zip(ctx.get_state(sid, n + 1), st):
                assert np.array_equal(a, b)
            assert ctx.get_log(sid, 4)["step_index"] == 7 + i
    finally:
        ctx.close()


def test_scene_after_larger_sdf_build():
    """A signed-distance build whose buffer grows between two scenes of one context leaves the transfers alone."""
    bank = scenes.ShapeBank(resolution=16)
    eng = scenes.new_engine(bank, dict(precision="fp64"))
    scenes.add_ground(eng, bank)
    ctx = native.Context(0, "fp64")
    try:
        V, T = MESH.create_sphere(0.5, 16, 16)
        for resolution in (8, 24, 48):
            ctx.sdf_build(V, T, V.min(0) - 0.2, V.max(0) + 0.2, resolution, resolution, resolution)
            desc, keep = engine_desc(eng, ctx)
            sid = ctx.scene_create(desc)
            st = [np.full((1, d), float(resolution)) for d in (3, 4, 3, 3)]
            ctx.set_state(sid, *st)
            for a, b in zip(ctx.get_state(sid, 1), st):
                assert np.array_equal(a, b)
    finally:
        ctx.close()
