"""GPU: hinge rows staged in LDS against rows read from memory.

A chain of 42 hinges is the longest that is staged in FP64 (64 KB), 83 in FP32.
The FP64 build must match the oracle on both sides of that line, and an FP32
scene must step the same alone as in a batch with a chain too long for it.
"""
import numpy as np
import pytest

import oracle.scene as OS
from rainbow_amd import native, scenes
from rainbow_amd.stepper import engine_desc, gather_state, upload_hinges
from test_gpu_hinges import check_step

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bank():
    return scenes.ShapeBank(resolution=16)


def chain(bank, n, precision):
    eng = scenes.cube_hinge_chain(bank, n=n, params=dict(precision=precision, max_iterations=12, absolute_tolerance=0.0,
                                                         relative_tolerance=0.0))
    rng = np.random.default_rng(n)
    for b in eng.bodies.values():
        if not b.is_fixed:
            b.v, b.w = rng.normal(0.0, 0.3, 3), rng.normal(0.0, 0.1, 3)
    return eng


@pytest.mark.parametrize("n", [2, 3, 42, 43, 44])
def test_chain_lengths_fp64(bank, n):
    eng = chain(bank, n, "fp64")
    sc = OS.from_engine(eng)
    for _ in range(2):
        check_step(eng, sc, 0.01)


@pytest.mark.parametrize("lengths", [(2, 5, 83, 84, 85, 130)])
def test_mixed_batch_bitwise_fp32(bank, lengths):
    engines = [chain(bank, n, "fp32") for n in lengths]
    ctx = native.Context(0, "fp32")
    try:
        def fresh(eng):
            desc, keep = engine_desc(eng, ctx)
            sid = ctx.scene_create(desc)
            upload_hinges(ctx, sid, eng)
            ctx.set_state(sid, *gather_state(list(eng.bodies.values())))
            return sid
        alone = []
        for eng in engines:
            sid = fresh(eng)
            ctx.step([sid], 3)
            alone.append(ctx.get_state(sid, len(eng.bodies)))
            ctx.scene_destroy(sid)
        ids = [fresh(eng) for eng in engines]
        ctx.step(ids, 3)
        for sid, eng, ref in zip(ids, engines, alone):
            for a, b in zip(ctx.get_state(sid, len(eng.bodies)), ref):
                assert np.array_equal(a, b)
    finally:
        ctx.close()
