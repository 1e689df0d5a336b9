"""GPU: transfers larger than the pinned memory a context keeps."""
import ctypes as C

import numpy as np
import pytest

from rainbow_amd import native

pytestmark = pytest.mark.gpu

KEEP = 64 << 20       # most pinned memory of a context (include/rbh.h)


def pinned(ctx):
    b = C.c_ulonglong()
    assert ctx.lib.rbh_transfer_buffer(ctx.h, C.byref(b)) == 0
    return b.value


# a state is four vec4s a body, 128 bytes in FP64: 64 MiB are 524,288 bodies
@pytest.mark.parametrize("bodies", [1, 524288, 524289, 560000])
def test_pinned_memory_is_bounded(bodies):
    ctx = native.Context(0, "fp64")
    try:
        V = np.array([(0.0, 0.0, 0.0), (1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (0.0, 0.0, 1.0)])
        T = np.array([(0, 1, 2), (0, 2, 3)], dtype=np.int32)
        shape = ctx.shape_upload(V, T, np.ones(8), 2, 2, 2, (-1.0, -1.0, -1.0), (2.0, 2.0, 2.0))
        params = native.Params()
        params.max_iterations = 1
        params.time_step = 0.01
        zero = np.zeros(bodies, np.int32)
        desc, keep = native.Context.make_desc(zero + shape, zero, zero, np.ones(bodies), np.ones((bodies, 3)),
                                              np.zeros((bodies, 3)), np.zeros((bodies, 2)), np.zeros((1, 4)), params)
        sid = ctx.scene_create(desc)
        rng = np.random.default_rng(bodies)
        want = [rng.normal(size=(bodies, d)) for d in (3, 4, 3, 3)]
        ctx.set_state(sid, *want)
        want[2] += 1.0
        ctx.set_state(sid, v=want[2])
        for a, b in zip(ctx.get_state(sid, bodies), want):
            assert np.array_equal(a, b)
        assert 0 < pinned(ctx) <= KEEP
    finally:
        ctx.close()
