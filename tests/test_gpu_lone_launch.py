"""GPU: a lone scene solved by one workgroup (an ordinary launch) and by several (a cooperative one)."""
import numpy as np
import pytest

from rainbow_amd import native, scenes
from test_gpu_solve import row_of_boxes, step_with

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 17])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("post", [False, True])
def test_one_workgroup_bitwise(n, precision, post):
    """lanes_per_group 64 puts every lane in one workgroup, 1 puts each in its own: the same bits, three steps on."""
    eng = row_of_boxes(scenes.ShapeBank(resolution=32), n,
                       dict(precision=precision, max_iterations=12, use_post_stabilization=post))
    ref = None
    for per in (64, 1):
        for steps in (1, 3):
            c, state, lg = step_with(eng, dict(lanes_per_group=per, unit_size=32), native.STEP_FORCE_MULTI, precision, steps)
            got = [c["impulse"], lg["residuals"], np.float64(lg["natural_residual"])] + list(state)
            if per == 64:
                ref = (ref or {}) | {steps: got}
            assert len(c["ia"]) >= n
            for a, b in zip(got, ref[steps]):
                assert np.array_equal(a, b), (per, steps)
