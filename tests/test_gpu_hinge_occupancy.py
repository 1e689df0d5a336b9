"""GPU: hinged scenes that share a compute unit."""
import pytest

from rainbow_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,waves", [("fp32", 8), ("fp64", 4)])
def test_rows_from_memory_leave_room(precision, waves):
    """Rows read from memory are hidden by other scenes' wavefronts: two a SIMD in FP32, one in FP64."""
    ctx = native.Context(0, precision)
    try:
        assert ctx.hinge_occupancy(False, 4096) >= waves
        assert ctx.hinge_occupancy(True, 62 * 1024) == 2
        assert ctx.hinge_occupancy(True, 16 * 1024) >= waves
    finally:
        ctx.close()
