"""Workgroups of a lone scene's solve, from the units of the last step (no GPU)."""
import os

import pytest

from rainbow_amd import native

pytestmark = pytest.mark.skipif(not os.path.exists(native.LIB_PATH), reason="librbh.so not built")


@pytest.mark.parametrize("units,grid", [(0, 64), (1, 1), (2, 1), (4, 1), (5, 5), (64, 64), (255, 255), (256, 256),
                                        (5000, 256)])
def test_one_lane_a_group_from_five_on(units, grid):
    """As many lanes as a workgroup has wavefronts share one; a scene of one unit is not one never seen."""
    assert native.load().rbh_coop_grid(units, 0, 256) == grid


@pytest.mark.parametrize("units,per,grid", [(0, 4, 16), (1, 4, 1), (5, 4, 2), (8, 1, 8), (2000, 4, 256)])
def test_lanes_per_group_as_set(units, per, grid):
    assert native.load().rbh_coop_grid(units, per, 256) == grid
