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


@pytest.mark.parametrize("units,bodies,per,grid", [
    (0, 2, 0, 1), (0, 64, 0, 1), (0, 65, 0, 64), (0, 64, 1, 64), (-1, 64, 0, 64), (5, 64, 0, 5), (4, 64, 0, 1),
    (300, 4096, 0, 256)])
def test_seen_without_contacts(units, bodies, per, grid):
    """A small scene known to have no contacts needs no cooperative launch; one never seen may have any number."""
    assert native.load().rbh_lone_grid(units, bodies, per, 256) == grid
