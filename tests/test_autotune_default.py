"""The autotuner's baseline is the shape a scene has without it."""
import pytest

from rainbow_amd import autotune

# rbh_tuning's defaults of the fields the candidates set (include/rbh.h)
VALUES = dict(unit_size=64, lanes_per_scene=0, lanes_per_group=0, waves_per_group=4, solve_groups_per_cu=0)


@pytest.mark.parametrize("candidates", [autotune.single_candidates, autotune.batch_candidates])
def test_first_candidate_is_the_default(candidates):
    first = candidates()[0]
    assert {k: v or VALUES[k] for k, v in first.items()} == {k: VALUES[k] for k in first}


def test_a_lone_scene_can_keep_its_rule():
    """lanes_per_group = 0, the rule by the unit count, is among what a lone scene is tuned over."""
    assert any(c["lanes_per_group"] == 0 for c in autotune.single_candidates())
