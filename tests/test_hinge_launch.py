"""How a batch's hinge solve is launched: rows staged in LDS or read from memory, and where they lie (no GPU)."""
import os

import pytest

from rainbow_amd import native

pytestmark = pytest.mark.skipif(not os.path.exists(native.LIB_PATH), reason="librbh.so not built")


def chains(precision, *counts):
    """(staged, bytes, row offsets) of a batch of chains on 256 compute units; counts: (scenes, links) pairs."""
    links = [n for scenes, n in counts for _ in range(scenes)]
    return native.hinge_launch(precision, 256, [n + 1 for n in links], links)


@pytest.mark.parametrize("precision,size", [("fp32", 16), ("fp64", 32)])
def test_rows_start_at_whole_vectors(precision, size):
    _, lds, rows = chains(precision, *((1, n) for n in range(1, 41)))
    assert all(int(r) % size == 0 for r in rows)
    # w of two vec4s a body and two iterates of five values a hinge lie below them
    assert all(int(r) >= 2 * size * (n + 1) + 10 * size // 4 * n for n, r in zip(range(1, 41), rows))
