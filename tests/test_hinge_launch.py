"""How a batch's hinge solve is launched: rows staged in LDS or read from memory, and where they lie (no GPU)."""
import os

import pytest

from rainbow_amd import native

pytestmark = pytest.mark.skipif(not os.path.exists(native.LIB_PATH), reason="librbh.so not built")


def chains(precision, *counts):
    """(staged, bytes, row offsets) of a batch of chains on 256 compute units; counts: (scenes, links) pairs."""
    links = [n for scenes, n in counts for _ in range(scenes)]
    return native.hinge_launch(precision, 256, [n + 1 for n in links], links)


@pytest.mark.parametrize("scenes,links,staged", [(1, 83, True), (1, 84, False), (512, 80, True), (1024, 80, True),
                                                 (1280, 80, False), (2048, 80, False), (4096, 80, False),
                                                 (2048, 60, False), (2048, 40, True), (4096, 40, True), (4096, 5, True)])
def test_staged_while_it_is_faster_fp32(scenes, links, staged):
    """A staged chain of 80 links keeps 62 KB of LDS: with two to a CU, eight scenes a CU are faster from memory."""
    got, lds, _ = chains("fp32", (scenes, links))
    assert got == staged
    assert lds <= 65536 and (lds > 600 * links) == staged


@pytest.mark.parametrize("mix,staged", [(((1024, 5), (1, 80)), True), (((2048, 40), (1, 80)), False),
                                        (((1, 5), (1, 200)), False)])
def test_the_batch_pays_for_its_longest_chain(mix, staged):
    assert chains("fp32", *mix)[0] == staged


@pytest.mark.parametrize("precision,size", [("fp32", 16), ("fp64", 32)])
def test_rows_start_at_whole_vectors(precision, size):
    _, lds, rows = chains(precision, *((1, n) for n in range(1, 41)))
    assert all(int(r) % size == 0 for r in rows)
    # w of two vec4s a body and two iterates of five values a hinge lie below them
    assert all(int(r) >= 2 * size * (n + 1) + 10 * size // 4 * n for n, r in zip(range(1, 41), rows))
