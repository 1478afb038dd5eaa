"""The order in which prompt kernels take the sequences of a batch (``sequence_turns.h``, compiled with g++): in every turn each
sequence once, and over the turns no place - of eight dies, by a workgroup's id, and four groups of compute units inside each, in
turn - gets more than twice its share of a sequence's workgroups, whatever the number of sequences and of heads side by side."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    at = tmp_path_factory.mktemp("turns")
    (at / "t.cpp").write_text('#include "sequence_turns.h"\nextern "C" int order(int x, int turn, int batch, int side) { return sequence_in_turn(x, turn, batch, turns_miss_groups(side, batch)); }\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "t.so"),
                    str(at / "t.cpp")], check=True)
    return ctypes.CDLL(str(at / "t.so")).order


@pytest.mark.parametrize("batch", [2, 4, 6, 8, 12, 16, 24, 32])
@pytest.mark.parametrize("side", [1, 2, 3, 4, 6, 8, 16])  # workgroups of a turn and sequence, side by side
def test_no_place_gets_most_of_a_sequence(order, batch, side):
    turns = 256
    seen = np.zeros((batch, 8, 4), dtype=np.int64)
    for turn in range(turns):
        took = [order(x, turn, batch, side) for x in range(batch)]
        assert sorted(took) == list(range(batch))
        for x, b in enumerate(took):
            for s in range(side):
                place = side * (batch * turn + x) + s
                seen[b, place % 8, place // 8 % 4] += 1
    assert seen.max() <= 2 * turns * side / 32, seen.max()
