"""Attention with mixed heads (``talking_plan.h``, compiled with g++): the lines between the kernels of prompts, and the division by a block's size that
one of them makes by a product."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "talking_plan.h"
extern "C" int takes(int heads, int kv, int batch, int most, long long rows, long long room) {
    return talk_pipe_takes(heads, heads / kv, batch, most, rows, room, 256);
}
extern "C" int in_order(int heads, int batch, int most) { return talk_pipe_in_order(heads, batch, most, 256); }
extern "C" long long wrong(int block_size, const long long *keys, int n) {  // a key whose block is another one; -1: there is none
    const TalkDivision d = talk_division(block_size);
    for (int i = 0; i < n; ++i) {
        const uint32_t key = (uint32_t)keys[i], by = (uint32_t)((uint64_t)(2u * key) * d.mul >> 32) >> d.shift;
        if (d.shift < 0 || d.shift > 31 || by != key / (uint32_t)block_size) return keys[i];
    }
    return -1;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    at = tmp_path_factory.mktemp("talking")
    (at / "t.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "t.so"),
                    str(at / "t.cpp")], check=True)
    lib = ctypes.CDLL(str(at / "t.so"))
    lib.takes.argtypes = [ctypes.c_int] * 4 + [ctypes.c_longlong] * 2
    lib.wrong.argtypes, lib.wrong.restype = [ctypes.c_int, ctypes.c_void_p, ctypes.c_int], ctypes.c_longlong
    return lib


def test_division_at_the_edges_of_blocks(plan):
    rng = np.random.default_rng(0)
    top = (1 << 31) - 1
    for size in [*range(1, 600), *(int(2 ** x) + d for x in range(9, 31) for d in (-1, 0, 1)), 70001, top - 1, top]:
        last = top // size
        blocks = np.unique(np.concatenate([np.arange(0, min(last, 40) + 1), rng.integers(0, last + 1, 60), [last, max(last - 1, 0)]]).astype(np.int64))
        keys = np.concatenate([blocks * size - 1, blocks * size, blocks * size + size // 2, [top - 1, top]])
        keys = np.ascontiguousarray(keys[(keys >= 0) & (keys <= top)])
        assert plan.wrong(size, keys.ctypes.data, len(keys)) == -1, size


def test_lines_of_the_kernel_with_waves_of_two_kinds(plan):
    def takes(heads, kv, lens, behind=0, most=None):
        most = most or max(lens)
        return bool(plan.takes(heads, kv, len(lens), most, sum(lens), behind + most))

    assert takes(8, 2, [1]) and takes(4, 1, [17] * 600) and takes(8, 1, [5], 3)                  # up to 8 heads: always
    assert not any(takes(h, kv, [4000]) for h, kv in ((6, 2), (8, 8), (10, 1), (12, 2), (16, 8), (20, 4), (32, 8)))
    for heads, kv in ((16, 4), (12, 3), (12, 1)):
        assert takes(heads, kv, [256]) and not takes(heads, kv, [254])                           # one round: 128 keys
        assert not takes(heads, kv, [300] * 18) and takes(heads, kv, [512] * 9)                  # two
        assert not takes(heads, kv, [512] * 50) and takes(heads, kv, [896] * 36)                 # three and more
        assert takes(heads, kv, [200] * 32 + [400] * 32) and not takes(heads, kv, [200] * 33 + [400] * 33)  # in order: up to 64 portions
        assert takes(heads, kv, [64] * 128, behind=300) and not takes(heads, kv, [64] * 128)
    assert takes(16, 4, [1] * 1023 + [300], 384, 65535) and not takes(16, 4, [1] * 1023 + [300], 0, 65535)  # (as far as shapes tell)


def test_blocks_go_in_order_where_they_do_not_begin_together(plan):
    assert not plan.in_order(16, 1, 4096) and plan.in_order(16, 1, 4097) and plan.in_order(12, 64, 65) and not plan.in_order(12, 65, 4096)
    assert not plan.in_order(8, 2, 4096) and plan.in_order(8, 2, 4097) and not plan.in_order(8, 64, 128) and plan.in_order(4, 64, 129)
