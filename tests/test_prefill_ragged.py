"""Prompts of unequal length: how many groups of rows a workgroup of the matrix-core prefill takes (``plan_ragged_groups`` of
``prefill_plan.h``).  The rule's lines on the CPU; on the device the same rows with and without the rule, which must be the same bits, and
against the vector kernel."""

import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "prefill_plan.h"
using namespace pa_decode_detail;
extern "C" int ragged(int most, int hkv, int batch, long long rows, long long max_q, long long per, long long keys, long long groups) {
    return plan_ragged_groups(most, groups, hkv, batch, rows, max_q, per, keys, 64, 256);
}
extern "C" int turned(int y, int b, int n_chunks) { return plan_turned_chunk(y, b, n_chunks); }
"""


@pytest.fixture(scope="module")
def ragged(tmp_path_factory):
    at = tmp_path_factory.mktemp("ragged")
    (at / "r.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "r.so"),
                    str(at / "r.cpp")], check=True)
    fn = ctypes.CDLL(str(at / "r.so")).ragged
    fn.argtypes = [ctypes.c_int] * 3 + [ctypes.c_longlong] * 5
    return lambda *args, groups=1: fn(*args, groups)


@pytest.fixture(scope="module")
def turned(ragged, tmp_path_factory):
    fn = ctypes.CDLL(str(tmp_path_factory.getbasetemp() / "ragged0" / "r.so")).turned
    return fn


def test_lines_of_the_rule(ragged):
    assert ragged(8, 8, 64, 64 * 512, 512, 64, 512) == 8            # equal
    assert ragged(4, 8, 32, 32 * 224, 256, 64, 2304) == 4           # seven eighths
    assert ragged(4, 8, 32, 32 * 224 - 1, 256, 64, 2304) == 1
    assert ragged(8, 8, 64, 0, 512, 64, 512) == 8                   # rows not known
    assert ragged(1, 8, 64, 64, 512, 64, 512) == 1 and ragged(2, 8, 64, 64, 512, 64, 512) == 2 and ragged(3, 8, 64, 64, 512, 64, 512) == 1
    assert ragged(8, 8, 1024, 1024 * 100, 250, 64, 256) in (4, 5, 6, 7)  # hundreds of groups a unit: set-ups count again
    assert ragged(8, 1 << 20, 65535, 1, 65535, 0, 1 << 40) >= 1     # (no overflow, no division by nothing)
    # 300 query heads on one kv head, prompts of 65535 and 10 rows: 76800 groups, of which a launch takes no more than 65535 workgroups
    assert ragged(8, 1, 2, 65545, 65535, 0, 65536, groups=65535) == 1 and ragged(8, 1, 2, 65545, 65535, 0, 65536, groups=76800) == 2
    assert ragged(8, 1, 2, 65545, 65535, 0, 65536, groups=65535 * 8) == 8
    # nearly equal ones wait less for the last: three groups of 64 prompts of 153 rows on average, the longest 182; of 100 rows one
    assert ragged(3, 8, 64, 64 * 153, 182, 64, 192) == 3 and ragged(3, 8, 64, 64 * 100, 182, 64, 192) == 1
    for rows in range(1, 64 * 512, 997):
        assert 1 <= ragged(5, 8, 64, rows, 512, 36, 4096) <= 5


@pytest.mark.parametrize("kv_heads,chunks", [(8, 4), (2, 4), (2, 3), (1, 4), (4, 4), (8, 2), (16, 3), (1, 8), (2, 16), (1, 5), (3, 6)])
def test_first_chunks_spread_over_the_turns(turned, kv_heads, chunks):
    """Workgroups go to eight dies in turn and, in a die, to four engines: each gets its share of the chunks that every sequence has."""
    seqs = 128
    first = np.zeros((8, 4), int)
    for z in range(seqs):
        assert sorted(turned(y, z, chunks) for y in range(chunks)) == list(range(chunks))
        for y in range(chunks):
            for x in range(kv_heads):
                at = x + kv_heads * (y + chunks * z)
                first[at % 8, at // 8 % 4] += turned(y, z, chunks) == 0
    mean = kv_heads * seqs / 32
    assert first.max() <= 2 * mean, first  # (up to sixteen times the mean with the same chunk for the same y)


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,prefix,lens", [
    (32, 8, 128, 0, [1, 33, 64, 65, 500, 129, 250, 12] * 8),
    (14, 2, 64, 48, [1, 37, 300, 72, 36, 35] * 20),
    (16, 16, 32, 16, [31, 1, 200, 64] * 16),
    (8, 8, 96, 0, [256, 1, 2, 257, 64] * 10),
    (8, 2, 128, 32, [0, 40, 0, 200, 7] * 60),
])
def test_same_bits_without_the_rule(hq, hkv, d, prefix, lens):
    from research_amd import _lib, ops

    bs, gen = 16, torch.Generator().manual_seed(d + hq)
    q_lens = torch.tensor(lens, dtype=torch.int32)
    ctx = q_lens + prefix
    width = -(-int(ctx.max()) // bs)
    blocks = len(lens) * width
    tables = torch.randperm(blocks, generator=gen).to(torch.int32).view(len(lens), width).cuda()
    pool = [torch.randn(blocks * bs, hkv, d, generator=gen).to(torch.bfloat16).cuda() for _ in range(2)]
    total = int(q_lens.sum())
    q = torch.randn(total, hq, d, generator=gen).to(torch.bfloat16).cuda()
    starts = (torch.cumsum(q_lens, 0) - q_lens).to(torch.int32).cuda()
    q_lens, ctx = q_lens.cuda(), ctx.cuda()
    call = (q, *pool, tables, ctx, q_lens, starts, max(lens), bs, d ** -0.5)
    got = ops.prefill_paged(*call)
    want = torch.empty_like(q)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check("pa_prefill_paged", _lib.load().pa_prefill_paged(
        q.data_ptr(), pool[0].data_ptr(), pool[1].data_ptr(), want.data_ptr(), tables.data_ptr(), width, ctx.data_ptr(), q_lens.data_ptr(),
        starts.data_ptr(), None, len(lens), max(lens), hq, hkv, d, bs, blocks, d ** -0.5, 0, _lib.PA_BF16, stream))
    assert torch.equal(got, want)
    plain = ops.prefill_paged(*call, rowwise=True)
    # (a weight's and a result's rounding to 16 bits, 2^-9 each, over values of unit variance: 1e-2 of the result is far outside)
    err = (got.double() - plain.double()).norm() / plain.double().norm()
    assert float(err) < 1e-2, float(err)
