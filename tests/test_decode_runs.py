"""Short launches of the split pass: runs of blocks, one workgroup each (``plan_run_blocks`` of ``decode_plan.h``, compiled with
g++).  Every (plane, sequence, block) lies in one run of one workgroup, and where the runs fit the grid no workgroup has two.
The waves of a workgroup fill the prefix table of runs without a barrier, so no word of it is ever stored with two values
(``plan_wave_prefix``).  On the device: launches of runs of two and four blocks, merged in either way."""

import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include <vector>
#include "decode_plan.h"
using namespace pa_decode_detail;
extern "C" int replay(const int *lens, int batch, int planes, int bs, int window, int grid) {
    auto runs = [&](int u) { int64_t n = 0; for (int b = 0; b < batch; ++b) n += plan_runs_of(plan_blocks_of(lens[b], bs, window), u); return n * planes; };
    const int64_t blocks = runs(1);
    const int u = plan_run_blocks(blocks, (int64_t)planes * batch, grid, runs);
    const int64_t total = runs(u), per_plane = total / planes;
    if (total == 0) return u;
    const int taking = plan_run_grid(total, grid);
    std::vector<std::vector<int>> seen((size_t)planes * batch);
    for (int i = 0; i < planes * batch; ++i) seen[i].resize(plan_blocks_of(lens[i % batch], bs, window));
    for (int w = 0; w < taking; ++w) {
        const int64_t lo = plan_unit_begin(w, total, taking), hi = plan_unit_begin(w + 1, total, taking);
        if (hi <= lo || (u > 1 && hi != lo + 1)) return -1;
        for (int64_t x = lo; x < hi; ++x) {
            if (plan_owner_of(x, total, taking) != w) return -2;
            int64_t off = x % per_plane;
            int b = 0;
            for (int n; off >= (n = plan_runs_of(plan_blocks_of(lens[b], bs, window), u)); ++b) off -= n;
            std::vector<int> &s = seen[x / per_plane * batch + b];
            for (int64_t k = off * u; k < (off + 1) * u && k < (int64_t)s.size(); ++k) ++s[k];
        }
    }
    for (auto &s : seen) for (int n : s) if (n != 1) return -3;
    return u;
}
// Every store that a wave makes to the prefix table, in order.  A wave reads the table behind its own stores, while another one may
// still have all of its own before it: each of them has to store what is already there.
extern "C" int stores(const int *lens, int batch, int planes, int bs, int window, int grid) {
    std::vector<std::vector<int>> stored(batch);
    int run = 0;
    auto scan = [&](int u, bool keep) {
        int carry = 0;
        for (int b = 0; b < batch; ++b) {
            if (keep) stored[b].push_back(carry);
            carry += plan_runs_of(plan_blocks_of(lens[b], bs, window), u);
        }
        return carry;
    };
    const int total = plan_wave_prefix(planes, batch, grid, run, scan);
    for (int b = 0, before = 0; b <= batch; ++b) {
        if (b == batch) return total == before ? run : -1;
        if (stored[b].empty()) return -2;
        for (int x : stored[b]) if (x != before) return -3;
        before += plan_runs_of(plan_blocks_of(lens[b], bs, window), run);
    }
    return -4;
}
"""


@pytest.fixture(scope="module")
def replay(tmp_path_factory):
    at = tmp_path_factory.mktemp("runs")
    (at / "r.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "r.so"),
                    str(at / "r.cpp")], check=True)
    lib = ctypes.CDLL(str(at / "r.so"))
    for fn in (lib.replay, lib.stores):
        fn.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 5

    def run(lens, planes, bs=16, window=0, grid=512):
        lens = np.ascontiguousarray(lens, np.int32)
        u = lib.replay(lens.ctypes.data, len(lens), planes, bs, window, grid)
        assert lib.stores(lens.ctypes.data, len(lens), planes, bs, window, grid) == u
        return u
    return run


@pytest.mark.parametrize("seed", range(4))
def test_every_block_lies_in_one_run(replay, seed):
    rng = np.random.default_rng(seed)
    taken = set()
    for _ in range(300):
        batch = int(rng.integers(1, 65))
        lens = np.exp(rng.uniform(0, np.log(rng.choice([40, 600, 8000])), batch)).astype(int) - 1  # (some are empty)
        u = replay(lens, int(rng.choice([1, 2, 4])), int(rng.choice([1, 16, 32])), int(rng.choice([0, 0, 100, -64])), int(rng.choice([2, 64, 512])))
        assert u in (1, 2, 4)
        taken.add(u)
    assert taken == {1, 2, 4}


def test_lines_of_the_rule(replay):
    assert replay([16] * 512, 1) == 1 and replay([32] * 256, 1) == 1    # a run per block fills the grid
    assert replay([32] * 512, 1) == 2 and replay([64] * 512, 1) == 4    # two, four blocks each
    assert replay([80] * 512, 1) == 1                                   # more than the grid takes in runs of four
    assert replay([768], 1) == 1 and replay([784], 1) == 4              # 48 and 49 blocks of a sequence
    assert replay([0, 0], 2) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("run,lens,hq,hkv,d,kv", [
    (2, [100] * 64, 32, 8, 128, "bf16"),                 # two launches
    (4, [4096], 32, 8, 128, "bf16"),
    (4, [2000, 0, 1999, 2000, 1], 32, 8, 128, "f16"),
    (4, [1000] * 16, 14, 2, 64, "bf16"),
    (2, [700] * 16, 8, 2, 64, "f32"),
    (2, [50, 49, 64, 33] * 32, 32, 8, 128, "bf16"),      # the pieces merged in the one launch
    (4, [128, 113, 97, 128] * 32, 32, 8, 128, "bf16"),
])
def test_launches_of_runs_on_the_device(replay, run, lens, hq, hkv, d, kv):
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, WIDE, announce, assert_close, decode_route, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    planes = {(32, 8, 128): 2, (14, 2, 64): 1, (8, 2, 64): 1}[hq, hkv, d]
    assert replay(lens, planes, grid=2 * torch.cuda.get_device_properties(0).multi_processor_count) == run
    announce(f"decode runs of {run}: {len(lens)} x {lens[0]} {hq}/{hkv}x{d} {kv}")
    b = Batch(lens, hq, hkv, d, kv, seed=run)
    (k, v, _, _), _ = b.device_pools()
    q, n = b.q.to(DEV), torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    ws, tables = ops.decode_workspace(q, k), tables_to_device(b.tables, WIDE)
    assert decode_route(len(lens), hq, hkv, d, q.dtype, k.dtype, WIDE, b.bs) == 0
    got = ops.decode(q, k, v, tables, n, b.bs, b.scale, ws)
    assert_close(got, po.paged_decode(b.q, b.k, b.v, b.tables, b.lens, b.bs, b.scale), b.tol, "runs of blocks")
    assert torch.equal(ops.decode(q, k, v, tables, n, b.bs, b.scale, ws), got)


@pytest.mark.gpu
@pytest.mark.parametrize("queries", ["bf16", "f16"])
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(14, 2), (16, 2), (32, 4), (8, 1), (64, 8)])
def test_pieces_of_wide_groups_over_fp8_pools(hq, hkv, d, queries):
    """Up to eight query heads per kv head: kernels that have no registers to spare, sequences in one piece and in several, merged in
    a second launch and in the one."""
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, WIDE, announce, assert_close, decode_route, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"fp8 pieces {hq}/{hkv}x{d} {queries}")
    for lens in ([12, 33, 16, 100], [300, 20, 40], [40, 17, 90, 5] * 70):
        b = Batch(lens, hq, hkv, d, "fp8", seed=d)
        (k, v, ks, vs), (kr, vr) = b.device_pools()
        q = b.q.to(torch.float16 if queries == "f16" else torch.bfloat16)
        assert decode_route(len(lens), hq, hkv, d, q.dtype, k.dtype, WIDE, b.bs) == 0
        got = ops.decode(q.to(DEV), k, v, tables_to_device(b.tables, WIDE), torch.tensor(b.lens, dtype=torch.int32, device=DEV), b.bs, b.scale,
                         ops.decode_workspace(q.to(DEV), k), None, ks, vs)
        # (weights are multiplied by scales and packed to 16 bits: 2^-9 of values of at most 4)
        assert_close(got, po.paged_decode(q.float(), kr.float(), vr.float(), b.tables, b.lens, b.bs, b.scale), 2e-2, f"{len(lens)} sequences")
