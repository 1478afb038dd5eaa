"""Decode with narrow block tables that the kernel for them does not take (blocks that are no whole tiles of 16 keys, 16-bit heads of up to 32, large
batches): a workgroup of the split pass takes a whole (plane, sequence), and one launch does (``plan_whole_sequences`` of ``decode_plan.h``).
The rule's lines on the CPU; on the device the same batch with narrow tables and with tables padded beyond the rule's line, which take the
split pass in ranges and the merge, against the oracle and against each other."""

import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "decode_plan.h"
using namespace pa_decode_detail;
extern "C" int whole(int batch, int hq, int hkv, int d, int bytes, long long table_blocks, int bs, int window) {
    return plan_whole_sequences(batch, plan_heads(hq, hkv, d, bytes), d, bytes, table_blocks, bs, window);
}
"""


@pytest.fixture(scope="module")
def whole(tmp_path_factory):
    at = tmp_path_factory.mktemp("whole")
    (at / "w.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "w.so"),
                    str(at / "w.cpp")], check=True)
    fn = ctypes.CDLL(str(at / "w.so")).whole
    fn.argtypes = [ctypes.c_int] * 5 + [ctypes.c_longlong] + [ctypes.c_int] * 2
    return lambda batch, shape, blocks, bs=16, window=0: bool(fn(batch, *shape, blocks, bs, window))


def test_lines_of_the_rule(whole):
    small, wide, f32 = (14, 2, 64, 2), (32, 8, 128, 2), (8, 2, 128, 4)  # 512, 2048 and 2048 bytes a key and plane
    assert whole(4, small, 16) and not whole(4, small, 17) and whole(16, small, 24) and not whole(16, small, 25)
    assert whole(4, wide, 6) and not whole(4, wide, 7)
    assert whole(4, f32, 4) and not whole(4, f32, 5)
    assert whole(96, wide, 12) and not whole(96, wide, 13) and not whole(95, wide, 7)
    assert whole(512, f32, 12) and not whole(511, f32, 5)
    assert whole(512, small, 48) and not whole(513, small, 1)
    assert whole(4, wide, 1 << 40, window=64) and not whole(4, wide, 1 << 40, window=81)  # (six blocks hold any 64 keys)
    assert whole(4, wide, 1 << 40, window=-64) and whole(4, wide, 16, bs=1) and not whole(4, wide, 17, bs=1)
    assert whole(8, wide, 32, bs=1) and not whole(8, wide, 33, bs=1) and whole(200, wide, 64, bs=1) and not whole(200, wide, 65, bs=1)
    assert whole(4, small, 2, bs=100) and not whole(4, small, 3, bs=100)                # (seven tiles of 16 each)
    fp8, d32 = (16, 2, 64, 1), (8, 2, 32, 2)  # eight query heads a kv head over fp8; the generic loop over 16 bits
    assert whole(4, fp8, 8) and not whole(4, fp8, 9) and whole(16, fp8, 16) and not whole(16, fp8, 17)
    assert all(whole(b, d32, 12) and not whole(b, d32, 13) for b in (1, 64)) and whole(200, d32, 32) and not whole(200, d32, 33)
    assert whole(1024, wide[:3] + (1,), 1) is False and not whole(500, (16, 8, 256, 2), 7) and whole(256, (16, 8, 256, 2), 12)  # (1024 workgroups)


CASES = [
    ([1, 2, 24, 47], 14, 2, 64, "bf16", 0, 8),              # (and where a workgroup's ranges end in the split pass: 0, 15, 16, 17)
    ([0, 96, 17, 16, 15, 0, 1, 81], 32, 8, 128, "bf16", 0, 8),
    ([64, 0, 33, 1], 8, 2, 128, "f32", 0, 8),
    ([96, 5, 0, 48], 16, 8, 128, "fp8", 0, 8),
    ([60, 1, 33], 16, 2, 64, "fp8", 0, 8),
    ([90, 16, 0, 31], 16, 8, 256, "f16", 0, 8),
    ([190, 3, 0, 129], 8, 2, 72, "f16", 0, 24),
    ([40, 64, 1, 0], 4, 4, 32, "f32", 0, 8),
    ([48, 7, 0, 25], 14, 2, 64, "f32", 0, 24),
    ([40, 64, 1, 0], 4, 4, 32, "bf16", 0, 16),
    ([5000, 63, 0, 64, 65, 999], 32, 8, 128, "bf16", 64, 8),  # (long tables, a short window)
    ([130, 64, 0, 65, 127], 32, 8, 128, "bf16", -64, 8),
    ([192, 17, 0, 100, 1, 64] * 64, 32, 8, 128, "bf16", 0, 16),  # more workgroups than the split pass has
    ([192, 17, 0, 100, 1, 64] * 50, 32, 8, 128, "bf16", 0, 8),
    ([64, 50, 49, 33] * 32, 32, 8, 128, "f16", 0, 8),
    ([40, 17, 90, 5] * 70, 14, 2, 64, "fp8", 0, 8),
]


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hq,hkv,d,kv,window,bs", CASES)
def test_narrow_and_wide_tables_agree(whole, lens, hq, hkv, d, kv, window, bs):
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, WIDE, announce, assert_close, decode_route, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"decode whole: {len(lens)} x {max(lens)} {hq}/{hkv}x{d} {kv} window {window} blocks of {bs}")
    b = Batch(lens, hq, hkv, d, kv, seed=len(lens) + d, bs=bs)
    (k, v, ks, vs), (kr, vr) = b.device_pools()
    q, n = b.q.to(DEV), torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    size = {"f32": 4, "fp8": 1}.get(kv, 2)
    narrow = tables_to_device(b.tables)
    assert whole(len(lens), (hq, hkv, d, size), narrow.shape[1], bs, window)
    assert decode_route(len(lens), hq, hkv, d, q.dtype, k.dtype, narrow.shape[1], bs, window) == -1
    ws, padding = ops.decode_workspace(q, k), max(lens) - n
    for ez in (None,) if window else (None, padding):
        got = ops.decode(q, k, v, narrow, n, b.bs, b.scale, ws, ez, ks, vs, window=window)
        first = [(n - 1) // -window * -window if window < 0 and n else 0 for n in b.lens]  # (chunks of whole blocks)
        want = po.paged_decode(b.q.float(), kr.float(), vr.float(), [t[f // b.bs:] for t, f in zip(b.tables, first)],
                               [n - f for n, f in zip(b.lens, first)], b.bs, b.scale, pad_zero_keys=ez is not None, window=max(window, 0))
        assert_close(got, want, b.tol if kv != "fp8" else 2e-2, "narrow tables")
        if not window:
            padded = tables_to_device(b.tables, WIDE)
            assert decode_route(len(lens), hq, hkv, d, q.dtype, k.dtype, WIDE, bs) == 0
            other = ops.decode(q, k, v, padded, n, b.bs, b.scale, ws, ez, ks, vs)
            # (both round to the type of q, at most 2^-8 of a value apart, weights to 16 bits on the way: 2^-9 of values of at most 5)
            assert_close(got, other.double().cpu().numpy(), 1e-5 if kv == "f32" else 2e-2, "wide tables")
        assert torch.equal(ops.decode(q, k, v, narrow, n, b.bs, b.scale, ws, ez, ks, vs, window=window), got)


@pytest.mark.gpu
def test_lengths_beyond_a_narrow_table_count_as_zero_keys():
    from research_amd import ops
    from tests.gpu_helpers import DEV, WIDE, announce, decode_route
    from tests.test_gpu_decode_merge import Batch

    announce("decode whole: lengths beyond the tables")
    b = Batch([64, 64, 64], 32, 8, 128, "bf16", seed=3, bs=8)
    (k, v, _, _), _ = b.device_pools()
    q = b.q.to(DEV)
    n = torch.tensor([64, 300, 2000], dtype=torch.int32, device=DEV)
    narrow = torch.tensor(b.tables, dtype=torch.int32, device=DEV)
    padded = torch.full((3, WIDE), -1, dtype=torch.int32, device=DEV)
    padded[:, :8] = narrow
    assert [decode_route(3, 32, 8, 128, q.dtype, k.dtype, t.shape[1], 8) for t in (narrow, padded)] == [-1, 0]
    ws = ops.decode_workspace(q, k)
    got, want = (ops.decode(q, k, v, t, n, b.bs, b.scale, ws).float() for t in (narrow, padded))
    assert (got - want).abs().max() < 2e-2 and torch.isfinite(got).all()
