"""Decode over narrow tables (``decode_short.h``): how a launch is divided (``plan_short_splits`` of ``decode_plan.h``) on the CPU; on the device
lengths around the edges of tiles, waves and runs against the oracle, for every kind of pool, head size and group that the kernel takes, and the
two passes as separate calls."""

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
extern "C" int runs(int batch, int hq, int hkv, int d, int bytes, long long blocks, int bs, int window, int cap) {
    const HeadPlan h = plan_heads(hq, hkv, d, bytes);
    return plan_short_splits(batch, h, plan_workspace(batch, h, plan_pad_dim(d), cap), bytes, blocks, bs, window, 256);
}
extern "C" int fits(int batch, int hq, int hkv, int d, int bytes, int runs, int cap) {  // the runs' results into the workspace's partials
    const HeadPlan h = plan_heads(hq, hkv, d, bytes);
    const WsPlan w = plan_workspace(batch, h, plan_pad_dim(d), cap);
    const size_t rows = (size_t)batch * hq * runs;
    return w.ml_off + rows * 8 <= w.acc_off && w.acc_off + rows * d * 4 <= w.total;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    at = tmp_path_factory.mktemp("short")
    (at / "s.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "research_amd", "csrc"), "-o", str(at / "s.so"),
                    str(at / "s.cpp")], check=True)
    lib = ctypes.CDLL(str(at / "s.so"))
    lib.runs.argtypes = [ctypes.c_int] * 5 + [ctypes.c_longlong] + [ctypes.c_int] * 3
    return lib


def test_lines_of_the_rule(plan):
    runs = lambda batch, shape, keys, bs=16, window=0, cap=4096: plan.runs(batch, *shape, keys // bs, bs, window, cap)
    wide, many, fp8, one = (32, 8, 128, 2), (14, 2, 64, 2), (32, 8, 128, 1), (8, 8, 64, 2)
    assert runs(1, wide, 592) == 1 and runs(1, wide, 608) == 4 and runs(1, wide, 4096) == 32 and runs(4, wide, 4096) == 8
    assert runs(16, wide, 1024) == 3 and runs(32, wide, 608) == 0 and runs(32, wide, 592) == 1 and runs(256, wide, 256) == 1 and runs(256, wide, 272) == 0
    assert runs(4, wide, 4096 + 16) == 0 and runs(1, wide, 1 << 20) == 0                      # long runs: the split pass
    assert runs(1, many, 16384) == 64 and runs(256, many, 3072) == 1 and runs(256, many, 3088) == 0
    four, eight, one8, two8 = (28, 4, 64, 2), (56, 8, 64, 2), (8, 8, 64, 1), (32, 16, 64, 1)  # (kv heads that a wave of the split pass takes at once)
    assert runs(256, four, 2048) == 1 and runs(256, four, 2064) == 0 and runs(256, eight, 1664) == 1 and runs(256, eight, 1680) == 0
    assert runs(64, one8, 768) == 1 and runs(64, one8, 784) == 0 and runs(64, two8, 512) == 1 and runs(64, two8, 528) == 0  # (32 MB in all)
    assert runs(16, fp8, 2048) == 3 and runs(1, one, 1200) == 1 and runs(96, one, 1216) == 0
    assert runs(1, wide, 1 << 20, window=500) == 1 and runs(1, wide, 1 << 20, window=-1024) == 8
    assert runs(4, wide, 64, bs=8) == 0 and runs(4, wide, 96, bs=48) == 1 and runs(513, wide, 16) == 0 and runs(4, wide, 0) == 1
    assert runs(4, (8, 2, 32, 2), 64) == runs(4, (3, 1, 8, 2), 64) == 0 and runs(4, (8, 2, 40, 2), 64) == 1  # (weights of 32 bits)
    assert runs(1, (8, 2, 128, 2), 4096) == 32 and runs(1, (8, 2, 128, 2), 4112) == 0


def test_lines_of_wide_groups_and_of_32_bits(plan):
    runs = lambda batch, shape, keys: plan.runs(batch, *shape, keys // 16, 16, 0, 4096)
    two, fp8 = (16, 2, 128, 2), (16, 2, 128, 1)  # eight query heads a kv head: long runs are cut in two while a unit has one workgroup or none
    assert runs(37, two, 6176) == 10 and runs(106, two, 1360) == 2 and runs(129, two, 1360) == 1 and runs(17, fp8, 12256) == 14 and runs(38, (14, 2, 256, 1), 4320) == 5
    assert runs(200, two, 1664) == 1 and runs(200, two, 1680) == 0                                     # 416 KB
    assert runs(68, (32, 8, 256, 1), 576) == 1 and runs(93, (32, 8, 128, 1), 768) == 1 and runs(93, (32, 8, 128, 1), 1040) == 0
    assert runs(3, (32, 8, 64, 2), 800) == 1 and runs(3, (32, 8, 64, 2), 816) == 6
    f32, wide = (14, 2, 64, 4), (32, 8, 128, 4)
    assert runs(4, f32, 512) == 1 and runs(4, f32, 528) == 4 and runs(4, wide, 256) == 1 and runs(4, wide, 272) == 4 and runs(140, (14, 2, 72, 4), 1600) == 3
    # the longest run that a batch may wait for: 384 KB of few sequences and where most units have a workgroup, else 192; above 64 elements 832 and 416
    assert runs(1, f32, 98352) == 64 and runs(1, f32, 98368) == 0 and runs(4, f32, 49168) == 32 and runs(4, f32, 49184) == 0 and runs(4, (8, 2, 32, 4), 64) == 1
    assert runs(5, f32, 19216) == 25 and runs(5, f32, 19232) == 0 and runs(63, f32, 6144) == 8 and runs(63, f32, 6160) == 0
    assert runs(64, f32, 12288) == 8 and runs(64, f32, 12304) == 0 and runs(1, (14, 2, 32, 4), 49200) == 64 and runs(1, (14, 2, 32, 4), 49216) == 0
    assert runs(15, (40, 8, 128, 4), 6656) == 8 and runs(15, (40, 8, 128, 4), 6672) == 0 and runs(16, (40, 8, 128, 4), 13312) == 8 and runs(16, (40, 8, 128, 4), 13328) == 0
    assert runs(200, (14, 2, 256, 4), 1664) == 2 and runs(200, (14, 2, 256, 4), 1680) == 0
    assert runs(3, wide, 3520) == 10 and runs(3, wide, 3536) == 0 and runs(3, (32, 8, 64, 4), 7040) == 10 and runs(3, (32, 8, 64, 4), 7056) == 0  # (176 KB)
    assert runs(7, wide, 33776) == runs(206, (32, 8, 64, 4), 64) == runs(16, (8, 8, 64, 4), 608) == runs(2, (8, 2, 128, 4), 4000) == 0


def test_results_of_the_runs_fit_the_workspace(plan):
    rng, took = np.random.default_rng(0), {1: 0, 2: 0, 4: 0}
    for _ in range(20000):
        hkv, rep = int(rng.choice([1, 2, 3, 4, 8, 16, 40])), int(rng.choice([1, 2, 3, 4, 5, 7, 8, 12, 16, 17, 40]))
        bytes_ = int(rng.choice([1, 2, 4]))
        d = int(rng.choice([64, 128, 256] if bytes_ == 1 else [8, 16, 24, 32, 40, 64, 72, 96, 128, 192, 256]))  # (32 bits: of up to 32 as of 64)
        bs, window = int(rng.choice([16, 32, 48, 256])), int(rng.choice([0, 0, 200, -5000]))
        batch, cap = int(rng.integers(1, 513)) if rng.random() < 0.5 else int(rng.integers(1, 9)), int(rng.choice([64, 512, 4096]))
        n = plan.runs(batch, hkv * rep, hkv, d, bytes_, int(2 ** rng.uniform(0, 14)), bs, window, cap)
        took[bytes_] += n > 1
        assert 0 <= n <= 64 and (n == 0 or plan.fits(batch, hkv * rep, hkv, d, bytes_, n, cap)), (batch, hkv, rep, d, bytes_, bs, window, cap, n)
    assert min(took.values()) > 500, took


EDGES = [1, 15, 16, 17, 31, 32, 33, 0, 47, 63, 64, 65, 127, 128, 129, 200, 255, 256, 257]
CASES = [(EDGES, *shape, kv, window, bs) for shape, kv, window, bs in [
    ((14, 2, 64), "bf16", 0, 16), ((32, 8, 128), "bf16", 0, 16), ((32, 8, 128), "f16", 50, 16), ((8, 2, 72), "f16", 0, 48), ((4, 4, 40), "bf16", -64, 16),
    ((20, 1, 96), "bf16", 0, 32), ((36, 2, 128), "f16", 0, 16), ((14, 2, 256), "bf16", 33, 16), ((32, 2, 256), "f16", 0, 16), ((6, 2, 192), "bf16", 0, 16),
    ((16, 8, 128), "fp8", 0, 16), ((14, 2, 256), "fp8", 17, 16), ((16, 16, 64), "fp8", 0, 32), ((34, 2, 64), "fp8", -48, 16), ((3, 1, 40), "f16", 0, 16),
]] + [
    ([1300, 2047, 1, 0, 16], 32, 8, 128, "bf16", 0, 16), ([4000, 129, 128], 14, 2, 64, "bf16", 0, 16), ([3000, 17], 16, 2, 128, "fp8", 0, 16),
    ([1025, 700, 64, 3], 14, 2, 256, "f16", 0, 16), ([5000, 2, 0], 14, 2, 64, "f16", 1500, 16), ([2500, 1200], 18, 1, 128, "bf16", -1300, 16),
    ([2000, 900, 1] * 30, 14, 2, 64, "fp8", 0, 16),
]


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hq,hkv,d,kv,window,bs", CASES)
def test_against_the_oracle(plan, lens, hq, hkv, d, kv, window, bs):
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce, assert_close, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"decode short: {len(lens)} x {max(lens)} {hq}/{hkv}x{d} {kv} window {window} blocks of {bs}")
    b = Batch(lens, hq, hkv, d, kv, seed=len(lens) + d, bs=bs)
    (k, v, ks, vs), (kr, vr) = b.device_pools()
    tables = tables_to_device(b.tables)
    assert plan.runs(len(lens), hq, hkv, d, 1 if kv == "fp8" else 2, tables.shape[1], bs, window, 4096) > 0
    holes = [list(t) for t in b.tables]
    if not window:  # blocks that are not there count as zero keys: a negative id, one past the pool
        for t in holes[:3]:
            if len(t) > 1:
                t[len(t) // 2] = -1
        holes[-1][:1] = [b.num_blocks] if holes[-1] else []
    spare = (set(range(b.num_blocks)) - {x for t in b.tables for x in t}).pop()  # (the oracle's zero keys)
    kr, vr = kr.float().clone(), vr.float().clone()
    kr[spare * bs: (spare + 1) * bs] = vr[spare * bs: (spare + 1) * bs] = 0
    q, n = b.q.to(DEV), torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    for t, ez in ((b.tables, None), (holes, None)) + (() if window else ((b.tables, max(lens) - n),)):
        ws = ops.decode_workspace(q, k)
        first = [(x - 1) // -window * -window if window < 0 and x else 0 for x in b.lens]
        if window < 0 and any(f % bs for f in first):
            continue  # (the oracle's stand-in for chunks, below, wants whole blocks)
        call = (k, v, tables_to_device(t), n, bs, b.scale, ws, ez, ks, vs)
        got = ops.decode(q, *call, window=window)
        want = po.paged_decode(b.q.float(), kr, vr, [[x if 0 <= x < b.num_blocks else spare for x in r[f // bs:]] for r, f in zip(t, first)],
                               [x - f for x, f in zip(b.lens, first)], bs, b.scale, pad_zero_keys=ez is not None, window=max(window, 0))
        # (weights carry 16 or more bits, sums are of 32: what is left is the output's rounding, half a unit of 2^-8 or 2^-11, doubled for sums)
        assert_close(got, want, 2.0 ** (-10 if kv == "f16" else -7), "one call")
        for i, x in enumerate(b.lens):
            assert x or not got[i].any()
        two = torch.full_like(q, float("nan"))
        for entry in ("pa_decode_split", "pa_decode_reduce"):
            ops.decode(q, *call, out=two, entry=entry, window=window)
        assert_close(two, got.double().cpu().numpy(), 2.0 ** (-10 if kv == "f16" else -7), "two calls")
        assert torch.equal(ops.decode(q, *call, window=window), got)
    # an output that starts between two 8-byte words
    room = torch.full((q.numel() + 1,), 7.0, dtype=q.dtype, device=DEV)
    out = room[1:].view(q.shape)
    call = (k, v, tables, n, bs, b.scale, ws, None, ks, vs)
    assert torch.equal(ops.decode(q, *call, out=out, window=window), ops.decode(q, *call, window=window)) and float(room[0]) == 7.0


@pytest.mark.gpu
def test_rows_that_are_not_seen_do_not_matter():
    """NaN and infinities in a block's rows past a sequence's end and ahead of its window."""
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce

    announce("decode short: rows out of sight")
    for dtype, window in ((torch.bfloat16, 0), (torch.float16, 37), (torch.bfloat16, -40)):
        gen = torch.Generator().manual_seed(5)
        n = [50, 33, 700, 1]
        k, v = (torch.randn(1024, 2, 64, generator=gen).to(dtype) for _ in range(2))
        tables = torch.arange(64, dtype=torch.int32).view(1, 64)[:, :48].repeat(4, 1)
        for i in range(4):  # every sequence its own call: the same pool, other rows out of sight
            kk, vv = k.clone(), v.clone()
            first = max(0, n[i] - window) if window > 0 else (n[i] - 1) // 40 * 40 if window < 0 else 0
            for t in (kk, vv):
                t[n[i]:] = float("nan")
                t[:first] = float("inf")
            q = torch.randn(1, 14, 64, generator=gen).to(dtype).to(DEV)
            call = lambda a, b: ops.decode(q, a.to(DEV), b.to(DEV), tables[:1].to(DEV), torch.tensor([n[i]], dtype=torch.int32, device=DEV), 16, 0.125,
                                           ops.decode_workspace(q, a.to(DEV)), window=window)
            assert torch.equal(call(kk, vv), call(k, v))


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hq,hkv,d,window,bs", [
    (EDGES, 14, 2, 64, 0, 16), (EDGES, 32, 8, 128, 50, 16), (EDGES, 8, 2, 72, 0, 48), (EDGES, 4, 4, 32, -64, 16), (EDGES, 6, 2, 8, 0, 16),
    (EDGES, 20, 1, 96, 0, 32), (EDGES, 36, 2, 128, 0, 16), (EDGES, 14, 2, 256, 33, 16), (EDGES, 6, 2, 192, 0, 16), ([1300, 2047, 1, 0, 16], 32, 8, 128, 0, 16),
    ([4000, 129, 128], 14, 2, 64, 0, 16), ([1025, 700, 64, 3], 14, 2, 256, 0, 16), ([2500, 1200], 18, 1, 128, -1300, 16), ([1500, 40], 8, 2, 40, 0, 16),
])
def test_pools_of_32_bits(plan, lens, hq, hkv, d, window, bs):
    """The same edges over 32-bit pools, with rows out of sight that are NaN or infinite; errors against 64 bits beside the split pass's."""
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce, assert_close, decode_by_split_pass, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"decode short, 32 bits: {len(lens)} x {max(lens)} {hq}/{hkv}x{d} window {window} blocks of {bs}")
    b = Batch(lens, hq, hkv, d, "f32", seed=len(lens) + d, bs=bs)
    (k, v, _, _), (kr, vr) = b.device_pools()
    tables = tables_to_device(b.tables)
    assert plan.runs(len(lens), hq, hkv, d, 4, tables.shape[1], bs, window, 4096) > 0
    q, n = b.q.to(DEV), torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    ws, want = ops.decode_workspace(q, k), np.zeros((len(lens), hq, d))
    for i, x in enumerate(b.lens):
        first = max(0, x - window) if window > 0 else (x - 1) // -window * -window if window < 0 and x else 0
        rows = np.array([b.tables[i][j // bs] * bs + j % bs for j in range(first, x)], dtype=np.int64)
        for pool in (k, v):  # (blocks are a sequence's own)
            own = np.array([c * bs + r for c in b.tables[i] for r in range(bs)], dtype=np.int64)
            pool[torch.from_numpy(np.setdiff1d(own, rows)).to(DEV)] = float("nan") if i % 2 else float("inf")
        if x:
            kk, vv = (t.double().cpu().numpy().reshape(-1, hkv, d)[rows].repeat(hq // hkv, axis=1) for t in (kr, vr))
            s = np.einsum("hd,jhd->hj", b.q[i].double().numpy(), kk) * b.scale
            w = np.exp(s - s.max(axis=1, keepdims=True))
            want[i] = np.einsum("hj,jhd->hd", w / w.sum(axis=1, keepdims=True), vv)
    call = (k, v, tables, n, bs, b.scale, ws)
    got = ops.decode(q, *call, window=window)
    other = decode_by_split_pass(q, k, v, b.tables, b.lens, bs, b.scale, window=window)[0]
    # (logits of 32 bits and of at most about 30, so weights to 2^-19 of themselves; sums of up to 4000 terms, in parts)
    assert_close(got, want, 1e-5, "against 64 bits")
    # (0.95 of the split pass's on average; a call's few hundred rows, whose logits share an error, scatter about that by a tenth)
    err = [np.sqrt(((t.double().cpu().numpy() - want) ** 2).mean()) for t in (got, other)]
    assert err[0] <= 1.25 * err[1], err
    two = torch.full_like(q, float("nan"))
    for entry in ("pa_decode_split", "pa_decode_reduce"):
        ops.decode(q, *call, out=two, entry=entry, window=window)
    assert_close(two, got, 1e-6, "two calls")
    assert torch.equal(ops.decode(q, *call, window=window), got) and not got[[x == 0 for x in b.lens]].any()
    room = torch.full((q.numel() + 1,), 7.0, device=DEV)  # an output that starts between two 8-byte words
    assert torch.equal(ops.decode(q, *call, out=room[1:].view(q.shape), window=window), got) and float(room[0]) == 7.0
    if not window:  # padding positions and blocks that are not there are zero keys
        clean, ez = (kr.float().to(DEV), vr.float().to(DEV)), max(lens) - n
        t = [[-1 if j == len(x) // 2 and len(x) > 1 else c for j, c in enumerate(x)] for x in b.tables]
        spare = (set(range(b.num_blocks)) - {x for y in b.tables for x in y}).pop()
        kz, vz = kr.float().clone(), vr.float().clone()
        kz[spare * bs: (spare + 1) * bs] = vz[spare * bs: (spare + 1) * bs] = 0
        got = ops.decode(q, *clean, tables_to_device(t), n, bs, b.scale, ws, ez)
        want = po.paged_decode(b.q, kz, vz, [[spare if c < 0 else c for c in x] for x in t], b.lens, bs, b.scale, pad_zero_keys=True)
        assert_close(got, want, 1e-5, "zero keys")


@pytest.mark.gpu
@pytest.mark.parametrize("bits", [12, 20, 24, 31, 40, 60])
@pytest.mark.parametrize("lens,hq,hkv,d", [([300, 40, 1, 0, 17], 14, 2, 64), ([1100, 40], 8, 2, 128), ([200, 64], 6, 1, 256)])
def test_far_logits_of_32_bits(plan, lens, hq, hkv, d, bits):
    """Logits about 2^bits, whose own rounding is much of a power of two or more: the largest key's value is what remains."""
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce, assert_close, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"decode short, 32 bits: logits of 2^{bits}, {hq}/{hkv}x{d}")
    b = Batch(lens, hq, hkv, d, "f32", seed=bits)
    (k, v, _, _), (kr, vr) = b.device_pools()
    tables = tables_to_device(b.tables)
    assert plan.runs(len(lens), hq, hkv, d, 4, tables.shape[1], 16, 0, 4096) > 0
    q, n = b.q * 2.0 ** bits, torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    want, tied = np.zeros((len(lens), hq, d)), np.zeros((len(lens), hq, 1), dtype=bool)
    for i, x in enumerate(b.lens):
        if x:
            rows = np.array([b.tables[i][j // 16] * 16 + j % 16 for j in range(x)], dtype=np.int64)
            kk, vv = (t.double().cpu().numpy().reshape(-1, hkv, d)[rows].repeat(hq // hkv, axis=1) for t in (kr, vr))
            s = np.einsum("hd,jhd->hj", q[i].double().numpy(), kk) * b.scale
            w = np.exp(s - s.max(axis=1, keepdims=True))
            want[i] = np.einsum("hj,jhd->hd", w / w.sum(axis=1, keepdims=True), vv)
            # (a sum of d products of 32 bits errs by less than d 2^-23 of the largest logit: rows whose two largest keys are closer have no one answer)
            top = np.sort(np.concatenate([s, s[:, :1] * 0 - np.inf], axis=1), axis=1)[:, -2:]
            tied[i, :, 0] = top[:, 1] - top[:, 0] < 16 + d * 2.0 ** -22 * np.abs(s).max(axis=1)
    got = ops.decode(q.to(DEV), k, v, tables, n, 16, b.scale, ops.decode_workspace(q.to(DEV), k)).double().cpu().numpy()
    assert np.isfinite(got).all() and tied.mean() < 0.25
    assert_close(np.where(tied, want, got), want, 1e-5, "the largest key's value")


@pytest.mark.gpu
@pytest.mark.parametrize("kv", ["bf16", "f32"])
@pytest.mark.parametrize("runs,batch", [(8, 16), (9, 14), (16, 8), (18, 7), (32, 4), (42, 3), (64, 2)])
def test_runs_that_several_waves_merge(plan, runs, batch, kv):
    """Around the eights of runs that a wave of the merge takes, with runs that hold no key and positions that count as zero keys."""
    from oracle import paged_oracle as po
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce, assert_close, tables_to_device
    from tests.test_gpu_decode_merge import Batch

    announce(f"decode short: {runs} runs, {kv}")
    most = 8180 if kv == "bf16" or runs > 9 else 6100
    b = Batch([most, 40] + [i % 3 for i in range(batch - 2)], 14, 2, 64, kv, seed=runs)
    (k, v, _, _), _ = b.device_pools()
    tables = tables_to_device(b.tables)
    assert plan.runs(batch, 14, 2, 64, 4 if kv == "f32" else 2, tables.shape[1], 16, 0, 4096) == runs
    q, n = b.q.to(DEV), torch.tensor(b.lens, dtype=torch.int32, device=DEV)
    for ez in (None, most - n):
        got = ops.decode(q, k, v, tables, n, 16, b.scale, ops.decode_workspace(q, k), ez)
        want = po.paged_decode(b.q.float(), b.k.float(), b.v.float(), b.tables, b.lens, 16, b.scale, pad_zero_keys=ez is not None)
        # (16 bits: the output's rounding, half a unit of 2^-8, doubled for sums)
        assert_close(got, want, 1e-5 if kv == "f32" else 2.0 ** -7, "merged")
