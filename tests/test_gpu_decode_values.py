"""Decode on values at the edges of the 16-bit types, on each way that a launch can take: a workgroup per sequence and runs with a merge
behind them (``decode_short.h``), and the split pass (``decode_impl.h``), which block tables far wider than the sequences lead to."""

import numpy as np
import pytest
import torch

from research_amd import ops
from tests.gpu_helpers import DEV, announce, assert_close

pytestmark = pytest.mark.gpu

BS = 16
WIDE = 1 << 16  # blocks of a table: no kernel for short sequences takes it


def _tables(lens, width=None):
    """Consecutive blocks; how many there are."""
    per = [-(-n // BS) for n in lens]
    out = np.full((len(lens), width or max(per)), -1, dtype=np.int32)
    at = 0
    for row, n in zip(out, per):
        row[:n] = np.arange(at, at + n)
        at += n
    return torch.from_numpy(out).to(DEV), at


def _attend(q, k, v, lens, scale):
    """64-bit outputs and what the weights' sizes let them err by: the sums of |weight * value|."""
    q, k, v = q.double(), k.double(), v.double()
    hq, hkv = q.shape[1], k.shape[1]
    out, size, at = [], [], 0
    for b, n in enumerate(lens):
        kk, vv = (t[at * BS: at * BS + n].repeat_interleave(hq // hkv, 1) for t in (k, v))
        w = torch.softmax(torch.einsum("hd,nhd->hn", q[b], kk) * scale, 1)
        out.append(torch.einsum("hn,nhd->hd", w, vv))
        size.append(torch.einsum("hn,nhd->hd", w, vv.abs()))
        at += -(-n // BS)
    return torch.stack(out), torch.stack(size)


WAYS = [("whole", [300, 33], None), ("runs", [1500, 40], None), ("split", [300, 33], WIDE), ("split", [1500, 40], WIDE)]
SHAPES = [(14, 2, 64), (8, 2, 128), (32, 8, 128), (6, 2, 256), (3, 3, 64)]


@pytest.mark.parametrize("what", ["small", "tiny", "large", "mixed", "zeros", "dominant"])
@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("way,lens,width", WAYS)
def test_fp8_pools_whose_values_are_far_from_one(way, lens, width, hq, hkv, d, what):
    """The weights of an fp8 pool meet its scales, which fp16 has no room for: values of 0.001, of 2000, of both, blocks of zeros (whose
    scale is one) beside small ones, and a key whose weight is nearly one and whose values are zero."""
    announce(f"decode values fp8 f16 {way} {hq}/{hkv}x{d} {what}")
    gen = torch.Generator().manual_seed(d + hq)
    tables, blocks = _tables(lens, width)
    k, v = (torch.randn(blocks * BS, hkv, d, generator=gen) for _ in range(2))
    q = torch.randn(len(lens), 1, d, generator=gen) + 0.1 * torch.randn(len(lens), hq, d, generator=gen)
    size = {"small": 0.03, "tiny": 1e-3, "large": 2000.0, "mixed": 1.0, "zeros": 1e-3, "dominant": 0.03}[what]
    v *= size
    if what == "mixed":
        v *= 10.0 ** (torch.arange(blocks) % 7 - 3.0).repeat_interleave(BS)[:, None, None]
    if what == "zeros":
        v[torch.arange(blocks).repeat_interleave(BS) % 3 == 1] = 0
    if what == "dominant":
        at = 0
        for b, n in enumerate(lens):
            k[at * BS + n // 2] = 11.0 * d ** 0.5 * q[b].mean(0) / (q[b].mean(0) ** 2).sum()
            v[at * BS + n // 2] = 0
            at += -(-n // BS)
    q = q.to(torch.float16)
    kb, ks = ops.quantize_kv_e4m3(k.to(torch.float16).to(DEV), BS)
    vb, vs = ops.quantize_kv_e4m3(v.to(torch.bfloat16).to(DEV), BS)
    every = lambda x, s: x.cpu().double() * s.cpu().double().repeat_interleave(BS, 0)[:, :, None]
    want, size = _attend(q, every(kb, ks), every(vb, vs), lens, d ** -0.5)
    qd = q.to(DEV)
    got = ops.decode(qd, kb, vb, tables, torch.tensor(lens, dtype=torch.int32, device=DEV), BS, d ** -0.5, ops.decode_workspace(qd, kb), k_scale=ks, v_scale=vs)
    err = (got.cpu().double() - want).abs()
    # (outputs are rounded to 11 bits, or to a multiple of 2^-24, weights to 11 bits at least)
    room = 2.0 ** -11 * want.abs() + 2.0 ** -25 + 2.0 ** -11 * size
    assert bool((err <= room).all()), (float((err / room).max()), float(err.norm() / want.norm()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", SHAPES + [(4, 4, 32)])
@pytest.mark.parametrize("way,lens,width", WAYS)
def test_infinities_among_the_values(way, lens, width, hq, hkv, d, dtype):
    """An infinite value of a key in sight is an infinite output of its column, not NaN; columns without one are what they are without it."""
    announce(f"decode values inf {way} {hq}/{hkv}x{d} {dtype}")
    gen = torch.Generator().manual_seed(d)
    tables, blocks = _tables(lens, width)
    k, v = (torch.randn(blocks * BS, hkv, d, generator=gen) for _ in range(2))
    q = (0.5 * torch.randn(len(lens), hq, d, generator=gen)).to(dtype).to(DEV)  # (no weight so small that it is zero in 16 bits)
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    bad = v.clone()
    up, down, both, nan = [0, 3], [5], [d - 1], [7]  # columns
    for at in (2, lens[0] // 2, lens[0] - 1):
        bad[at, :, up] = float("inf")
    bad[lens[0] - 2, :, down] = -float("inf")
    bad[1, :, both], bad[lens[0] - 1, :, both] = float("inf"), -float("inf")
    bad[4, :, nan] = float("nan")
    kd = k.to(dtype).to(DEV)
    call = lambda x: ops.decode(q, kd, x.to(dtype).to(DEV), tables, n, BS, d ** -0.5, ops.decode_workspace(q, kd)).cpu()
    clean, got = call(v), call(bad)
    assert torch.equal(got[1], clean[1])
    assert bool((got[0][:, up] == float("inf")).all()) and bool((got[0][:, down] == -float("inf")).all())
    assert bool(got[0][:, both + nan].isnan().all())
    rest = [c for c in range(d) if c not in up + down + both + nan]
    # (both round to 2^-9 or 2^-12, and the weights of one do)
    assert_close(got[0][:, rest], clean[0][:, rest], {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 32), (3, 1, 8), (8, 2, 24)])
def test_weights_of_head_sizes_up_to_32_have_32_bits(hq, hkv, d, dtype):
    """Large values whose weighted sum is nearly zero: what is left are the weights' own errors."""
    announce(f"decode values cancel {hq}/{hkv}x{d} {dtype}")
    gen, n = torch.Generator().manual_seed(d), 33
    tables, blocks = _tables([n])
    k, v = (torch.randn(blocks * BS, hkv, d, generator=gen).to(dtype) for _ in range(2))
    q = torch.randn(1, hkv, d, generator=gen).to(dtype).repeat_interleave(hq // hkv, 1)  # (the heads of a group are alike: one sum to cancel)
    w = torch.softmax(torch.einsum("hd,nhd->hn", q[0, :: hq // hkv].double(), k[:n].double()) * d ** -0.5, 1)
    v *= 1000
    for at in (n - 1, n - 2):  # two keys take what the others leave, the second the rest of the first's rounding
        others = torch.einsum("hn,nhd->hd", w, v[:n].double()) - w[:, at, None] * v[at].double()
        v[at] = (-others / w[:, at, None]).to(dtype)
    want, size = _attend(q, k, v, [n], d ** -0.5)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    got = ops.decode(qd, kd, vd, tables, torch.tensor([n], dtype=torch.int32, device=DEV), BS, d ** -0.5, ops.decode_workspace(qd, kd)).cpu().double()
    err = (got - want).abs()
    # (the outputs' own rounding, and of the sums what one weight can err by: a logit of up to 8 in base 2 by half a unit of 2^-21, its exponential by 2^-23)
    room = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype] * want.abs() + 2.0 ** -21 * size
    assert bool((err <= room).all()), (float((err / room).max()), float((err / size).max()))
