"""Attention with score terms over prompts whose workgroups start in an order of their own: more of them than the device holds
at once, of unequal sequences, over blocks of any size, against the plain product in 32-bit floats."""

import numpy as np
import pytest
import torch

from research_amd import ops
from tests.gpu_helpers import DEV, announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block,window,cap", [(16, 0, 0.0), (1, 70, 8.0), (24, 300, 0.0), (48, 0, 20.0), (100, 512, 20.0)])
@pytest.mark.parametrize("lens,before", [([1500, 1, 40, 700, 33, 64], [0, 9, 0, 0, 100, 64]), ([31], [0]), ([1100], [37])])
def test_prompts_in_their_order_of_starting(lens, before, block, window, cap):
    heads, kv, dim, most = 32, 8, 64, 200
    announce(f"scored order {lens} {block} {window} {cap}")
    g = torch.Generator().manual_seed(block)
    ctx = [n + m for n, m in zip(lens, before)]
    need = [-(-n // block) for n in ctx]
    blocks = np.random.default_rng(block).permutation(sum(need) + 3)
    tables = torch.full((len(lens), max(need) + 1), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = torch.from_numpy(blocks[at: at + n].astype(np.int32))
        at += n
    k, v = (torch.randn(len(blocks) * block, kv, dim, generator=g).bfloat16().to(DEV) for _ in range(2))
    q = torch.randn(sum(lens), heads, dim, generator=g).bfloat16().to(DEV)
    bias, sink = torch.randn(heads, most, generator=g).to(DEV), torch.randn(heads, generator=g).to(DEV)
    starts = np.cumsum([0] + lens[:-1])
    i32 = lambda x: torch.tensor([int(n) for n in x], dtype=torch.int32, device=DEV)
    por = ops.Portions(i32(ctx), i32(range(len(lens))), i32(lens), i32(starts), None, max(lens))
    out = torch.full((sum(lens), heads, dim), float("nan"), dtype=torch.bfloat16, device=DEV)
    scale = 2.0 * dim ** -0.5
    ops.scored_attention((q,), k, v, dim, por, tables.to(DEV), block, scale, window, out, softcap=cap, bias=bias, sink=sink)
    for b, n in enumerate(lens):
        keys = torch.arange(ctx[b], device=DEV)
        slots = tables[b].to(DEV).long()[keys // block] * block + keys % block
        rows = keys[before[b]:]
        gap = rows[:, None] - keys[None]
        seen = (gap >= 0) & ((gap < window) if window else True)
        for h in range(heads):
            s = scale * q[starts[b]: starts[b] + n, h].float() @ k[slots, h // (heads // kv)].float().t()
            s = (cap * torch.tanh(s / cap) if cap else s) + bias[h][gap.clamp(0, most - 1)]
            s = torch.cat([s.masked_fill(~seen, float("-inf")), sink[h].expand(n, 1)], 1).softmax(1)[:, :-1]
            want = s @ v[slots, h // (heads // kv)].float()
            got = out[starts[b]: starts[b] + n, h].float()
            # weights and results are rounded to bf16: 2^-9 each, of values of at most 5
            assert (got - want).abs().max() < 2e-2, (b, h)
