"""Products of experts whose lists fill large tiles partly: every fill of a tile's quarters beside full and empty ones, against the
plain products in 32-bit floats."""

import os
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (a long list beside the short ones: above 160 items an expert large tiles run whatever their number is)
COUNTS = [[0, 1, 63, 64, 65, 127, 128, 129, 1500], [191, 192, 193, 255, 256, 257, 0, 320], [30] * 40 + [6000], [400, 3, 0, 0, 700, 64, 130]]
SIZES = [(256, 2048), (2560, 264)]


def test_which_tiles_run(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text('''
#include "moe_plan.h"
int main() {
    if (moe_shape(4 * 64, 64) != kMoeStream || moe_shape(8 * 64, 64) != kMoeTile64 || moe_shape(9 * 64, 64) != kMoeTile256) return 1;
    if (!moe_stays(161 * 2, 2, 1, 256) || moe_stays(160 * 2, 2, 1, 256)) return 2;       // long lists, whatever their tiles
    if (!moe_stays(9 * 64, 64, 9, 256) || moe_stays(9 * 64, 64, 8, 256)) return 3;       // short ones, more than two tiles each
    if (!moe_stays(25 * 19, 19, 9, 256) || moe_stays(25 * 10, 10, 17, 256) || moe_stays(24 * 19, 19, 9, 256)) return 4;
    const long long of[][2] = {COUNTS};  // the products below: items and experts; tiles over their outputs, of at least one
    for (auto &c : of)
        if (moe_shape(c[0], (int)c[1]) != kMoeTile256 || !moe_stays(c[0], (int)c[1], 1, 256)) return 5;
}
'''.replace("COUNTS", ", ".join(f"{{{sum(c)}, {len(c)}}}" for c in COUNTS)))
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "research_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


@pytest.mark.gpu
@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("width,ff", SIZES)
def test_partly_filled_tiles(counts, width, ff):
    from research_amd import ops
    from tests.gpu_helpers import DEV, announce

    announce(f"expert tiles {counts[:8]} {width} {ff}")
    g = torch.Generator().manual_seed(len(counts))
    experts, rows, pad = len(counts), sum(counts), -(-ff // 64) * 64
    of = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))[torch.randperm(rows, generator=g)]
    logits = torch.full((rows, experts), -9.0).scatter_(1, of[:, None], 9.0)
    c = ops.moe_choose(logits.to(DEV), experts, 1, 1, 1)
    assert c.counts.cpu()[:experts].tolist() == counts
    h = torch.randn(rows, width, generator=g).bfloat16().to(DEV)
    w_in = torch.zeros(experts, 2 * pad, width, dtype=torch.bfloat16)
    w_in[:, :ff], w_in[:, pad: pad + ff] = (torch.randn(experts, ff, width, generator=g) * width ** -0.5 for _ in range(2))
    w_out = torch.zeros(experts, width, pad, dtype=torch.bfloat16)
    w_out[..., :ff] = torch.randn(experts, width, ff, generator=g) * ff ** -0.5
    w_in, w_out = w_in.to(DEV), w_out.to(DEV)
    act = ops.moe_product(h, c, w_in, pad, width, glu=True)
    y = ops.moe_product(act, c, w_out, width, pad, glu=False)
    for e in range(experts):
        at = torch.nonzero(of == e)[:, 0].to(DEV)
        if not len(at):
            continue
        x = h[at].float() @ w_in[e].float().t()
        want = torch.nn.functional.silu(x[:, :pad]) * x[:, pad:]
        # one rounding to bf16, of the result: 2^-9 of it; sums of 2560 products in 32 bits differ by about 1e-6
        assert ((act[at].float() - want).abs() / (want.abs() + 0.01)).max() < 2.0 ** -8, e
        want = act[at].float() @ w_out[e].float().t()
        assert (y[at].float() - want).abs().max() < 2.0 ** -8 * (1 + want.abs().max()), e
