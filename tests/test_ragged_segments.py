"""Segments of prompts of unequal lengths: the rule that chooses them, in a plain C++ build, and launches that it cuts, of every
recurrence, head counts below and above the dies' number, value slices and more sequences than a wave has lanes, against the oracle's
token-by-token recurrence."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_which_delta_rule_walks_go_to_pairs_of_waves(tmp_path):
    """(workgroups, walks a compute unit has, of four waves, prompts, chunks of the longest, rows, pairs) on 256 compute units."""
    batches = [(256, 2, 0, 16, 1, 800, 1), (400, 2, 0, 25, 1, 1300, 0), (288, 2, 0, 18, 2, 2050, 0), (288, 2, 0, 18, 2, 700, 0),
               (384, 2, 0, 3, 1, 90, 0), (288, 2, 0, 9, 7, 1290, 1), (320, 2, 0, 20, 16, 20200, 0), (320, 2, 0, 20, 17, 20800, 1),
               (640, 2, 0, 40, 2, 4600, 0), (640, 2, 0, 40, 8, 20200, 1), (400, 1, 0, 25, 1, 1300, 1), (640, 2, 1, 20, 3, 3700, 0), (800, 2, 0, 50, 8, 25300, 0),
               (256, 2, 1, 8, 1, 400, 0), (257, 2, 1, 8, 4, 2000, 0), (256, 2, 1, 8, 4, 2000, 1), (640, 1, 1, 20, 3, 3700, 1), (640, 1, 1, 20, 1, 900, 1),
               (400, 2, 0, 25, 3, 1 << 40, 0), (400, 2, 0, 25, 3, 0, 1)]
    src = tmp_path / "plan.cpp"
    src.write_text('#include "lightning_plan.h"\nint main() {\n' + "".join(
        f"    if (la_delta_pairs({w}LL, {walks}, {four}, {batch}, {chunks}, {rows}LL, 256) != {want}) return {i + 1};\n"
        for i, (w, walks, four, batch, chunks, rows, want) in enumerate(batches)) + "}\n")
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "research_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def test_segments_follow_the_rows_of_a_batch(tmp_path):
    src = tmp_path / "plan.cpp"
    src.write_text('''
#include "lightning_plan.h"
#include <cstdio>
#include <initializer_list>
int main() {
    for (double together : {0.0, 1.25, 1.6})
        for (long long batch : {1LL, 2LL, 7LL, 40LL, 3000LL})
            for (int per : {1, 5, 16, 64})
                for (int len = 1; len < 40000; len = len * 3 / 2 + 1)
                    for (double part : {0.0, 0.3, 1.0}) {
                        const size_t one = la_workspace_bytes(batch, per, 128, 128, 2) / 2;
                        const int most = la_most_segments(one, len);
                        if (most < 1 || most > kLaMaxSegments || (most > 1 && most * one > kLaMostSegBytes)) return 1;
                        const long long rows = (long long)(batch * len * part) + 1;
                        const int s = la_launch_segments(batch, per, 256, together, len, rows, one, most * one, true);
                        if (s < 1 || s > most || (long long)s * la_segment_rows(len, s) < len) return 2;
                        for (size_t room : {(size_t)0, one, 3 * one + 5}) {  // a workspace too small for all of them
                            const int t = la_launch_segments(batch, per, 256, together, len, rows, one, room, true);
                            if (t < 1 || (t > 1 && t * one > room)) return 3;
                        }
                        // unaligned: refused where few sequences need it, ignored where the batch fills the device
                        const int u = la_launch_segments(batch, per, 256, together, len, rows, one, most * one, false);
                        if (u != (most > 1 && la_segments(batch * per, 256, len) > 1 ? 0 : 1)) return 4;
                        if (la_launch_segments(batch, per, 256, together, len, rows, one, 0, false) != 1) return 5;
                    }
    const size_t big = (size_t)1 << 20;
    if (la_balanced_segments(16, 16, 256, 0.0, 4096, 16 * 4096, 64) != 1) return 6;  // equal and full: no segments
    if (la_balanced_segments(16, 16, 256, 0.0, 4096, 5 * 4096, 64) < 2) return 7;    // a few long ones: segments
    if (la_balanced_segments(1, 16, 256, 0.0, 4096, 4096, la_most_segments(big, 4096)) < 4) return 8;
    if (la_balanced_segments(0, 16, 256, 0.0, 4096, 0, 64) != 1 || la_balanced_segments(4, 16, 256, 0.0, 0, 0, 64) != 1) return 9;
    if (la_most_segments(big * 300, 40000) != 1 || la_most_segments(0, 40000) != 64) return 10;
    if (la_balanced_segments(2, 24, 256, 0.0, 2570, 5123, 5) != 5) return 11;   // as many as fit whatever the lengths
    if (la_balanced_segments(5, 16, 256, 0.0, 2066, 8293, 4) != 4) return 12;   // some last ones more than compute units
    if (la_balanced_segments(1, 16, 256, 0.0, 12000, 12000, 23) != 16) return 13;  // equal segments: one each
    if (la_launch_segments(3, 64, 256, 1.25, 4096, 3 * 4096, big, 64 * big, false, 2) != 0) return 15;  // refused: two workgroups a unit
    if (la_launch_segments(3, 64, 256, 1.25, 4096, 3 * 4096, big, 64 * big, false) != 1) return 16;     // ... one: taken for none
    for (int segments = 1; segments < 9; ++segments)  // before a portion's last one
        for (int rows : {-3, 0, 1, 511, 512, 513, 1024, 1025, 2560, 9999}) {
            const int full = la_full_segments(rows, segments, 512);
            if (full < 0 || full >= segments || (rows > 0 && full * 512 >= rows) || (full < segments - 1 && (full + 1) * 512 < rows)) return 14;
        }
    std::puts("ok");
}
''')
    exe = tmp_path / "plan"
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "research_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], stdout=subprocess.PIPE).returncode == 0


@pytest.mark.parametrize("kind", ["lightning", "gated_linear", "channel_linear"])
def test_a_batch_in_one_piece_asks_for_no_workspace(kind):
    from research_amd import ops

    need = getattr(ops, kind + "_workspace_bytes")
    assert need(32, 16, 128, 128, 4096, rows=32 * 4096) == 0              # equal portions that fill the device
    ragged, most = need(32, 16, 128, 128, 4096, rows=9 * 4096), need(32, 16, 128, 128, 4096)
    assert 0 < ragged <= most <= 256 << 20                                # a few long ones among them
    assert need(1, 16, 128, 128, 4096) == need(1, 16, 128, 128, 4096, rows=4096) >= 4 * 16 * 128 * 128 * 4
    for rows in range(2000, 16000, 700):                                  # (no launch takes more than what any may)
        assert need(8, 16, 128, 128, 2000, rows=rows) <= need(8, 16, 128, 128, 2000)
    assert need(64, 16, 128, 128, 900) == 0                               # too short to be cut


@pytest.mark.gpu
@pytest.mark.parametrize("kind,heads,dim,vdim", [("lightning", 8, 128, 128), ("lightning", 4, 64, 64), ("mlstm", 4, 256, 512), ("mlstm", 4, 64, 128),
                                                 ("ssd", 16, 128, 64), ("ssd", 2, 64, 128), ("channel", 8, 128, 128), ("channel", 3, 96, 80)])
@pytest.mark.parametrize("lens", [[257], [128, 700, 1, 65], [1500], [6000, 130], [0, 640, 513]])
def test_few_prompts_in_short_segments(kind, heads, dim, vdim, lens):
    """A workgroup for each of more segments than a prompt has eights of chunks, the scan over more of them than it loads at once: as in one piece."""
    import torch

    from research_amd import ops
    from tests.gpu_helpers import DEV, announce

    announce(f"short segments {kind} {heads}x{dim}x{vdim} {lens}")
    gen, batch, before = torch.Generator().manual_seed(dim + len(lens)), len(lens), 70
    parts = {"lightning": (heads * dim, heads * dim, heads * vdim), "channel": (heads * dim, heads * dim, heads * vdim)}.get(
        kind, (heads * dim, heads * dim, heads * vdim, 2 * heads))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    pad = lambda x: -(-x // 16) * 16
    need = {"lightning": ops.lightning_workspace_bytes, "channel": ops.channel_linear_workspace_bytes}.get(kind, ops.gated_linear_workspace_bytes)
    room = need(batch, heads, dim, vdim, max(lens), rows=sum(lens))
    if max(lens) >= 1500:
        assert room >= 8 * heads * pad(dim) * pad(vdim) * 4
    shape = (batch, heads, ops.gated_linear_state_floats(kind, dim, vdim)) if kind in ("ssd", "mlstm") else (batch, heads, pad(dim), pad(vdim))
    constant = lambda a, b, m=heads: (a + (b - a) * torch.rand(m, generator=gen)).to(DEV)
    decay = torch.tensor([1.0 - 0.5 ** (3 + i) for i in range(heads)], dtype=torch.float64)
    powers = (decay[:, None] ** torch.arange(65, dtype=torch.float64)).float().to(DEV)
    gates = (constant(-5, -3), constant(1, 16), constant(-1, 1)) if kind == "ssd" else (constant(-1, 1), constant(3, 6), None)
    f_bias, lower = constant(1, 4, heads * dim), constant(0, 0.9, heads * dim)

    def run(u, behind, new, state, ws):
        p = ops.Portions(i32([behind + x for x in new]), i32(list(range(batch))), i32(new), i32([sum(new[:i]) for i in range(batch)]), None, max(new))
        out = torch.full((sum(new), heads * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
        q, k, v = u.split(parts, 1)[:3]
        if kind == "lightning":
            ops.lightning(u, p, state, powers, heads, dim, vdim, out, workspace=ws)
        elif kind == "channel":
            ops.channel_linear(q, k, v, f_bias, lower, p, state, heads, dim, vdim, out, q_act="silu", workspace=ws)
        else:
            a, b = u[:, -2 * heads: -heads], u[:, -heads:]
            ops.gated_linear(kind, q, k, v, (a, None if kind == "ssd" else b), gates, p, state, heads, dim, vdim, out, cap=15.0, q_scale=dim ** -0.5,
                             den_eps=1e-6, workspace=ws)
        return out

    rows = lambda m: torch.randn(m, sum(parts), generator=gen).to(torch.bfloat16).to(DEV)
    first = torch.zeros(shape, device=DEV)
    run(rows(before * batch), 0, [before] * batch, first, None)
    u, results = rows(sum(lens)), []
    for ws in (None, torch.full((max(room, 16),), 0x7f, dtype=torch.uint8, device=DEV)):
        state = first.clone()
        results.append((run(u, before, lens, state, ws).double(), state.double()))
    (out, state), (want, want_state) = results[1], results[0]
    assert torch.isfinite(out).all() and torch.isfinite(state).all()
    # (both round an output of 32-bit sums to 16 bits: 2^-9 of it each; states carry two 16-bit terms of every factor, 2^-16, over sums of many)
    assert float((out - want).norm() / want.norm()) < 2.0 ** -8
    assert float((state - want_state).norm() / want_state.norm()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dim,vdim,longest", [(32, 64, 64, 2500), (32, 64, 128, 2500), (16, 128, 128, 2500), (16, 128, 128, 8000)])
def test_a_batch_of_unequal_prompts_in_segments(heads, dim, vdim, longest):
    import torch

    from tests.gpu_helpers import announce
    from tests.test_gpu_lightning import Case

    announce(f"ragged segments {heads}x{dim}x{vdim} {longest}")
    decay = [1.0 - 0.5 ** (1 + i * 12 / heads) for i in range(heads)]
    # one sequence of many segments, some that end inside the first, on and beside a segment's edge
    # (8000: more of them than compute units, two of which then share one)
    lens = [longest, 1, 64, 511, 512, 513, longest // 3, 700, 30, longest * 3 // 5]
    case = Case(lens, heads, dim, vdim, decay, torch.bfloat16, seed=5)
    slots = [(3 * b + 1) % len(lens) for b in range(len(lens))]
    head = [(b, 0, (n + 1) // 2) for b, n in enumerate(lens)]
    tail = [(b, (n + 1) // 2, n // 2) for b, n in enumerate(lens) if n > 1]
    for picks in (head, tail):  # (the second starts from the states that the first left)
        for (b, lo, _), got in zip(picks, case.run(picks, slots)):
            case.check(b, lo, got)
    for b, n in enumerate(lens):
        case.check_state(b, slots[b])


RAGGED = [("mlstm", 16, 64, 192), ("mlstm", 24, 64, 40), ("ssd", 16, 128, 128), ("ssd", 24, 64, 64), ("channel", 16, 64, 64), ("channel", 8, 64, 200), ("channel", 4, 128, 128),
          ("lightning", 24, 64, 64), ("lightning", 3, 128, 256)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,heads,dim,vdim", RAGGED)
def test_every_recurrence_over_unequal_prompts(kind, heads, dim, vdim):
    import torch

    from tests.gpu_helpers import announce
    from tests.test_gpu_lightning import Case as Lightning
    from tests.test_gpu_loluzen_ops import Channels
    from tests.test_gpu_tevirax_ops import Case as Gated

    announce(f"ragged segments {kind} {heads}x{dim}x{vdim}")
    lens, bf = [2500, 40, 513, 1024, 1, 1025, 700, 100], torch.bfloat16
    slots = [(3 * b + 1) % len(lens) for b in range(len(lens))]
    whole = [(b, 0, n) for b, n in enumerate(lens)]
    cuts = [(b, 0, (n + 1) // 2) for b, n in enumerate(lens)], [(b, (n + 1) // 2, n // 2) for b, n in enumerate(lens) if n > 1]
    if kind == "channel":  # (its rows are checked where they are run)
        case = Channels(lens, heads, dim, vdim, bf, seed=6)
        for picks in (whole, *cuts):
            case.run(picks, slots)
        case.check_states(slots)
        return
    case = Lightning(lens, heads, dim, vdim, [1.0 - 0.5 ** (1 + i * 12 / heads) for i in range(heads)], bf, seed=6) if kind == "lightning" else \
        Gated(kind, lens, heads, dim, vdim, bf, 8 if kind == "ssd" else None, seed=6, remember=4.5)
    for picks in (whole, *cuts):
        for (b, lo, _), got in zip(picks, case.run(picks, slots)):
            case.check(b, lo, got)
    for b in range(len(lens)):
        case.check_state(b, slots[b])


@pytest.mark.gpu
def test_more_unequal_prompts_than_a_wave_has_lanes():
    import torch

    from tests.gpu_helpers import announce
    from tests.test_gpu_lightning import Case

    announce("ragged segments of 150 sequences")
    lens = [1 + 37 * b % 90 for b in range(150)]
    lens[3], lens[70], lens[149] = 1100, 1600, 1300
    case = Case(lens, 2, 32, 32, [0.99, 0.9], torch.bfloat16, seed=7)
    slots = list(range(150))
    for (b, lo, _), got in zip(((b, 0, n) for b, n in enumerate(lens)), case.run([(b, 0, n) for b, n in enumerate(lens)], slots)):
        case.check(b, lo, got)
    for b in (0, 3, 64, 70, 148, 149):
        case.check_state(b, b)
