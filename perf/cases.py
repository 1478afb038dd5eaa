"""What the speed of this framework is measured on: attention over paged pools, recurrences and experts as a serving engine calls
them, through the tensor-level entry points of ``research_amd.ops``.

A case is a dictionary of sizes.  ``path`` says what is called:

``decode``    one new token for each of ``batch`` sequences of ragged lengths (``ops.decode``)
``chunk``     prompts, or parts of prompts, behind a prefix that the sequences share: their keys and values are appended, then
              their rows attend (``ops.kv_scatter``, ``ops.prefill_paged``)
``lightning`` / ``mlstm`` / ``ssd`` / ``delta`` / ``channel``
              a linear recurrence over whole prompts, then over ``steps`` further tokens of every sequence, one at a time, with
              the state carried (``ops.lightning``, ``ops.gated_linear``, ``ops.delta_rule``, ``ops.channel_linear``)
``scored``    attention with a cap on the scores, distance biases and sinks (``ops.scored_attention``); ``token``: one new
              token per sequence, else whole prompts
``talking``   attention whose heads' weights are mixed (``ops.talking_attention``); ``token`` as above
``experts``   router, choice, the two products of the chosen experts, and the residual sum and norm behind them
              (``ops.narrow_linear``, ``ops.moe_choose``, ``ops.moe_product``, ``ops.residual_norm``)

Lengths are spread by ``spread`` between ``low`` and ``high`` (over their logarithm) and belong to the case; values come from the
seed.  Head counts and sizes are those of the shapes in ``bench.py`` and of its engine workload, and generic ones.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from research_amd import ops

BLOCK = 16
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.bfloat16}
SIZES = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1}
RECURRENT = ("lightning", "mlstm", "ssd", "delta", "channel")
GATE_CAP, DEN_EPS = 15.0, 1e-6
SOFTCAP, DISTANCES = 30.0, 129


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # A handful of rollouts of a small model (the engine workload's heads): launches and waits count, not bytes.
        dict(name="decode_few", path="decode", batch=4, low=1, high=600, spread=11, heads=14, kv_heads=2, dim=64, dtype="bf16", window=0),
        # A full batch in the middle of generation: lengths from short to very long, as rollouts have them.
        dict(name="decode_full", path="decode", batch=256, low=64, high=32768, spread=12, heads=32, kv_heads=8, dim=128, dtype="bf16", window=0),
        # Few sequences with long contexts over an fp8 pool.
        dict(name="decode_fp8_long", path="decode", batch=8, low=65536, high=131072, spread=13, heads=32, kv_heads=8, dim=128, dtype="fp8", window=0),
        # Prompts that share a system prompt: their own parts, of ragged lengths, behind it.
        dict(name="chunk_shared", path="chunk", batch=32, prefix=2048, low=97, high=256, spread=14, heads=32, kv_heads=8, dim=128, dtype="bf16"),
        # A step of admitted prompts in a layer of each recurrence, and the tokens after it.
        dict(name="lightning_prompts", path="lightning", batch=8, low=700, high=4000, spread=15, heads=16, groups=16, dim=128, vdim=128, steps=2),
        # One long document: nothing but its segments can run side by side.
        dict(name="mlstm_long", path="mlstm", batch=1, low=15999, high=15999, spread=16, heads=4, groups=4, dim=256, vdim=512, steps=1),
        # Many short prompts, then their generation: states are read and written once per token.
        dict(name="ssd_short", path="ssd", batch=128, low=16, high=130, spread=17, heads=64, groups=8, dim=128, vdim=64, steps=8),
        dict(name="delta_prompts", path="delta", batch=8, low=700, high=4000, spread=18, heads=16, groups=8, dim=128, vdim=128, steps=2),
        dict(name="channel_prompts", path="channel", batch=8, low=700, high=4000, spread=19, heads=32, groups=32, dim=128, vdim=128, steps=2),
        # Prompts in an attention layer with score terms and a window.
        dict(name="scored_prompts", path="scored", batch=8, low=700, high=4000, spread=20, heads=16, kv_heads=4, dim=128, vdim=128, window=1024,
             cap=True, token=False),
        # Prompts in an attention layer with mixed heads.
        dict(name="talking_prompts", path="talking", batch=8, low=700, high=4000, spread=21, heads=16, kv_heads=4, dim=128, vdim=128, token=False),
        # The experts of a wide layer over a prefill step.
        dict(name="experts_prompts", path="experts", rows=6001, width=4096, inner=1408, experts=64, top=8),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "chunk", "lightning", "mlstm", "ssd", "delta", "channel", "scored", "talking", "experts"])
    case = dict(path=path, spread=rng.randrange(1, 1 << 20))
    if path == "experts":
        width, inner, top = rng.choice([(2048, 768, 6), (4096, 1408, 8), (1024, 512, 4)])
        return dict(path=path, rows=_log(rng, 1, 6000), width=width, inner=inner, experts=rng.choice([16, 64]), top=top)

    def lengths(batch, tokens, most):
        """Between two lengths such that the batch has at most about `tokens` tokens."""
        high = _log(rng, 16, max(17, min(most, tokens // batch)))
        case.update(batch=batch, low=_log(rng, 1 if high < 64 else high // 8, high), high=high)

    if path == "decode":
        case["dtype"] = rng.choice(["bf16", "bf16", "f16", "fp8", "f32"])
        case["heads"], case["kv_heads"] = rng.choice([(32, 8), (16, 8), (14, 2), (8, 2), (16, 2)])
        case["dim"] = rng.choice([64, 128, 128, 256] + ([] if case["dtype"] == "fp8" else [72]))
        per = {64: 1 << 19, 72: 1 << 19, 128: 1 << 19, 256: 1 << 18}[case["dim"]] // (2 if case["dtype"] == "f32" else 1)
        lengths(_log(rng, 1, 256), per, 1 << 17)
        case["window"] = rng.choice([0, 0, 0, 1024])
        return case
    if path == "chunk":
        case["dtype"] = rng.choice(["bf16", "bf16", "f16"])
        case["heads"], case["kv_heads"] = rng.choice([(32, 8), (16, 8), (14, 2), (8, 2)])
        case["dim"] = rng.choice([64, 96, 128, 128, 256])
        case["prefix"] = rng.choice([0, BLOCK * _log(rng, 1, 512)])
        most = int(3e11 / (4.0 * case["heads"] * case["dim"] * (case["prefix"] + 1024)))
        lengths(_log(rng, 1, 64), min(16384, most), 2048)
        return case
    if path in ("scored", "talking"):
        case["heads"], case["kv_heads"] = rng.choice([(16, 4), (32, 8), (8, 2)])
        case["dim"], case["vdim"] = rng.choice([(128, 128), (128, 128), (64, 64), (96, 64)])
        case["token"] = rng.random() < 0.35
        if path == "scored":
            case["window"], case["cap"] = rng.choice([0, 512, 1024]), rng.random() < 0.7
        lengths(_log(rng, 1, 128 if case["token"] else 32), 1 << 17 if case["token"] else 1 << 13, 1 << 13 if case["token"] else 4000)
        return case
    if path == "mlstm":
        case["heads"], case["dim"], case["vdim"] = rng.choice([(4, 256, 512), (8, 128, 256), (4, 64, 128)])
        case["groups"] = case["heads"]
    elif path == "ssd":
        case["heads"], case["groups"] = rng.choice([(64, 8), (32, 8), (16, 1)])
        case["dim"], case["vdim"] = rng.choice([(128, 64), (64, 64), (128, 128)])
    else:
        case["heads"] = rng.choice([8, 16, 32])
        case["groups"] = case["heads"] // (rng.choice([1, 2]) if path == "delta" else 1)
        case["dim"], case["vdim"] = rng.choice([(128, 128), (128, 128), (128, 64), (64, 64), (96, 80)])
    lengths(_log(rng, 1, 64), 16000, 16000)
    case["steps"] = rng.randrange(0, 5)
    return case


# ------------------------------------------------------------------ lengths, values, tables


def _lens(case):
    """The sequences' lengths: what the case is, whatever the seed."""
    rng = np.random.default_rng(case["spread"])
    if case["path"] == "decode" and case["low"] == 64 and case["high"] == 32768:  # rollouts: around 2048, some very long
        return np.clip(np.rint(np.exp(rng.normal(math.log(2048.0), 1.0, case["batch"]))), 64, 32768).astype(np.int64)
    low, high = math.log(case["low"]), math.log(case["high"])
    return np.clip(np.rint(np.exp(rng.uniform(low, high, case["batch"]))), case["low"], case["high"]).astype(np.int64)


class _Values:
    """Random values on the device, the same for the same seed and order of calls."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).mul_(scale).to(dtype)

    def uniform(self, low, high, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda") * (high - low) + low


def _i32(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.int32).cuda()


def _tables(lens, seed):
    """Block tables over a pool whose blocks are in no order; rows padded with -1."""
    per = -(-lens // BLOCK)
    perm = np.random.default_rng(int(seed)).permutation(int(per.sum()))
    out = np.full((len(lens), int(per.max())), -1, dtype=np.int32)
    at = 0
    for b, n in enumerate(per):
        out[b, :n] = perm[at: at + n]
        at += n
    return out, at


def _portions(lens, slots):
    """Whole prompts, one after the other."""
    starts = np.cumsum(lens) - lens
    tiles = [(b, r) for b, n in enumerate(lens) for r in range(0, int(n), ops.QKV_TILE_ROWS)]
    return ops.Portions(_i32(lens), slots, _i32(lens), _i32(starts), _i32(np.asarray(tiles)), int(lens.max()))


def _fp8_pool(pool):
    """Bytes and scales per (block, head): the largest value of a tile becomes 448."""
    slots, kv, d = pool.shape
    tiles = pool.float().view(slots // BLOCK, BLOCK, kv, d)
    top = tiles.abs().amax((1, 3))
    scale = torch.where(top > 0, top / 448.0, torch.ones_like(top))
    return (tiles / scale[:, None, :, None]).to(torch.float8_e4m3fn).view(slots, kv, d), scale


def _pad16(n):
    return -(-n // 16) * 16


# ------------------------------------------------------------------ prepare


def _inputs(case, seed):
    """The values of a case by name, from the seed alone."""
    val, path = _Values(seed), case["path"]
    bf = torch.bfloat16
    if path == "experts":
        rows, width, inner, e = case["rows"], case["width"], case["inner"], case["experts"]
        return dict(x=val.normal(rows, width), h=val.normal(rows, width, dtype=bf), router=val.normal(e + 1, width, dtype=bf, scale=width ** -0.5),
                    w_in=val.normal(e, 2 * inner, width, dtype=bf, scale=width ** -0.5), w_out=val.normal(e, width, inner, dtype=bf, scale=inner ** -0.5),
                    shared=val.normal(rows, width, dtype=bf, scale=0.5), y_weight=val.uniform(0.5, 1.5, width))
    lens = _lens(case)
    if path in RECURRENT:
        heads, groups, dim, vdim = case["heads"], case["groups"], case["dim"], case["vdim"]
        rows = int(lens.sum()) + case["steps"] * len(lens)
        parts = {"q": groups * dim, "k": groups * dim, "v": heads * vdim, "a": heads, "b": heads}
        if path == "lightning":
            del parts["a"], parts["b"]
        if path == "channel":
            del parts["a"], parts["b"]
            parts = {"q": heads * dim, "f": heads * dim, "v": heads * vdim}
        wide = sum(parts.values())
        u = val.normal(rows, -(-wide // 8) * 8, dtype=bf)
        d = dict(u=u, lens=lens, sizes=tuple(parts.values()))
        if path == "lightning":
            decay = torch.tensor([1.0 - 2.0 ** -(2 + 6 * h / heads) for h in range(heads)], dtype=torch.float64)
            d["powers"] = (decay[:, None] ** torch.arange(65, dtype=torch.float64)).float().cuda()
        elif path == "mlstm":
            d.update(i_bias=val.normal(heads), f_bias=val.uniform(3.0, 6.0, heads))
        elif path == "ssd":
            d.update(dt_bias=val.uniform(-5.0, -3.0, heads), rate=val.uniform(1.0, 16.0, heads), skip=val.normal(heads))
        elif path == "delta":
            d.update(dt_bias=val.uniform(-5.0, -3.0, heads), rate=val.uniform(1.0, 16.0, heads))
        else:
            u[:, parts["q"]: parts["q"] + parts["f"]] += 2.5
            d.update(f_bias=val.normal(heads * dim), lower=val.uniform(0.0, 0.9, heads * dim))
        return d
    dtype, heads, kv, dim = DTYPES[case.get("dtype", "bf16")], case["heads"], case["kv_heads"], case["dim"]
    if path == "chunk":
        lens = lens + case["prefix"]
        shared = case["prefix"] // BLOCK
        tables, own = _tables(lens - case["prefix"], seed)
        if shared:
            tables = np.concatenate([np.broadcast_to(own + np.arange(shared, dtype=np.int32), (len(lens), shared)), tables], 1)
        blocks = own + shared
    else:
        tables, blocks = _tables(lens, seed)
    vdim = case.get("vdim", dim)
    pools = [val.normal(blocks * BLOCK, kv, n, dtype=dtype) for n in (dim, dim if path in ("decode", "chunk") else vdim)]
    d = dict(lens=lens, tables=np.ascontiguousarray(tables), k_pool=pools[0], v_pool=pools[1])
    one = path == "decode" or case.get("token", False)
    new = np.ones(len(lens), dtype=np.int64) if one else lens - case.get("prefix", 0)
    d["new"] = new
    d["q"] = val.normal(int(new.sum()), heads, dim, dtype=dtype)
    if case.get("dtype") == "fp8":
        d["k_pool"], d["k_scale"] = _fp8_pool(pools[0])
        d["v_pool"], d["v_scale"] = _fp8_pool(pools[1])
    if path == "chunk":
        pos = np.concatenate([np.arange(n - m, n) for n, m in zip(lens, new)])
        seq = np.repeat(np.arange(len(lens)), new)
        slots = tables[seq, pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK
        d.update(slots=torch.from_numpy(slots).cuda(), k_new=val.normal(len(slots), kv, dim, dtype=dtype), v_new=val.normal(len(slots), kv, dim, dtype=dtype))
    if path == "scored":
        d.update(bias=val.normal(heads, DISTANCES), sink=val.normal(heads))
    if path == "talking":
        d.update(talk=torch.eye(heads, device="cuda") + val.normal(heads, heads, scale=0.2), size=val.uniform(0.05, 1.05, heads), rate=val.uniform(0.05, 0.55, heads))
    return d


def _bytes(need):
    return torch.empty(need, dtype=torch.uint8, device="cuda") if need else None


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], path = case, case["path"]
    if path == "experts":
        return s
    lens, batch = s["lens"], len(s["lens"])
    if path in RECURRENT:
        heads, dim, vdim, rows = case["heads"], case["dim"], case["vdim"], int(lens.sum())
        slots = _i32(np.random.default_rng(int(seed)).permutation(batch))
        s["portions"] = _portions(lens, slots)
        s["tokens"] = [ops.Portions(_i32(lens + t + 1), slots) for t in range(case["steps"])]
        shape = (batch, heads, _pad16(dim), _pad16(vdim))
        if path in ("mlstm", "ssd"):
            shape = (batch, heads, ops.gated_linear_state_floats(path, dim, vdim))
        s["state"] = torch.zeros(shape, device="cuda")
        need = {"lightning": ops.lightning_workspace_bytes, "delta": ops.delta_workspace_bytes, "channel": ops.channel_linear_workspace_bytes}
        s["workspace"] = _bytes(need.get(path, ops.gated_linear_workspace_bytes)(batch, heads, dim, vdim, int(lens.max())))
        s["out"] = torch.empty(s["u"].shape[0], heads * vdim, dtype=s["u"].dtype, device="cuda")
        s["cuts"] = [(0, rows)] + [(rows + t * batch, rows + (t + 1) * batch) for t in range(case["steps"])]
        return s
    s["bt"], s["ctx"] = _i32(s["tables"]), _i32(lens)
    if path == "decode":
        s["workspace"] = ops.decode_workspace(s["q"], s["k_pool"])
    elif path == "chunk":
        new = s["new"]
        s["q_lens"], s["q_starts"] = _i32(new), _i32(np.cumsum(new) - new)
        s["workspace"] = _bytes(ops.prefill_workspace_bytes(s["q"], s["bt"], int(new.max()), BLOCK, case["kv_heads"]))
    else:
        slots = _i32(np.arange(batch))
        s["portions"] = ops.Portions(s["ctx"], slots) if case["token"] else _portions(lens, slots)
        heads, kv, keys = case["heads"], case["kv_heads"], s["bt"].shape[1] * BLOCK
        if path == "scored":
            need = ops.scored_workspace_bytes(batch, heads, kv, case["dim"], case["vdim"], False, keys, case["window"]) if case["token"] else 0
        else:
            need = ops.talking_workspace_bytes(s["q"].shape[0], s["portions"], heads, kv, case["vdim"], keys)
        s["workspace"] = _bytes(need)
        s["out"] = torch.empty(s["q"].shape[0], heads, case["vdim"], dtype=s["q"].dtype, device="cuda")
    return s


# ------------------------------------------------------------------ run


def _recurrence(s, case, cut, portions, workspace):
    rows = slice(*cut)
    u, out = s["u"][rows], s["out"][rows]
    sizes = (case["heads"], case["dim"], case["vdim"])
    if case["path"] == "lightning":
        ops.lightning(u, portions, s["state"], s["powers"], *sizes, out, workspace=workspace)
        return
    parts = u[:, : sum(s["sizes"])].split(s["sizes"], 1)
    per = case["heads"] // case["groups"]
    if case["path"] == "channel":
        ops.channel_linear(*parts, s["f_bias"], s["lower"], portions, s["state"], *sizes, out, q_act="silu", workspace=workspace)
        return
    q, k, v, a, b = parts
    if case["path"] == "mlstm":
        ops.gated_linear("mlstm", q, k, v, (a, b), (s["i_bias"], s["f_bias"], None), portions, s["state"], *sizes, out, cap=GATE_CAP,
                         q_scale=case["dim"] ** -0.5, den_eps=DEN_EPS, workspace=workspace)
    elif case["path"] == "ssd":
        ops.gated_linear("ssd", q, k, v, (a, None), (s["dt_bias"], s["rate"], s["skip"]), portions, s["state"], *sizes, out,
                         heads_per_group=per, workspace=workspace)
    else:
        ops.delta_rule(q, k, v, a, b, s["dt_bias"], s["rate"], portions, s["state"], *sizes, case["dim"] ** -0.5, out, heads_per_group=per,
                       workspace=workspace)


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "decode":
        return ops.decode(s["q"], s["k_pool"], s["v_pool"], s["bt"], s["ctx"], BLOCK, case["dim"] ** -0.5, s["workspace"],
                          k_scale=s.get("k_scale"), v_scale=s.get("v_scale"), window=case["window"])
    if path == "chunk":
        ops.kv_scatter(s["k_pool"], s["v_pool"], s["k_new"], s["v_new"], s["slots"])
        out = ops.prefill_paged(s["q"], s["k_pool"], s["v_pool"], s["bt"], s["ctx"], s["q_lens"], s["q_starts"], int(s["new"].max()), BLOCK,
                                case["dim"] ** -0.5, workspace=s["workspace"])
        return out, s["k_pool"], s["v_pool"]
    if path in RECURRENT:
        _recurrence(s, case, s["cuts"][0], s["portions"], s["workspace"])
        for cut, portions in zip(s["cuts"][1:], s["tokens"]):
            _recurrence(s, case, cut, portions, None)
        return s["out"], s["state"]
    if path == "scored":
        return ops.scored_attention((s["q"],), s["k_pool"], s["v_pool"], case["vdim"], s["portions"], s["bt"], BLOCK, case["dim"] ** -0.5,
                                    case["window"], s["out"], softcap=SOFTCAP if case["cap"] else 0.0, bias=s["bias"], sink=s["sink"],
                                    workspace=s["workspace"])
    if path == "talking":
        return ops.talking_attention(s["q"], s["k_pool"], s["v_pool"], case["vdim"], s["portions"], s["bt"], BLOCK, case["dim"] ** -0.5, s["talk"],
                                     s["out"], s["size"], s["rate"], workspace=s["workspace"])
    rows, width, inner, e, top = (case[n] for n in ("rows", "width", "inner", "experts", "top"))
    choice = ops.moe_choose(ops.narrow_linear(s["h"], s["router"]), e, top, 8, 4, "gated")
    act = ops.moe_product(s["h"], choice, s["w_in"], inner, width, glu=True)
    y = ops.moe_product(act, choice, s["w_out"], width, inner, glu=False)
    x = s["x"].clone()  # (the residual is updated in place; the next pass starts from the same one)
    h = ops.residual_norm(x, torch.bfloat16, y=y, mix=choice.weights, y_extra=s["shared"], y_weight=s["y_weight"], y_eps=1e-6)
    return x, h


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    path = case["path"]
    if path == "experts":
        rows, width, inner, e, top = (case[n] for n in ("rows", "width", "inner", "experts", "top"))
        used = e * (1.0 - (1.0 - top / e) ** rows)  # experts that some row chooses
        return dict(bytes=rows * width * (4 + 4 + 2 + 2 + 2.0) + used * 3.0 * inner * width * 2 + (e + 1) * width * 2.0,
                    flops=6.0 * rows * top * inner * width + 2.0 * rows * width * (e + 1))
    lens = _lens(case).astype(np.float64)
    batch, tokens = len(lens), float(lens.sum())
    if path in RECURRENT:
        heads, groups, dim, vdim, steps = (case[n] for n in ("heads", "groups", "dim", "vdim", "steps"))
        gates = {"lightning": 0, "channel": 0, "ssd": heads}.get(path, 2 * heads)
        rows = tokens + steps * batch
        state = batch * heads * _pad16(dim) * _pad16(vdim) * 4.0
        # (a whole prompt leaves a state, a further token reads one and writes one; per row and head the products with the state, and
        # of a chunk of 64 rows the scores and their products with the values, half of them under the causal mask)
        return dict(bytes=rows * 2.0 * (2 * groups * dim + 2 * heads * vdim + gates) + state * (1 + 2 * steps),
                    flops=rows * heads * ((6.0 if path == "delta" else 4.0) * dim * vdim) + tokens * heads * 64.0 * (dim + vdim) * (2 if path == "delta" else 1))
    heads, kv, dim = case["heads"], case["kv_heads"], case["dim"]
    vdim, window, size = case.get("vdim", dim), case.get("window", 0), SIZES[case.get("dtype", "bf16")]
    if path == "decode" or case.get("token"):
        seen = float(np.minimum(lens, window).sum()) if window else tokens
        io = 4 if case.get("dtype") == "f32" else 2
        scales = 2 * seen / BLOCK * kv * 4.0 if case.get("dtype") == "fp8" else 0.0
        mix = 2.0 * heads * heads * seen if path == "talking" else 0.0
        return dict(bytes=seen * kv * (dim + vdim) * size + batch * heads * (dim + vdim) * io + seen / BLOCK * 4 + batch * 4 + scales,
                    flops=2.0 * heads * (dim + vdim) * seen + mix)
    prefix = case.get("prefix", 0)
    pairs = tokens * prefix + float((lens * (lens + 1) / 2).sum())
    if window:
        full = np.maximum(lens - window, 0)
        pairs = float((full * window + (lens - full) * (lens - full + 1) / 2).sum())
    appended = tokens * kv * 2 * dim * size * 2 if path == "chunk" else 0.0
    return dict(bytes=(tokens + prefix) * kv * (dim + vdim) * size + tokens * heads * (dim + vdim) * size + appended,
                flops=heads * pairs * (2.0 * (dim + vdim) + (2.0 * heads if path == "talking" else 0.0)))


def tolerance(case):
    # About four times what the path is off the same result in 64 bits (the outputs' own rounding to 16 bits is 1.7e-3 of it).
    if case["path"] == "decode":
        return {"f32": dict(rel=4e-6), "bf16": dict(rel=1.2e-2), "f16": dict(rel=2e-3), "fp8": dict(rel=1.2e-2)}[case["dtype"]]
    if case["path"] == "chunk":
        return dict(rel=1.2e-2) if case["dtype"] == "bf16" else dict(rel=2e-3)
    # (experts: two that are almost equal for a row may change places, and that row's result with them)
    return dict(rel=1.2e-2, max=0.99) if case["path"] == "experts" else dict(rel=1.2e-2)


# ------------------------------------------------------------------ the same in 64 bits


def _silu(x):
    return x * torch.sigmoid(x)


def _attend64(q, k, v, first, scale, window=0, cap=0.0, bias=None, sink=None, talk=None, size=None, rate=None):
    """``q [n, H, D]`` at positions ``first ...`` over ``k [L, G, D]``, ``v [L, G, E]``."""
    n, heads, _ = q.shape
    keys, kv = k.shape[:2]
    per = heads // kv
    out = torch.empty(n, heads, v.shape[2], dtype=torch.float64, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    step = max(1, (1 << 26) // (heads * keys))
    at = torch.arange(keys, device=q.device)
    for r in range(0, n, step):
        rows = q[r: r + step]
        m = rows.shape[0]
        s = torch.matmul(rows.view(m, kv, per, -1).permute(1, 2, 0, 3).reshape(kv, per * m, -1), kt).view(heads, m, keys) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        back = torch.arange(first + r, first + r + m, device=q.device)[:, None] - at
        if bias is not None:
            s = s + bias[:, back.clamp(0, bias.shape[1] - 1)]
        if size is not None:
            s = s - size[:, None, None] * torch.log1p(rate[:, None, None] * back.clamp(min=0))
        hidden = (back < 0) | (back >= window) if window else back < 0
        s.masked_fill_(hidden, -math.inf)
        top = s.amax(2, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[:, None, None])
        s = torch.exp(s - top)
        den = s.sum(2, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink[:, None, None] - top)
        s = s / den
        if talk is not None:
            s = torch.matmul(talk, s.view(heads, -1)).view(heads, m, keys)
        out[r: r + step] = torch.matmul(s.view(kv, per * m, keys), vt).view(kv, per, m, -1).permute(2, 0, 1, 3).reshape(m, heads, -1)
    return out


def _attention64(case, s):
    path, kw = case["path"], {}
    k_pool, v_pool = s["k_pool"], s["v_pool"]
    if path == "chunk":
        k_pool, v_pool = k_pool.clone(), v_pool.clone()
        k_pool[s["slots"]], v_pool[s["slots"]] = s["k_new"], s["v_new"]
    if path == "scored":
        kw = dict(window=case["window"], cap=SOFTCAP if case["cap"] else 0.0, bias=s["bias"].double(), sink=s["sink"].double())
    elif path == "talking":
        kw = dict(talk=s["talk"].double(), size=s["size"].double(), rate=s["rate"].double())
    elif path == "decode":
        kw = dict(window=case["window"])
    out, at = [], 0
    for b, (n, new) in enumerate(zip(s["lens"], s["new"])):
        ids = torch.from_numpy(s["tables"][b, : -(-int(n) // BLOCK)].astype(np.int64)).cuda()
        rows = (ids[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)[: int(n)]
        k, v = k_pool[rows].double(), v_pool[rows].double()
        if "k_scale" in s:
            k, v = (t * sc[ids].double().repeat_interleave(BLOCK, 0)[: int(n), :, None] for t, sc in ((k, s["k_scale"]), (v, s["v_scale"])))
        out.append(_attend64(s["q"][at: at + int(new)].double(), k, v, int(n - new), case["dim"] ** -0.5, **kw))
        at += int(new)
    out = torch.cat(out)
    return (out, k_pool.double(), v_pool.double()) if path == "chunk" else out


def _recurrence64(case, s, seed):
    path, lens, steps = case["path"], s["lens"], case["steps"]
    heads, groups, dim, vdim, batch = case["heads"], case["groups"], case["dim"], case["vdim"], len(s["lens"])
    u = s["u"][:, : sum(s["sizes"])]
    # every sequence's rows, its further tokens behind them; -1: none
    total, starts = int(lens.sum()), np.cumsum(lens) - lens
    at = np.full((batch, int(lens.max()) + steps), -1, dtype=np.int64)
    for b, n in enumerate(lens):
        at[b, :n] = starts[b] + np.arange(n)
        at[b, n: n + steps] = total + b + batch * np.arange(steps)
    at = torch.from_numpy(at).cuda()
    state = torch.zeros(batch, heads, dim, vdim, dtype=torch.float64, device="cuda")
    norm, top = torch.zeros(batch, heads, dim, dtype=torch.float64, device="cuda"), torch.zeros(batch, heads, dtype=torch.float64, device="cuda")
    out = torch.zeros(u.shape[0], heads, vdim, dtype=torch.float64, device="cuda")
    wide = lambda t, n: t.view(batch, -1, n).repeat_interleave(heads * n // t.shape[1], 1)  # noqa: E731
    for t in range(at.shape[1]):
        rows, live = at[:, t], at[:, t] >= 0
        on = live.double()[:, None]
        parts = u[rows.clamp(min=0)].double().split(s["sizes"], 1)
        v = parts[2].view(batch, heads, vdim)
        if path == "channel":
            q, f = _silu(parts[0]).view(batch, heads, dim), s["lower"] + (1 - s["lower"].double()) * torch.sigmoid(parts[1] + s["f_bias"])
            k = (1 - f).view(batch, heads, dim)
            keep = f.view(batch, heads, dim, 1)
        else:
            q, k = wide(parts[0], dim), wide(parts[1], dim)
        if path == "lightning":
            q, k, v = _silu(q), _silu(k), _silu(v)
            keep = s["powers"][:, 1].double()[None, :, None, None]
        elif path == "mlstm":
            i = GATE_CAP * torch.tanh((parts[3] + s["i_bias"]) / GATE_CAP)
            f = torch.nn.functional.logsigmoid(GATE_CAP * torch.tanh((parts[4] + s["f_bias"]) / GATE_CAP))
            new = torch.maximum(f + top, i)
            keep, k = torch.exp(f + top - new)[..., None, None], k * torch.exp(i - new)[..., None]
            top = torch.where(live[:, None], new, top)
            q = q * dim ** -0.5
        elif path == "ssd":
            dt = torch.nn.functional.softplus(parts[3] + s["dt_bias"])
            keep, k = torch.exp(-s["rate"] * dt)[..., None, None], k * dt[..., None]
        elif path == "delta":
            q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
            q = q * dim ** -0.5
            keep = torch.exp(-s["rate"] * torch.nn.functional.softplus(parts[3] + s["dt_bias"]))[..., None, None]
            v = torch.sigmoid(parts[4])[..., None] * (v - torch.matmul((k[..., None, :]), keep * state)[..., 0, :])
        k = k * on[..., None]
        state = torch.where(live[:, None, None, None], keep * state, state) + k[..., None] * v[..., None, :]
        o = torch.matmul(q[..., None, :], state)[..., 0, :]
        if path == "mlstm":
            norm = torch.where(live[:, None, None], keep[..., 0] * norm, norm) + k
            o = o / (torch.maximum((norm * q).sum(-1).abs(), torch.exp(-top)) + DEN_EPS)[..., None]
        elif path == "ssd":
            o = o + s["skip"][:, None] * v
        out[rows[live]] = o[live]
    state = torch.nn.functional.pad(state, (0, _pad16(vdim) - vdim, 0, _pad16(dim) - dim))
    slots = torch.from_numpy(np.random.default_rng(int(seed)).permutation(batch)).cuda()
    kept = torch.empty_like(state)
    kept[slots] = state
    if path == "ssd":
        kept = kept.view(batch, heads, -1)
    return out.view(u.shape[0], -1), None if path == "mlstm" else kept


def _experts64(case, s):
    rows, width, inner, e, top = (case[n] for n in ("rows", "width", "inner", "experts", "top"))
    h = s["h"].double()
    logits = h @ s["router"].double().t()
    scores = torch.sigmoid(logits[:, :e])
    best = scores.view(rows, 8, e // 8).topk(min(2, e // 8), 2).values.sum(2).topk(4, 1).indices
    stay = torch.zeros(rows, 8, dtype=torch.bool, device="cuda").scatter_(1, best, True).repeat_interleave(e // 8, 1)
    picked = scores.masked_fill(~stay, -1.0).topk(top, 1)
    weights = picked.values / (picked.values.sum(1, keepdim=True) + 1e-20)
    y = torch.sigmoid(logits[:, e:]) * s["shared"].double()
    for n in range(e):
        row, place = (picked.indices == n).nonzero(as_tuple=True)
        if row.numel():
            u = h[row] @ s["w_in"][n].double().t()
            y.index_add_(0, row, weights[row, place, None] * ((_silu(u[:, :inner]) * u[:, inner:]) @ s["w_out"][n].double().t()))
    x = s["x"].double() + y / torch.sqrt((y * y).mean(1, keepdim=True) + 1e-6) * s["y_weight"]
    return x, x


def exact(case, seed):
    s = _inputs(case, seed)
    if case["path"] == "experts":
        return _experts64(case, s)
    return _recurrence64(case, s, seed) if case["path"] in RECURRENT else _attention64(case, s)
