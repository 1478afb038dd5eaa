"""Helpers shared by the GPU parity tests: move a synthetic workload to the
device and run the C-ABI entry points on it (through research_amd.ops)."""

import ctypes

import numpy as np
import torch

from research_amd import _lib, ops

DEV = "cuda:0"


def announce(msg):
    """Name the case before its first kernel launch, flushed, so a fault can be attributed."""
    print(f"[gpu-case] {msg}", flush=True)


def tables_to_device(tables, width=None):
    w = max(max((len(t) for t in tables), default=1), 1) if width is None else width
    out = np.full((len(tables), w), -1, dtype=np.int32)
    for i, t in enumerate(tables):
        out[i, : len(t)] = np.asarray(t, dtype=np.int64)
    return torch.from_numpy(out).to(DEV)


WIDE = 1 << 16  # columns of a block table that only the split pass takes


def decode_route(batch, hq, hkv, d, q_dtype, kv_dtype, columns, bs, window=0):
    """What pa_decode launches: 0: the split pass; -1: that pass, a workgroup for each sequence; else runs of the kernel for narrow tables."""
    runs = ctypes.c_int()
    assert _lib.load().pa_decode_launches(batch, hq, hkv, d, columns, bs, window, ops.PA_DTYPE[q_dtype], ops.PA_DTYPE[kv_dtype], ctypes.byref(runs)) > 0
    return runs.value


def decode_by_split_pass(q, k_pool, v_pool, tables, lens, bs, scale, extra_zero=None, k_scale=None, v_scale=None, window=0):
    """pa_decode by the split pass, whatever the lengths: over tables padded far beyond them or, under a window, which bounds what a table's
    width says, with so many copies of the batch that no other way takes it.  q, pools and scales on the device, the rest host lists."""
    batch, hq, d = q.shape
    copies = 1 if not window else 512 // batch + 1
    dev = lambda x: torch.tensor(list(x) * copies, dtype=torch.int32, device=DEV)
    padded = tables_to_device(tables, None if window else WIDE).repeat(copies, 1)
    assert decode_route(batch * copies, hq, k_pool.shape[1], d, q.dtype, k_pool.dtype, padded.shape[1], bs, window) == 0
    got = ops.decode(q.repeat(copies, 1, 1), k_pool, v_pool, padded, dev(lens), bs, scale, ops.decode_workspace(q.repeat(copies, 1, 1), k_pool),
                     None if extra_zero is None else dev(extra_zero), k_scale, v_scale, window=window)
    return got.view(copies, batch, hq, d)


def run_decode(q, k_pool, v_pool, tables, seq_lens, block_size, scale, extra_zero=None, k_scale=None, v_scale=None,
               wgs_per_call=None):
    """q [B,Hq,D] and pools already on the device; tables/seq_lens host lists.  Returns a device tensor.  (Where the call does not take the split
    pass by its tables' width, that pass has to agree.)"""
    lens = np.asarray(seq_lens, dtype=np.int32)
    ws = ops.decode_workspace(q, k_pool)
    ez = None if extra_zero is None else torch.from_numpy(np.asarray(extra_zero, dtype=np.int32)).to(DEV)
    narrow = tables_to_device(tables)
    got = ops.decode(q, k_pool, v_pool, narrow, torch.from_numpy(lens).to(DEV), block_size, scale, ws, ez, k_scale, v_scale)
    if decode_route(*q.shape[:2], k_pool.shape[1], q.shape[2], q.dtype, k_pool.dtype, narrow.shape[1], block_size) != 0:
        wide = decode_by_split_pass(q, k_pool, v_pool, tables, lens.tolist(), block_size, scale, extra_zero, k_scale, v_scale)[0]
        # (both round to the type of q, at most 2^-8 of a value apart, and one has weights of 16 bits: 2^-9 of values of at most 5)
        assert_close(wide, got, 1e-5 if q.dtype == torch.float32 else 2e-2, "the split pass")
    return got


def assert_close(got, want, tol, what=""):
    """|got - want| <= tol * (1 + |want|): the absolute/relative bar used for attention outputs."""
    got = got.detach().to(torch.float64).cpu().numpy() if isinstance(got, torch.Tensor) else np.asarray(got)
    want = want.detach().to(torch.float64).cpu().numpy() if isinstance(want, torch.Tensor) else np.asarray(want)
    assert got.shape == want.shape, f"{what}: shape {got.shape} vs {want.shape}"
    assert np.isfinite(got).all(), f"{what}: non-finite output"
    err = np.abs(got - want) / (1.0 + np.abs(want))
    assert err.max() <= tol, f"{what}: max err {err.max():.3e} > {tol:.1e} at {np.unravel_index(err.argmax(), err.shape)}"
