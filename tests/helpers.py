"""Shared test helpers: package loading, device transfer and the parity tolerance."""
from __future__ import annotations

import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

import __graft_entry__  # noqa: E402

RTOL = 1e-2  # the path's bar: max relative error 1e-2 vs fp32 dequant-then-matmul


def pkg():
    return __graft_entry__.load_package()


def route(fmt, M, N, K, G, bf16=False, has_g_idx=False):
    """The instance a call runs: ("direct", r, nwn, kw, K split), ("prefill", rows, columns, 0, K split)
    or ("other", 0, 0, 0, 0); fmt "prep": the prepared layout beyond the kernels for few rows."""
    import ctypes
    P = pkg()
    out = (ctypes.c_int32 * 5)()
    P.lib().w4a16_internal_route((3 if fmt == "prep" else P.FORMATS[fmt]) | (P.BF16 if bf16 else 0),
                                 M, N, K, G, int(has_g_idx), out)
    return (("other", "direct", "prefill")[out[0]], *out[1:])


def moe_route(fmt, T, K, I, E, topk, G):
    """What the expert GEMMs of a fused layer run: ("direct", tile rows, (r, nwn, kw) of gate/up, of down)
    or ("prefill", tile rows, (columns, 0, 0) of gate/up, (columns, 0, K split) of down)."""
    import ctypes
    P = pkg()
    out = (ctypes.c_int32 * 8)()
    P.lib().w4a16_internal_moe_route(3 if fmt == "prep" else P.FORMATS[fmt], T, K, I, E, topk, G, out)
    return ("", "direct", "prefill")[out[0]], out[1], tuple(out[2:5]), tuple(out[5:8])


def to_dev(a, device="cuda:0"):
    import torch
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint32:
        a = a.view(np.int32)
    return torch.from_numpy(a).to(device)


def rel_err(got, ref) -> float:
    """max |got - ref| / max(|ref|, rms(ref)) -- relative error with an rms floor.

    A pure per-element relative error is unbounded where the reference is ~0; the floor
    (the reference's own rms) follows the reference's tol = max(atol, rel*|want|) pattern
    (crates/triton-runtime/examples/run_vec_add.rs:142)."""
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    floor = np.sqrt(np.mean(ref ** 2)) if ref.size else 0.0
    scale = np.maximum(np.abs(ref), floor)
    scale[scale == 0] = 1.0
    return float(np.max(np.abs(got - ref) / scale)) if ref.size else 0.0


def assert_parity(got, ref, tol=RTOL, what=""):
    e = rel_err(got, ref)
    assert e <= tol, f"{what}: max relative error {e:.3e} > {tol}"
    return e
