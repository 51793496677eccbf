"""What is timed of this library, as a serving program uses it: the int4 linear layers of
transformer blocks from one decode row to a prefill chunk, on checkpoints as stored and in the
prepared layout, in plain and in act-order, fp16 and bfloat16; a fused mixture-of-experts layer
in decode and in prefill; and the standalone dequantisation.

A case is a dict of plain values. `op` names the entry point, `shapes` the layers of one pass
("KxN,KxN", each with its own weights and activations), `blocks` how often that list repeats
(with new weights each time, so that one pass reads more than stays in a cache), `graph` whether
the program captures the pass into a HIP graph once and replays it, which is how a decode step is
run, where a call takes a few microseconds.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
AWQ_ORDER = (0, 4, 1, 5, 2, 6, 3, 7)   # column n of a group of 8 sits in nibble AWQ_ORDER[n]
# the linear layers of one transformer block: fused q, k, v; attention output; fused gate and
# up; down (hidden size 4096, intermediate size 14336)
BLOCK = "4096x6144,4096x4096,4096x28672,14336x4096"
# its share on each of eight GPUs, tensor parallel: gate or up, and down
SHARE = "4096x1792,1792x4096"


def _package():
    """The package of the tree this process runs in (its folder is no Python identifier)."""
    name = "triton_rs_amd"
    if name not in sys.modules:
        path = os.path.join(ROOT, "triton-rs_amd")
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(path, "__init__.py"), submodule_search_locations=[path])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------ the cases

def _linear(name, op, fmt, M, shapes, G=128, dtype="f16", blocks=1, graph=False):
    c = {"op": op, "fmt": fmt, "M": M, "shapes": shapes, "G": G, "dtype": dtype,
         "blocks": blocks, "graph": graph}
    return {"name": name, **c} if name else c


def _moe(name, fmt, T, K, I, E, topk, G=128, graph=False):
    c = {"op": "moe", "fmt": fmt, "T": T, "K": K, "I": I, "E": E, "topk": topk, "G": G,
         "graph": graph}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest: one row through one square projection, a single call
        _linear("call_gptq_sym_m1", "gemm", "gptq_sym", 1, "4096x4096"),
        # one decode step of one sequence through the linear layers of two blocks, AWQ weights
        # prepared at load time
        _linear("decode_awq_prepared_m1", "prepared", "awq", 1, BLOCK, blocks=2, graph=True),
        # one decode step of eight sequences, GPTQ checkpoint as stored
        _linear("decode_gptq_m8", "gemm", "gptq", 8, BLOCK, graph=True),
        # sixteen sequences on an act-order (desc_act) GPTQ checkpoint
        _linear("decode_actorder_m16", "actorder", "gptq", 16, BLOCK, graph=True),
        # forty-eight sequences, AWQ checkpoint as stored
        _linear("decode_awq_m48", "gemm", "awq", 48, BLOCK, graph=True),
        # a short prompt, or a mixed batch of decodes and a prefill chunk, in bfloat16
        _linear("chunk_gptq_bf16_m200", "gemm", "gptq", 200, BLOCK, dtype="bf16"),
        # a ragged chunk on one GPU's share of a tensor-parallel MLP, groups of 64, prepared
        _linear("chunk_share_prepared_m333", "prepared", "awq", 333, SHARE, G=64, blocks=2),
        # a full prefill chunk through the MLP projections
        _linear("prefill_awq_m2048", "gemm", "awq", 2048, "4096x14336,14336x4096"),
        # the same on an act-order checkpoint, one projection
        _linear("prefill_actorder_m2048", "actorder", "gptq", 2048, "4096x6144"),
        # a mixture-of-experts layer in decode: sixteen sequences, two of eight experts each
        _moe("moe_decode_t16", "gptq", 16, 4096, 14336, 8, 2, graph=True),
        # and in prefill
        _moe("moe_prefill_t512", "gptq", 512, 4096, 14336, 8, 2),
        # a checkpoint matrix to dense fp16 weights, [N, K], for a program's own GEMM
        {"name": "dequant_gptq_transposed", "op": "dequant", "fmt": "gptq",
         "shapes": "4096x14336", "G": 128, "dtype": "f16", "transposed": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _size(rng, lo, hi, step):
    return max(lo, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["call", "prepared", "decode", "actorder", "chunk", "prefill", "moe", "moe",
                       "dequant"])
    fmt = rng.choice(["gptq", "gptq_sym", "awq", "awq"])
    G = rng.choice([32, 64, 128, 128, 128])
    dtype = rng.choice(["f16", "f16", "bf16"])
    K, N = _size(rng, 1024, 14336, 128), _size(rng, 1024, 16384, 64)
    if kind == "call":
        return _linear(None, "gemm", fmt, _log_int(rng, 1, 4), f"{K}x{N}", G, dtype)
    if kind == "prepared":
        # decode batches and chunks on prepared weights (fp16); the chunks in whole tiles
        if rng.random() < 0.6:
            return _linear(None, "prepared", fmt, _log_int(rng, 1, 64), f"{K}x{N},{N // 128 * 128}x{K}", G,
                           graph=True)
        return _linear(None, "prepared", fmt, _log_int(rng, 65, 1024),
                       f"{K}x{N // 256 * 256},{N // 256 * 256}x{K // 256 * 256}", max(G, 64))
    if kind == "decode":
        return _linear(None, "gemm", fmt, _log_int(rng, 1, 64), f"{K}x{N},{N // 128 * 128}x{K}", G, dtype,
                       graph=True)
    if kind == "actorder":
        # groups of 128 rows as stored, from a decode row to a chunk
        return _linear(None, "actorder", rng.choice(["gptq", "gptq_sym"]), _log_int(rng, 2, 1024),
                       f"{K}x{N // 256 * 256}", 128, dtype, graph=rng.random() < 0.5)
    if kind == "chunk":
        if rng.random() < 0.25:   # a width that is no multiple of a tile, as tensor parallelism leaves
            return _linear(None, "gemm", fmt, _log_int(rng, 65, 200),
                           f"{_size(rng, 1024, 4096, 128)}x{_size(rng, 512, 4096, 16)}", 128, dtype)
        return _linear(None, "gemm", fmt, _log_int(rng, 65, 512), f"{K}x{N // 128 * 128}", max(G, 64), dtype)
    if kind == "prefill":
        return _linear(None, "gemm", fmt, _log_int(rng, 513, 2048), f"{K}x{N // 128 * 128}", max(G, 64),
                       dtype)
    if kind == "moe":
        T, decode = (_log_int(rng, 1, 48), True) if rng.random() < 0.6 else (_log_int(rng, 49, 512), False)
        return _moe(None, fmt, T, _size(rng, 1024, 4096, 256), _size(rng, 1024, 14336, 256),
                    rng.choice([4, 8, 8, 16]), rng.choice([1, 2, 2]), max(G, 64), decode)
    return {"op": "dequant", "fmt": fmt, "shapes": f"{K}x{N}", "G": G, "dtype": dtype,
            "transposed": rng.random() < 0.7}


# ------------------------------------------------------------------ inputs

def _shapes(case):
    one = [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]
    return one * case.get("blocks", 1)


def _words(gen, rows, cols, mean, std):
    """Packed int32 words whose nibbles are quantised normal weights: round(N(mean, std)),
    clamped to 0..15."""
    w = torch.zeros((rows, cols), dtype=torch.int32, device="cuda")
    for i in range(8):
        q = torch.randn((rows, cols), generator=gen, device="cuda").mul_(std).add_(mean)
        w |= q.round_().clamp_(0, 15).to(torch.int32) << (4 * i)
    return w


def _weights(gen, fmt, K, N, G, dtype):
    """(qweight, scales, qzeros) of a K -> N matrix: values of about 0.02, zero points near the
    middle of the range."""
    qw = _words(gen, K, N // 8, 7.5, 2.7) if fmt == "awq" else _words(gen, K // 8, N, 7.5, 2.7)
    sc = (torch.rand((K // G, N), generator=gen, device="cuda") * 0.008 + 0.004).to(dtype)
    qz = None if fmt == "gptq_sym" else _words(gen, K // G, N // 8, 7.0, 1.0)
    return qw, sc, qz


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    fmt, G = case["fmt"], case["G"]
    if case["op"] == "moe":
        T, K, I, E = case["T"], case["K"], case["I"], case["E"]
        w13 = [_weights(gen, fmt, K, 2 * I, G, torch.float16) for _ in range(E)]
        w2 = [_weights(gen, fmt, I, K, G, torch.float16) for _ in range(E)]
        x = torch.randn((T, K), generator=gen, device="cuda").half()
        logits = torch.randn((T, E), generator=gen, device="cuda")
        return {"w13": w13, "w2": w2, "x": x, "logits": logits}
    dt = DTYPES[case["dtype"]]
    layers = []
    for K, N in _shapes(case):
        lay = {"K": K, "N": N, "w": _weights(gen, fmt, K, N, G, dt)}
        if case["op"] != "dequant":
            lay["x"] = torch.randn((case["M"], K), generator=gen, device="cuda").to(dt)
        if case["op"] == "actorder":
            groups = torch.arange(K // G, dtype=torch.int32, device="cuda").repeat_interleave(G)
            lay["g_idx"] = groups[torch.randperm(K, generator=gen, device="cuda")].contiguous()
        layers.append(lay)
    return {"layers": layers}


def _stack(mats):
    return [None if m[0] is None else torch.stack(m) for m in zip(*mats)]


_capture_stream = None


def _captured(step):
    """`step`, run once (the library's workspaces grow to their size), then captured."""
    global _capture_stream
    if _capture_stream is None:
        _capture_stream = torch.cuda.Stream()
    _capture_stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_capture_stream):
        step()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=_capture_stream):
        step()
    return g.replay


def prepare(case, seed):
    pkg = _package()
    pkg.init(0)
    fmt, G, op = case["fmt"], case["G"], case["op"]
    d = _inputs(case, seed)
    if op == "moe":
        T, K, I, E = case["T"], case["K"], case["I"], case["E"]
        w13, w2, x, logits = _stack(d.pop("w13")), _stack(d.pop("w2")), d["x"], d["logits"]
        need = pkg.lib().w4a16_fused_moe_workspace_size(T, E, case["topk"], I, K, 64)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        out = torch.empty((T, K), dtype=torch.float16, device="cuda")
        outs = [out]

        def step():
            pkg.fused_moe(x, logits, w13, w2, topk=case["topk"], fmt=fmt, group_size=G, out=out,
                          workspace=ws)
    elif op == "dequant":
        (qw, sc, qz), t = d["layers"][0]["w"], case["transposed"]
        return {"run": lambda: pkg.dequant(qw, sc, qz, fmt=fmt, group_size=G, transposed=t)}
    else:
        layers = d["layers"]
        outs = [torch.empty((case["M"], lay["N"]), dtype=lay["x"].dtype, device="cuda") for lay in layers]
        if op == "prepared":
            for lay in layers:
                qw, sc, qz = lay.pop("w")
                lay["p"] = pkg.prepare_layout(qw, sc, qz, fmt=fmt, group_size=G)
            calls = [(lay["x"], lay["p"], o) for lay, o in zip(layers, outs)]

            def step():
                for x, p, o in calls:
                    pkg.gemm_prepared(x, p, out=o)
        else:
            calls = [(lay["x"], *lay["w"], lay.get("g_idx"), o) for lay, o in zip(layers, outs)]

            def step():
                for x, qw, sc, qz, gi, o in calls:
                    pkg.gemm(x, qw, sc, qz, fmt=fmt, group_size=G, g_idx=gi, out=o)
    go = _captured(step) if case["graph"] else step

    def run_once():
        go()
        return outs
    # a captured graph holds addresses only: the state keeps every tensor that the step uses
    return {"run": run_once, "step": step, "inputs": d}


def run(state):
    return state["run"]()


# ------------------------------------------------------------------ what a pass cannot do without

def _weight_bytes(fmt, K, N, G):
    return K * N / 2 + K // G * N * 2 + (0 if fmt == "gptq_sym" else K // G * N / 2)


def work(case):
    fmt, G = case["fmt"], case["G"]
    if case["op"] == "moe":
        T, K, I, E, topk = (case[k] for k in ("T", "K", "I", "E", "topk"))
        touched = E * (1 - (1 - topk / E) ** T)   # experts that some token is routed to
        return {"bytes": touched * (_weight_bytes(fmt, K, 2 * I, G) + _weight_bytes(fmt, I, K, G))
                + T * K * 4 + T * E * 4,
                "flops": 6.0 * T * topk * K * I}
    b = f = 0.0
    for K, N in _shapes(case):
        b += _weight_bytes(fmt, K, N, G)
        if case["op"] == "dequant":
            b += 2 * K * N
            f += 2.0 * K * N
        else:
            b += 2 * case["M"] * (K + N) + (4 * K if case["op"] == "actorder" else 0)
            f += 2.0 * case["M"] * K * N
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Measured against exact(): 2.1e-4 (fp16) and 1.7e-3 (bf16), the rounding of the result to 16
    # bits, where the weights are rounded as the formats define them, and 2.8e-4 where a kernel
    # applies a group's scale to the sum of unrounded products; 4.1e-4 through the layer of
    # experts, which rounds twice more in between. Four times that; single values by about two
    # units in the last place.
    if case["op"] == "dequant":
        return "exact"
    if case["op"] == "moe":
        return {"rel": 1.6e-3, "max": 1e-2}
    return {"rel": 1.2e-3, "max": 5e-3} if case["dtype"] == "f16" else {"rel": 7e-3, "max": 4e-2}


# ------------------------------------------------------------------ the same in 64 bits

def _nibbles(w, axis):
    """The 8 nibbles of each word, along a new last axis (axis 1) or after the rows (axis 0)."""
    n = torch.stack([(w >> (4 * i)) & 0xF for i in range(8)], dim=-1)   # [R, C, 8]
    if axis == 1:
        return n.reshape(w.shape[0], -1)
    return n.permute(0, 2, 1).reshape(-1, w.shape[1])


def _dense(fmt, w, K, N, G, dtype, g_idx=None, zero_offset=1):
    """The matrix [K, N] that the packed weights stand for: (q - z) s, rounded to the element
    type, which is how the formats define a weight."""
    qw, sc, qz = w
    if fmt == "awq":
        at = (torch.arange(N, device="cuda") // 8 * 8
              + torch.tensor(AWQ_ORDER, device="cuda").repeat(N // 8))
        q, z = _nibbles(qw, 1)[:, at], _nibbles(qz, 1)[:, at]
    else:
        q = _nibbles(qw, 0)
        z = torch.full((K // G, N), 8, dtype=torch.int32, device="cuda") if qz is None \
            else _nibbles(qz, 1) + zero_offset
    g = torch.arange(K, device="cuda") // G if g_idx is None else g_idx.long()
    return ((q - z[g]).double() * sc.double()[g]).to(dtype).double()


def exact(case, seed):
    d = _inputs(case, seed)
    fmt, G = case["fmt"], case["G"]
    if case["op"] == "moe":
        T, K, I, E = case["T"], case["K"], case["I"], case["E"]
        prob = torch.softmax(d["logits"].double(), dim=1)
        wt, ids = torch.topk(prob, case["topk"], dim=1)
        wt = wt / wt.sum(dim=1, keepdim=True)
        y = torch.zeros((T, K), dtype=torch.float64, device="cuda")
        for e in range(E):
            rows, slot = (ids == e).nonzero(as_tuple=True)
            if not len(rows):
                continue
            h = d["x"][rows].double() @ _dense(fmt, d["w13"][e], K, 2 * I, G, torch.float16)
            a = h[:, :I] * torch.sigmoid(h[:, :I]) * h[:, I:]
            y.index_add_(0, rows, wt[rows, slot].unsqueeze(1)
                         * (a @ _dense(fmt, d["w2"][e], I, K, G, torch.float16)))
        return [y]
    outs = []
    for lay in d["layers"]:
        w = _dense(fmt, lay["w"], lay["K"], lay["N"], G, DTYPES[case["dtype"]], lay.get("g_idx"))
        if case["op"] == "dequant":
            return w.t().contiguous() if case["transposed"] else w
        outs.append(lay["x"].double() @ w)
    return outs
