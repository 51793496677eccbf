"""GPU parity of the direct kernel (csrc/direct_body.h: weights dequantised in registers, tiles of
16 to 112 rows) at the sizes where it can go wrong: remainders of its row and column tiles, K in
shares that its wave groups and workgroups do not divide evenly, every group size, format, element
type and instance (each case names its own, which a test without GPU holds it to). x holds whole numbers up to 2 in size and the scales are powers of two, so that
every product and partial sum (below 2^24 units) is exact in fp32 in any order: the output must be
the exact sum rounded once, bit for bit."""
import math

import numpy as np
import pytest

from helpers import moe_route, pkg, route, to_dev
from synth import Problem

NAME = {0: "gptq", 1: "gptq_sym", 2: "awq"}


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def exact_problem(fmt, M, K, N, G, ao=False):
    p = Problem(fmt, M=M, K=K, N=N, G=G, seed=9000 + M + K + N + G, act_order=ao)
    g = np.random.default_rng(M * 31 + N)
    p.x = g.integers(-2, 3, size=(M, K)).astype(np.float16)
    p.scales = (2.0 ** -g.integers(6, 9, size=p.scales.shape)).astype(np.float16)
    row_group = np.arange(K) // G if p.g_idx is None else p.g_idx
    w = (p.q - p.zero_int()[row_group]) * p.scales.astype(np.float32)[row_group]
    return p, p.x.astype(np.float32) @ w.astype(np.float32)     # exact: below 2^24 units of 2^-8


def check(torch, y, want, dtype):
    torch.cuda.synchronize()
    assert torch.equal(y.cpu(), torch.from_numpy(want).to(dtype))


CASES = [                                   # rows, N, K, group, element type, instance
    # AWQ, up to 64 rows: one tile of 16 R rows; one to eight splits of K
    (2, 9, 544, 640, 64, "f16", "1x2x2/1"), (2, 16, 4096, 4096, 128, "f16", "other"),
    (2, 17, 1056, 4096, 256, "f16", "2x2x2/8"),
    (2, 33, 1056, 512, 32, "f16", "3x2x2/1"), (2, 48, 2080, 1152, 128, "f16", "3x2x2/2"),
    (2, 49, 6144, 1024, 64, "f16", "4x2x2/1"),
    (2, 64, 4096, 4096, 128, "bf16", "4x2x2/4"), (2, 31, 512, 192, 64, "bf16", "2x2x2/1"),
    # GPTQ, 4 rows: wide shapes from K = 4096; bf16 where it stays below and from 17 rows
    (0, 4, 20480, 4096, 128, "f16", "1x2x2/1"), (1, 4, 28672, 4096, 64, "f16", "1x2x2/1"),
    (2, 9, 4096, 1792, 128, "bf16", "other"), (0, 17, 20480, 256, 64, "bf16", "2x2x2/1"),
    # GPTQ: wide shapes up to 64 rows, ragged widths, tiles of 64 and 112 rows by 128 and 256 columns
    (0, 16, 20480, 256, 64, "f16", "1x2x2/1"), (0, 48, 20488, 320, 32, "f16", "3x2x2/1"),
    (0, 64, 20480, 256, 128, "bf16", "4x2x2/1"),
    (0, 65, 520, 320, 64, "f16", "4x2x2/1"), (0, 113, 1096, 4096, 128, "f16", "4x2x2/8"),
    (0, 200, 6144, 4096, 128, "f16", "4x2x4/1"),
    (1, 200, 1544, 2048, 32, "bf16", "4x2x2/4"), (0, 224, 3080, 8192, 64, "f16", "4x2x4/2"),
    (1, 700, 3072, 1024, 128, "f16", "7x2x2/1"),
    (0, 1024, 6144, 512, 128, "f16", "7x4x1/1"), (1, 300, 8192, 4096, 512, "f16", "7x2x2/1"),
    (2, 100, 1024, 4096, 128, "bf16", "4x2x2/8"),
    (2, 581, 6144, 576, 64, "f16", "7x4x1/1"),
    # many rows: rounds of workgroups on one instance
    (0, 3072, 4096, 1792, 128, "f16", "7x4x1/1"), (2, 1280, 3584, 4096, 64, "bf16", "7x4x1/1"),
    (1, 1537, 1792, 1024, 64, "f16", "7x2x2/1"),
    (2, 3001, 1056, 1088, 32, "f16", "7x2x2/1"), (0, 2100, 1096, 640, 64, "bf16", "7x2x2/1"),
]

# every instance in both formats and element types, without and with K split over workgroups
INSTANCES = [
    (0, 9, 544, 192, 64, "f16", "1x2x2/1"), (0, 9, 544, 1984, 64, "f16", "1x2x2/4"),
    (0, 17, 544, 192, 64, "f16", "2x2x2/1"), (0, 17, 544, 1984, 64, "f16", "2x2x2/4"),
    (0, 33, 544, 192, 64, "f16", "3x2x2/1"), (0, 33, 544, 1088, 64, "f16", "3x2x2/2"),
    (0, 49, 544, 192, 64, "f16", "4x2x2/1"), (0, 49, 544, 1088, 64, "f16", "4x2x2/2"),
    (0, 65, 6176, 1984, 64, "f16", "4x2x4/1"), (0, 400, 544, 5888, 64, "f16", "4x2x4/4"),
    (0, 200, 8224, 320, 64, "f16", "7x2x2/1"), (0, 200, 2080, 6848, 64, "f16", "7x2x2/4"),
    (0, 200, 8224, 192, 64, "f16", "7x4x1/1"), (0, 447, 3616, 11968, 64, "f16", "7x4x1/4"),
    (0, 9, 544, 192, 64, "bf16", "1x2x2/1"), (0, 9, 544, 1088, 64, "bf16", "1x2x2/2"),
    (0, 17, 544, 192, 64, "bf16", "2x2x2/1"), (0, 17, 544, 1088, 64, "bf16", "2x2x2/2"),
    (0, 33, 544, 192, 64, "bf16", "3x2x2/1"), (0, 33, 544, 1088, 64, "bf16", "3x2x2/2"),
    (0, 49, 544, 192, 64, "bf16", "4x2x2/1"), (0, 49, 544, 1088, 64, "bf16", "4x2x2/2"),
    (0, 65, 8224, 1984, 64, "bf16", "4x2x4/1"), (0, 400, 544, 6848, 64, "bf16", "4x2x4/4"),
    (0, 200, 8224, 320, 64, "bf16", "7x2x2/1"), (0, 200, 2080, 3968, 64, "bf16", "7x2x2/4"),
    (0, 200, 8224, 192, 64, "bf16", "7x4x1/1"), (0, 200, 8224, 12288, 64, "bf16", "7x4x1/2"),
    (2, 9, 544, 192, 64, "f16", "1x2x2/1"), (2, 9, 544, 1984, 64, "f16", "1x2x2/4"),
    (2, 17, 544, 192, 64, "f16", "2x2x2/1"), (2, 17, 544, 1088, 64, "f16", "2x2x2/2"),
    (2, 33, 544, 192, 64, "f16", "3x2x2/1"), (2, 33, 544, 1088, 64, "f16", "3x2x2/2"),
    (2, 49, 544, 192, 64, "f16", "4x2x2/1"), (2, 49, 544, 1088, 64, "f16", "4x2x2/2"),
    (2, 1300, 544, 1984, 64, "f16", "4x2x4/1"), (2, 400, 544, 6848, 64, "f16", "4x2x4/4"),
    (2, 200, 8224, 320, 64, "f16", "7x2x2/1"), (2, 65, 4128, 4608, 64, "f16", "7x2x2/4"),
    (2, 200, 8224, 192, 64, "f16", "7x4x1/1"), (2, 447, 3616, 12288, 64, "f16", "7x4x1/4"),
    (2, 9, 544, 192, 64, "bf16", "1x2x2/1"), (2, 9, 544, 1088, 64, "bf16", "1x2x2/2"),
    (2, 17, 544, 192, 64, "bf16", "2x2x2/1"), (2, 17, 544, 1088, 64, "bf16", "2x2x2/2"),
    (2, 33, 544, 192, 64, "bf16", "3x2x2/1"), (2, 33, 544, 1088, 64, "bf16", "3x2x2/2"),
    (2, 49, 544, 192, 64, "bf16", "4x2x2/1"), (2, 49, 544, 1088, 64, "bf16", "4x2x2/2"),
    (2, 900, 1056, 1984, 64, "bf16", "4x2x4/1"), (2, 400, 544, 6848, 64, "bf16", "4x2x4/4"),
    (2, 200, 8224, 320, 64, "bf16", "7x2x2/1"), (2, 200, 2080, 3648, 64, "bf16", "7x2x2/4"),
    (2, 200, 8224, 192, 64, "bf16", "7x4x1/1"), (2, 223, 8224, 11968, 64, "bf16", "7x4x1/2"),
]


@pytest.mark.parametrize("fmt,M,N,K,G,et,instance", CASES + INSTANCES)
def test_cases_take_their_instance(fmt, M, N, K, G, et, instance):
    """R x waves along N x wave groups along K / K split ("other": not the direct kernel). No GPU."""
    kind, *shape = route(NAME[fmt], M, N, K, G, et == "bf16")
    assert instance == ("{}x{}x{}/{}".format(*shape) if kind == "direct" else "other")


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,M,N,K,G,et,instance", CASES + INSTANCES)
def test_direct_bit_exact(torch_cuda, fmt, M, N, K, G, et, instance):
    torch = torch_cuda
    dt = torch.float16 if et == "f16" else torch.bfloat16
    p, want = exact_problem(fmt, M, K, N, G)
    y = pkg().gemm(to_dev(p.x).to(dt), to_dev(p.qweight), to_dev(p.scales).to(dt),
                   None if fmt == 1 else to_dev(p.qzeros), fmt=NAME[fmt], group_size=G)
    check(torch, y, want, dt)


PREPARED = [    # checkpoint format, rows, N, K, group; instance (groups under 128 and 9 rows or more, or 65)
    (0, 2, 528, 384, 32, "other"), (2, 20, 272, 1024, 64, "2x2x2/2"), (1, 70, 1040, 1024, 128, "4x2x2/2"),
    (0, 333, 1792, 4096, 64, "4x2x4/2"), (2, 1000, 6160, 640, 128, "7x4x1/1"), (0, 130, 4096, 2048, 256, "4x2x2/2"),
    (0, 1281, 3584, 1024, 64, "7x4x1/1"),
    # every instance, without and with K split over workgroups
    (0, 9, 528, 128, 64, "1x2x2/1"), (0, 9, 528, 1920, 64, "1x2x2/4"), (0, 17, 528, 128, 64, "2x2x2/1"),
    (0, 33, 528, 128, 64, "3x2x2/1"), (0, 33, 528, 1152, 32, "3x2x2/2"), (0, 49, 528, 128, 64, "4x2x2/1"),
    (0, 65, 4112, 4096, 64, "4x2x4/2"), (0, 200, 8208, 256, 64, "7x2x2/1"), (0, 65, 4112, 6272, 64, "7x2x2/4"),
    (0, 200, 8208, 12288, 64, "7x4x1/2"),
]


@pytest.mark.parametrize("fmt,M,N,K,G,instance", PREPARED)
def test_prepared_cases_take_their_instance(fmt, M, N, K, G, instance):
    if instance != "other":              # that one: the GEMV for few rows
        kind, *shape = route("prep", M, (N + 31) // 32 * 32 if fmt == 2 else N, K, G)
        assert kind == "direct" and instance == "{}x{}x{}/{}".format(*shape)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,M,N,K,G,instance", PREPARED)
def test_direct_prepared_bit_exact(torch_cuda, fmt, M, N, K, G, instance):
    P = pkg()
    if fmt == 2 and N % 32:
        N = N // 32 * 32 + 32                # the AWQ checkpoint's own width
    p, want = exact_problem(fmt, M, K, N, G)
    w = P.prepare_layout(to_dev(p.qweight), to_dev(p.scales), None if fmt == 1 else to_dev(p.qzeros),
                         fmt=NAME[fmt], group_size=G, zero_offset=p.zero_offset)
    check(torch_cuda, P.gemm_prepared(to_dev(p.x), w), want, torch_cuda.float16)


GATED = [(200, 1096, 1024, True), (300, 6144, 512, True), (200, 1096, 1024, False),
         (300, 6144, 512, False), (150, 1024, 4096, True), (150, 1024, 4096, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,valid", GATED)
def test_direct_behind_act_order_gate(torch_cuda, M, N, K, valid):
    """Beyond the small-batch kernel's rows, on rows put in group order (K whole, K split over
    workgroups); with groups of other sizes the gate leaves the output to the generic kernel. Widths
    without a prefill plan (1096) go to that one at once."""
    kind, _, _, _, split = route("gptq", M, N, K, 128, has_g_idx=True)
    assert kind == ("other" if N == 1096 else "direct") and (split > 1) == (K == 4096)
    p, want = exact_problem(0, M, K, N, 128, ao=True)
    if not valid:
        p.g_idx = np.where(np.arange(K) == 3, (p.g_idx + 1) % (K // 128), p.g_idx).astype(np.int32)
        w = (p.q - p.zero_int()[p.g_idx]) * p.scales.astype(np.float32)[p.g_idx]
        want = p.x.astype(np.float32) @ w.astype(np.float32)
    args = [to_dev(v) for v in (p.x, p.qweight, p.scales, p.qzeros)]
    for _ in range(2):                       # the split's counters are left at zero either way
        y = pkg().gemm(*args, fmt="gptq", group_size=128, g_idx=to_dev(p.g_idx))
        check(torch_cuda, y, want, torch_cuda.float16)


def test_plan_of_widths_other_kernels_do_not_tile():
    """Widths that no tile of the other kernels divides leave the generic kernel from 512 columns on."""
    P = pkg()
    for fmt, N in (("gptq", 520), ("gptq_sym", 1544), ("awq", 544)):
        for bf16 in (False, True):
            assert P.plan(fmt, 100, N, 640, 64, bf16=bf16) == "prefill"
            assert P.plan(fmt, 20, N, 640, 64, bf16=bf16) == "skinny"
    assert P.plan("gptq", 100, 504, 640, 64) == "strided"
    assert P.plan("gptq", 100, 520, 1632, 96) == "strided"      # groups that share a stage unevenly
    assert P.plan("gptq", 100, 520, 96, 32) == "strided"        # K that no stage divides


# ------------------------------------------------------------------ by expert

# rows per expert, at the edges of 16-row blocks, of tiles of 64 and of 112 rows: one to four tiles each
FEW = [0, 1, 15, 16, 17, 32, 33, 48, 49, 64]
MANY = [0, 1, 17, 49, 64, 65, 80, 81, 96, 97, 112, 113, 160, 225]
LONG = [65, 96, 97, 112, 160, 208]


def expert_layer(counts, fmt, K, I, G, seed):
    """x, logits (expert e chosen by exactly counts[e] tokens, interleaved) and stacked weights."""
    g = np.random.default_rng(seed)
    ids = g.permutation(np.repeat(np.arange(len(counts)), counts))
    x = g.standard_normal((len(ids), K)).astype(np.float16)
    logits = np.where(np.arange(len(counts)) == ids[:, None], 4.0, 0.0).astype(np.float32)

    def stack(rows, cols, s):
        ps = [Problem(fmt, M=1, K=rows, N=cols, G=G, seed=s + e) for e in range(len(counts))]
        cat = lambda f: None if getattr(ps[0], f) is None else to_dev(np.stack([getattr(q, f) for q in ps]))
        return cat("qweight"), cat("scales"), cat("qzeros")
    return to_dev(x), to_dev(logits), stack(K, 2 * I, seed * 100), stack(I, K, seed * 100 + 50)


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [FEW, MANY], ids=["few", "many"])
@pytest.mark.parametrize("fmt,K,I,G", [(0, 512, 256, 64), (1, 256, 384, 64), (2, 256, 640, 128), (0, 256, 8192, 128),
                                       (2, 256, 8192, 64)])
def test_direct_by_expert(torch_cuda, counts, fmt, K, I, G):
    """Experts whose rows end at the edges of the tiles, which are 64 rows high for these narrow layers
    (test_direct_by_expert_tall: 112). With K in one chain the layer is the
    composition of the public pieces bit for bit; a long down projection (I = 8192) adds the sums of
    its wave groups in another order: within the fp32 rounding of the sums, two roundings of the
    16-bit results (h, y) and the weights' share: 2e-3 of the largest."""
    from test_gpu_moe import _layer_by_pieces
    P = pkg()
    x, logits, w13, w2 = expert_layer(counts, fmt, K, I, G, 7 + fmt)
    args = dict(topk=1, fmt=NAME[fmt], group_size=G)
    tiles = moe_route(NAME[fmt], sum(counts), K, I, len(counts), 1, G)
    assert tiles == ("direct", 64, (7, 4, 1), (7, 4, 1) if I < 8192 else (4, 2, 4))
    y = P.fused_moe(x, logits, w13, w2, **args)
    again = P.fused_moe(x, logits, w13, w2, **args)
    want = _layer_by_pieces(P, x, logits, w13, w2, 1, NAME[fmt], G, 64)
    assert torch_cuda.equal(y, again)
    if I < 8192:
        assert torch_cuda.equal(y, want)
    prep = [y] if fmt == 1 else [y, P.fused_moe_prepared(
        x, logits, *(P.prepare_layout_experts(*w, fmt=NAME[fmt], group_size=G) for w in (w13, w2)), topk=1)]
    for got in prep:
        err = (got.float() - want.float()).abs().max() / want.float().abs().max()
        assert err.item() <= 2e-3


def random_layer(torch, counts, fmt, K, I, G, seed):
    """As expert_layer, the weights' words and scales drawn on the device."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    E = len(counts)
    ids = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(len(ids), generator=g, device="cuda")]
    x = torch.randn((len(ids), K), generator=g, device="cuda").half()
    logits = torch.where(torch.arange(E, device="cuda") == ids[:, None], 4.0, 0.0)

    def stack(rows, cols):
        def words(*shape):
            return torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, device="cuda", dtype=torch.int64).int()
        q = words(E, rows, cols // 8) if fmt == 2 else words(E, rows // 8, cols)
        sc = torch.rand((E, rows // G, cols), generator=g, device="cuda") * 0.01 + 0.002
        return q, sc.half(), None if fmt == 1 else words(E, rows // G, cols // 8)
    return x, logits.float(), stack(K, 2 * I), stack(I, K)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,counts,K,I,G", [
    (0, MANY, 2048, 1536, 128), (1, MANY, 2048, 1536, 64), (2, MANY, 2048, 1536, 128),
    (0, LONG, 2048, 8192, 64), (2, LONG, 2048, 8192, 128)], ids=["gptq", "sym", "awq", "gptq-long", "awq-long"])
def test_direct_by_expert_tall(torch_cuda, fmt, counts, K, I, G):
    """Tiles of up to 112 rows, every height from one to seven 16-row blocks, the long down projection
    over two wave groups. Equal to the pieces, or within the bounds of test_direct_by_expert."""
    from test_gpu_moe import _layer_by_pieces
    P = pkg()
    down = (7, 4, 1) if I < 8192 else (7, 4, 2)
    for f in (NAME[fmt], "prep"):
        assert moe_route(f, sum(counts), K, I, len(counts), 1, G) == ("direct", 112, (7, 4, 1), down)
    x, logits, w13, w2 = random_layer(torch_cuda, counts, fmt, K, I, G, 70 + fmt)
    args = dict(topk=1, fmt=NAME[fmt], group_size=G)
    y = P.fused_moe(x, logits, w13, w2, **args)
    again = P.fused_moe(x, logits, w13, w2, **args)
    want = _layer_by_pieces(P, x, logits, w13, w2, 1, NAME[fmt], G, 64)
    assert torch_cuda.equal(y, again)
    if I < 8192:
        assert torch_cuda.equal(y, want)
    prep = [] if fmt == 1 else [P.fused_moe_prepared(
        x, logits, *(P.prepare_layout_experts(*w, fmt=NAME[fmt], group_size=G) for w in (w13, w2)), topk=1)]
    for got in [y] + prep:
        err = (got.float() - want.float()).abs().max() / want.float().abs().max()
        assert err.item() <= 2e-3


def test_expert_tiles_are_direct_or_of_256_rows():
    """Over layers of every size: tiles of 64 or 112 rows on the direct kernel, of 256 on the prefill
    kernel, there where they are over 0.83 full or an expert has over 1024 rows."""
    seen = set()
    for E in (1, 4, 8, 60, 256):
        for T in (1, 5, 60, 400, 880, 1900, 3600, 8000):
            for topk in (1, 2):
                for K, I in ((256, 256), (1024, 896), (4096, 2048), (4096, 14336)):
                    kind, rows, _, _ = moe_route("gptq", T, K, I, E, min(topk, E), 128)
                    mean = T * min(topk, E) / E
                    full = math.ceil((mean + math.sqrt(mean)) / 256)
                    assert kind == ("prefill" if mean > 1024 or mean > 0.83 * 256 * full else "direct")
                    seen.add((kind, rows))
    assert seen == {("direct", 64), ("direct", 112), ("prefill", 256)}


# 256-row tiles of the prefill kernel: rows of experts on average, experts, K, I; columns of gate/up, of
# down, K split of down
FULL = [(216, 4, 256, 512, 128, 128, 1), (216, 16, 256, 1792, 224, 128, 1), (216, 10, 256, 2048, 256, 128, 1),
        (240, 4, 256, 8192, 256, 256, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("mean,E,K,I,bn13,bn2,ks2", FULL)
def test_expert_tiles_of_256_rows(torch_cuda, fmt, mean, E, K, I, bn13, bn2, ks2):
    """Experts of about 216 or 240 rows, one of 256 and one just above: the prefill kernel's tiles.
    Equal to the pieces where K is whole, else (and prepared) within the bounds above."""
    from test_gpu_moe import _layer_by_pieces
    P = pkg()
    counts = [mean] * (E - 4) + [257, 256, 2 * mean - 257 + 16, 2 * mean - 256 - 16]
    assert sum(counts) == mean * E
    for f in (NAME[fmt], "prep"):
        assert moe_route(f, mean * E, K, I, E, 1, 128) == ("prefill", 256, (bn13, 0, 0), (bn2, 0, ks2))
    x, logits, w13, w2 = random_layer(torch_cuda, counts, fmt, K, I, 128, 90 + fmt)
    args = dict(topk=1, fmt=NAME[fmt], group_size=128)
    y = P.fused_moe(x, logits, w13, w2, **args)
    again = P.fused_moe(x, logits, w13, w2, **args)
    want = _layer_by_pieces(P, x, logits, w13, w2, 1, NAME[fmt], 128, 64)
    assert torch_cuda.equal(y, again)
    if ks2 == 1:
        assert torch_cuda.equal(y, want)
    prep = [] if fmt == 1 else [P.fused_moe_prepared(
        x, logits, *(P.prepare_layout_experts(*w, fmt=NAME[fmt], group_size=128) for w in (w13, w2)), topk=1)]
    for got in [y] + prep:
        err = (got.float() - want.float()).abs().max() / want.float().abs().max()
        assert err.item() <= 2e-3


# ------------------------------------------------------------------ under capture

def fresh_stream(torch):
    """A stream the library has not seen (torch's own streams come from a pool and are reused)."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    h = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(h)) == 0
    return torch.cuda.ExternalStream(h.value)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,M,N,K,warm", [
    (0, 48, 1032, 4096, 0), (2, 17, 1056, 4096, 0), (0, 113, 1096, 4096, 0), ("prep", 80, 1040, 2048, 0),
    (0, 333, 4104, 14336, 9), (2, 200, 3104, 14336, 9)])
def test_direct_captured_without_its_workspace(torch_cuda, fmt, M, N, K, warm):
    """A call that splits K, captured on a stream with no workspace or one too small for the split (that
    of a call of `warm` rows), runs with fewer splits instead of asking for one."""
    torch, P = torch_cuda, pkg()
    prep = fmt == "prep"
    f = 0 if prep else fmt
    assert route("prep" if prep else NAME[f], M, N, K, 128)[0] == "direct"
    assert route("prep" if prep else NAME[f], M, N, K, 128)[4] > 1
    p, want = exact_problem(f, M, K, N, 128)
    x, qw, sc, qz = (to_dev(v) for v in (p.x, p.qweight, p.scales, p.qzeros))
    out = torch.empty((M, N), dtype=torch.float16, device="cuda:0")
    w = P.prepare_layout(qw, sc, qz, fmt="gptq", group_size=128) if prep else None
    s = fresh_stream(torch)

    def call(xs, o):
        if prep:
            P.gemm_prepared(xs, w, out=o)
        else:
            P.gemm(xs, qw, sc, qz, fmt=NAME[f], group_size=128, out=o)
    if warm:
        with torch.cuda.stream(s):
            call(x[:warm], out[:warm])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(x, out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        check(torch, out, want, torch.float16)


BESIDE_A_CAPTURE = """
import sys
sys.path[:0] = [{root!r}, {tests!r}]
import torch
from helpers import pkg, to_dev
from test_gpu_direct import exact_problem
P = pkg()
p, want = exact_problem({fmt}, {M}, {K}, {N}, 128)
args = [to_dev(v) for v in (p.x, p.qweight, p.scales, p.qzeros)]
out = torch.zeros(({M}, {N}), dtype=torch.float16, device="cuda")
y = torch.zeros(16, device="cuda")
a, b = torch.cuda.Stream(), torch.cuda.Stream()
torch.cuda.synchronize()
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g, stream=a):
    y.add_(1)
    with torch.cuda.stream(b):
        P.gemm(*args, fmt={name!r}, out=out)
g.replay()
torch.cuda.synchronize()
assert torch.equal(out.cpu(), torch.from_numpy(want).to(torch.float16)) and y.eq(1).all()
print("both right")
"""


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,M,K,N", [(0, 48, 512, 512), (2, 33, 512, 1056)], ids=["small-batch", "direct"])
def test_first_call_beside_a_capture(torch_cuda, fmt, M, K, N):
    """The first call of a process, on the kernels that use neither scratch nor the workgroups'
    placement, allocates nothing: a capture on another stream, which an allocation would
    invalidate, goes on."""
    import os
    import subprocess
    import sys
    from helpers import ROOT
    assert fmt == 0 or route(NAME[fmt], M, N, K, 128) == ("direct", 3, 2, 2, 1)
    src = BESIDE_A_CAPTURE.format(root=ROOT, tests=os.path.join(ROOT, "tests"), fmt=fmt, M=M, K=K, N=N, name=NAME[fmt])
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "both right" in r.stdout, r.stderr[-1500:]
