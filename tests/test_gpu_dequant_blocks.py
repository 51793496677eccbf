"""Standalone dequantisation in 8 x 8 blocks (csrc/kernels_strided.hip, dequant_block_kernel) at the
sizes where it can go wrong: one block, remainders of a wave's and a workgroup's blocks in either
direction, groups of 8 rows and of all rows; and the per-word kernel that takes what the blocks do
not (group indexes, tensors off 16 bytes). Bit for bit against the oracle."""
import numpy as np
import pytest

from helpers import pkg, to_dev
from synth import Problem

pytestmark = pytest.mark.gpu
NAME = {0: "gptq", 1: "gptq_sym", 2: "awq"}


@pytest.fixture(scope="module")
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("K,N,G", [(8, 8, 8), (24, 40, 24), (264, 520, 88), (2048, 264, 64), (256, 2056, 256)])
def test_dequant_blocks(torch_cuda, orc, fmt, K, N, G, transposed):
    p = Problem(fmt, M=1, K=K, N=N, G=G, seed=K + N)
    out = pkg().dequant(to_dev(p.qweight), to_dev(p.scales), None if fmt == 1 else to_dev(p.qzeros),
                        fmt=NAME[fmt], group_size=G, transposed=transposed)
    torch_cuda.cuda.synchronize()
    want = orc.dequant(fmt, p.qweight, p.scales, p.qzeros, K, N, G, transposed=transposed)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("fmt", [0, 2])
def test_dequant_off_16_bytes(torch_cuda, orc, fmt):
    """Packed words and scales that start off 16 bytes: the same weights from the per-word kernel."""
    p = Problem(fmt, M=1, K=128, N=72, G=32, seed=5)

    def off(a):
        t = to_dev(a)
        buf = torch_cuda.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        buf[1:] = t.flatten()
        return buf[1:].view(t.shape)
    out = pkg().dequant(off(p.qweight), off(p.scales), to_dev(p.qzeros), fmt=NAME[fmt], group_size=32,
                        transposed=True)
    torch_cuda.cuda.synchronize()
    want = orc.dequant(fmt, p.qweight, p.scales, p.qzeros, 128, 72, 32, transposed=True)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), want.view(np.uint16))
