"""256x256 grids whose last round is split into smaller tiles: bit-identical to
calls on 1024-row slices, which are not."""

import pytest
import torch

from vflash_amd import kernels
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu


def operands(dev, m, k, n):
    g = torch.Generator(device=dev).manual_seed(m + n)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    codes, sa = kernels.quantize_rows(x)
    w, sw = quantize_weight_rows(torch.randn((n, k), generator=g, device=dev) * 0.02)
    return g, x, codes, sa, w, sw, torch.randn(n, generator=g, device=dev).to(torch.bfloat16)


# On 256 CUs: 33 x 25 tiles (three rounds and 57 tiles, as 256x128; both edges
# partial, the last row of tiles within its upper half) and 16 x 20 (one round and
# 64 tiles, as 128x128).  K 128 is one stage, 640 runs past every ring.
@pytest.mark.parametrize("m,n", [(32 * 256 + 77, 24 * 256 + 144), (4095, 5120)])
@pytest.mark.parametrize("k", [128, 640])
def test_split_last_round(dev, m, n, k):
    g, _, codes, sa, w, sw, bias = operands(dev, m, k, n)
    whole = kernels.fp8_gemm(codes, sa, w, sw, m, bias)
    residual = torch.randn((m, n), generator=g, device=dev).to(torch.bfloat16)
    gate = torch.rand((m, n), generator=g, device=dev).to(torch.bfloat16)
    gated = kernels.fp8_gemm_gate_residual(codes, sa, w, sw, m, gate, residual, bias)
    for s in range(0, m, 1024):
        e = min(s + 1024, m)
        part = kernels.fp8_gemm(codes[s:e], sa[s:e], w, sw, e - s, bias)
        assert torch.equal(part, whole[s:e]), s
        part = kernels.fp8_gemm_gate_residual(codes[s:e], sa[s:e], w, sw, e - s, gate[s:e], residual[s:e], bias)
        assert torch.equal(part, gated[s:e]), s
