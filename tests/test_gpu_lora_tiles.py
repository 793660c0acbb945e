"""256x192 tiles of a merged projection whose tiles and waves straddle adapter
branches: bit-identical to each branch by itself, on another tiling."""

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


# Three branches of 7168 (not a multiple of the 96 columns of a 256x192 wave) on
# 1000 rows; each branch alone is a plain adapter call on another tiling.
@pytest.mark.parametrize("rank", [16, 100])
def test_branches_inside_a_wave(dev, rank):
    m, k, inner = 1000, 256, 7168
    g, x, codes, sa, w, sw, bias = operands(dev, m, k, 3 * inner)
    width = -(-rank // 16) * 16
    down = torch.zeros((3 * width, k), device=dev, dtype=torch.bfloat16)
    for b in range(3):
        down[b * width : b * width + rank] = (torch.randn((rank, k), generator=g, device=dev) * 0.1).to(torch.bfloat16)
    up = torch.zeros((3 * inner, -(-rank // 8) * 8), device=dev, dtype=torch.bfloat16)
    up[:, :rank] = (torch.randn((3 * inner, rank), generator=g, device=dev) * 0.1).to(torch.bfloat16)
    up = up[:, :rank]
    t = kernels.lora_down(x, down)
    scales = (1.0, 0.5, 0.3)
    out = kernels.fp8_gemm_lora_branches(codes, sa, w, sw, m, t, width, up, rank, scales, bias=bias)
    planes = kernels.fp8_gemm_lora_branches(codes, sa, w, sw, m, t, width, up, rank, scales, bias=bias, planes=3)
    for b in range(3):
        c = slice(b * inner, (b + 1) * inner)
        one = kernels.fp8_gemm_lora(codes, sa, w[c], sw[c], m, t[:, b * width : b * width + rank].contiguous(),
                                    up[c], scale=scales[b], bias=bias[c])
        assert torch.equal(out[:, c], one), b
        assert torch.equal(planes[b], one), b
