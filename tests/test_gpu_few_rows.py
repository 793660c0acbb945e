"""The few-row E4M3 GEMM (one 32-column block per workgroup): the same bits as the
rows of a call on the tiled kernel, under each epilogue that it serves."""

import pytest
import torch

from vflash_amd import kernels
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu


# On 256 CUs 2000 rows (9000 at 48 columns) are tiled; 1 and 17 rows take 32-row
# workgroups at every width, 40 and 64 rows 32-row ones at 48 and 1008 columns and
# 64-row ones at 5136.  300 rows are ten 32-row workgroups high at 48 columns and five
# 64-row ones at 1008 (128x64 tiles at 5136).  Widths end inside a 32-column block; K 16 and 144 end
# inside a stage, 1280 runs past the ring.
@pytest.mark.parametrize("k", [16, 144, 1280])
@pytest.mark.parametrize("n", [48, 1008, 5136])
def test_few_rows_match_the_tiled_kernel(dev, k, n):
    whole = 9000 if n == 48 else 2000
    g = torch.Generator(device=dev).manual_seed(k + n)
    x = torch.randn((whole, k), generator=g, device=dev).to(torch.bfloat16)
    codes, sa = kernels.quantize_rows(x)
    w, sw = quantize_weight_rows(torch.randn((n, k), generator=g, device=dev) * 0.05)
    bias = torch.randn(n, generator=g, device=dev).to(torch.bfloat16)
    residual = torch.randn((whole, n), generator=g, device=dev).to(torch.bfloat16)
    gate = torch.rand((whole, n), generator=g, device=dev).to(torch.bfloat16)
    rank = 24
    t = kernels.lora_down(x, (torch.randn((rank, k), generator=g, device=dev) * 0.1).to(torch.bfloat16))
    up = (torch.randn((n, rank), generator=g, device=dev) * 0.1).to(torch.bfloat16)

    def calls(m):
        c, s, r, gt, tt = codes[:m], sa[:m], residual[:m], gate[:m], t[:m]
        lora = kernels.LoraOperands(tt, up, 0.5)
        yield kernels.fp8_gemm(c, s, w, sw, m, bias)
        yield kernels.fp8_gemm(c, s, w, sw, m)
        yield kernels.fp8_gemm_planes(c, s, w, sw, m, 3, bias).transpose(0, 1)
        yield kernels.fp8_gemm_gate_residual(c, s, w, sw, m, gt, r, bias)
        yield kernels.fp8_gemm_lora(c, s, w, sw, m, tt, up, scale=0.5, bias=bias)
        yield kernels.fp8_gemm_gate_residual(c, s, w, sw, m, gt, r, bias, lora=lora)

    expected = list(calls(whole))
    for m in (1, 17, 40, 64, 300):
        for i, got in enumerate(calls(m)):
            assert torch.equal(got, expected[i][:m]), (m, i)
