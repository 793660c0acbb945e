"""The NVFP4 GEMM's tilings give one result: row slices that take the smaller
tiles equal the same rows of a call on 256x256 tiles, bit for bit (the oracle
comparison of each arithmetic is in test_gpu_nvfp4.py)."""

import pytest
import torch

from vflash_amd import kernels
from vflash_amd.prepare import quantize_nvfp4_weight

pytestmark = pytest.mark.gpu


# N = 1152 ends inside a 256-column tile and puts every other 64-column tile in
# the upper half of its 128-row scale tile.  On 256 CUs 8192 rows take 256x256;
# 17 rows 64x64, 1000 64x128, 2047 128x128 and 4001 256x128.  K = 320 ends inside
# a 128-K stage, 64 is half a stage, 640 runs past the deepest ring.
@pytest.mark.parametrize("k", [64, 320, 640])
@pytest.mark.parametrize("activations", ["nvfp4", "e4m3"])
def test_tilings_agree_bit_for_bit(dev, k, activations):
    n, whole_rows = 1152, 8192
    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randn((whole_rows, k), generator=g, device=dev).to(torch.bfloat16)
    packed, scales, alpha, input_scale = quantize_nvfp4_weight(
        torch.randn((n, k), generator=g, device=dev) * 0.02, input_scale=400.0)
    bias = torch.randn(n, generator=g, device=dev).to(torch.bfloat16)

    def linear(rows):
        if activations == "nvfp4":
            codes, s = kernels.nvfp4_quantize_rows(rows, input_scale)
            return kernels.nvfp4_w4a4_gemm(codes, s, packed, scales, alpha, rows.shape[0], bias)
        codes, s = kernels.quantize_rows(rows)
        return kernels.nvfp4_gemm(codes, s, packed, scales, alpha, rows.shape[0], bias)

    whole = linear(x)
    for m in (1, 17, 65, 300, 1000, 2047, 4001):
        assert torch.equal(linear(x[:m]), whole[:m]), m


@pytest.mark.parametrize("m,k", [(1, 64), (300, 512)])
def test_output_scale_of_the_quantizer_is_the_device_division(dev, m, k):
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    for a, b in ((0.0123, 487.3), (3.0, 0.1), (1e-38, 3e5), (float("inf"), 2.0)):
        alpha, gsf = torch.tensor(a, device=dev), torch.tensor(b, device=dev)
        codes, scales, out_scale = kernels.nvfp4_quantize_rows(x, gsf, alpha)
        plain_codes, plain_scales = kernels.nvfp4_quantize_rows(x, gsf)
        assert torch.equal(out_scale, alpha / gsf)
        assert torch.equal(codes, plain_codes) and torch.equal(scales, plain_scales)
