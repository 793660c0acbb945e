"""Row kernels that share a row between waves, or split it over workgroups, when
rows are few: the same bits as the one-wave-per-row form of a long call (which
test_gpu_quant.py and test_gpu_nvfp4.py pin to the oracle)."""

import pytest
import torch

from vflash_amd import kernels

pytestmark = pytest.mark.gpu

ROWS = 4400  # past the row counts at which rows are shared or split


# Widths around the vector counts of one wave (512 elements), of four waves and
# of the 256-vector segments, and the widest row the register kernels hold.  (The
# E4M3 quantizer shares rows wider than 4096 in long calls too; there the
# requantizer, one wave per row, is the other side.)
@pytest.mark.parametrize("k", [512, 576, 2048, 2112, 4160, 8256, 14336, 16384])
def test_few_rows_match_many(dev, k):
    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randn((ROWS, k), generator=g, device=dev).to(torch.bfloat16)
    x[3, k - 1] = float("nan")
    x[4, k // 2] = float("-inf")
    x[6] = 0
    x[7] = 2.0**-100
    bits = lambda t: t.view(torch.uint8) if t.element_size() == 1 else t.view(torch.int32)
    gsf = torch.tensor(300.0, device=dev)
    codes, scales = kernels.quantize_rows(x)
    finite = x[5:]
    f_codes, _ = kernels.nvfp4_quantize_rows(finite, gsf)
    parts = x.abs().reshape(ROWS, k // 64, 64).amax(dim=2).float()  # NaN propagates, as the epilogue's
    r_codes, r_scales = kernels.requant_rows(x, parts)
    assert torch.equal(bits(r_codes), bits(codes)) and torch.equal(bits(r_scales), bits(scales))
    for m in (1, 17, 700, 2048):
        c, s = kernels.quantize_rows(x[:m])
        assert torch.equal(bits(c[:m]), bits(codes[:m])) and torch.equal(bits(s[:m]), bits(scales[:m])), m
        assert not c[m:].view(torch.uint8).any() and bool((s[m:] == 1).all())
        c, s = kernels.requant_rows(x[:m], parts[:m])
        assert torch.equal(bits(c[:m]), bits(codes[:m])) and torch.equal(bits(s[:m]), bits(scales[:m])), m
        assert not c[m:].view(torch.uint8).any() and bool((s[m:] == 1).all())
        c, s = kernels.nvfp4_quantize_rows(finite[:m], gsf)
        whole = kernels.nvfp4_quantize_rows(torch.cat([finite[:m], finite.new_zeros((ROWS, k))]), gsf)[1]
        tiles = (m + 127) // 128
        assert torch.equal(c, f_codes[:m]), m
        assert torch.equal(s.reshape(tiles, -1), whole.reshape(-1, s.numel() // tiles)[:tiles]), m


# 3000 rows take one wave a row on 256 CUs; 1, 17 and 700 four, 1500 two, and
# 4095 (two rounds of whole rows) two.
@pytest.mark.parametrize("k", [8, 520, 4104, 13824, 16384])
def test_gelu_rows_shared_between_waves(dev, k):
    g = torch.Generator(device=dev).manual_seed(k)
    y = (torch.randn((4095, k), generator=g, device=dev) * 2).to(torch.bfloat16)
    y[3, k - 1] = float("nan")
    y[4, k // 2] = float("inf")
    y[6] = 0
    bits = lambda t: t.contiguous().view(torch.uint8)
    codes, scales, values = kernels.gelu_quantize_rows(y[:3000], keep_values=True)
    for m in (1, 17, 700, 1500, 4095):
        c, s, v = kernels.gelu_quantize_rows(y[:m], keep_values=True)
        n = min(m, 3000)
        assert torch.equal(bits(c[:n]), bits(codes[:n])) and torch.equal(bits(s[:n]), bits(scales[:n])), m
        assert torch.equal(bits(v[:n]), bits(values[:n])), m
        assert not c[m:].view(torch.uint8).any() and bool((s[m:] == 1).all()), m
    c, s, v = kernels.gelu_quantize_rows(y[3000:], keep_values=True)
    whole = kernels.gelu_quantize_rows(y, keep_values=True)
    assert torch.equal(bits(whole[0][3000:4095]), bits(c[:1095])) and torch.equal(bits(whole[2][3000:]), bits(v))
