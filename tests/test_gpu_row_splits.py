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


def test_rows_past_one_grid_dimension(dev):
    # A workgroup per row: rows past 2^22 start in the grid's second dimension, and
    # the last workgroups of that one lie past the end.
    from vflash_amd._lib import call, ptr, stream_of

    n, k = 2**22 + 5, 16
    g = torch.Generator(device=dev).manual_seed(0)
    codes = torch.randint(0, 127, (n, k), generator=g, device=dev, dtype=torch.uint8).view(torch.float8_e4m3fn)
    scale = torch.rand((n, 1), generator=g, device=dev)
    out = torch.zeros((n + 3, k), device=dev, dtype=torch.bfloat16)
    call("vflash_restore_rows_bf16", ptr(codes), ptr(scale), k, n, k, ptr(out), stream_of(dev))
    assert torch.equal(out[:n], (codes.float() * scale).to(torch.bfloat16)) and not out[n:].any()
    k = 4104  # 34 GB of rows, of which the first and the last few are not zero
    x = torch.zeros((n, k), device=dev, dtype=torch.bfloat16)
    ends = torch.cat([torch.arange(3), torch.arange(n - 9, n)]).to(dev)
    x[ends] = torch.randn((12, k), generator=g, device=dev).to(torch.bfloat16)
    codes, scales = kernels.quantize_rows(x)
    few_codes, few_scales = kernels.quantize_rows(x[ends])
    assert torch.equal(codes[ends].view(torch.uint8), few_codes[:12].view(torch.uint8))
    assert torch.equal(scales[ends], few_scales[:12]) and bool((scales[3:n - 9] == 1).all())
    assert not codes[n:].view(torch.uint8).any() and bool((scales[n:] == 1).all())
    del x, codes
    torch.cuda.empty_cache()
