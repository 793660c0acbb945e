"""SwiGLU calls whose 256x256 tiles run partly, or all, as 64x256 tiles: the same
activation and row maxima, bit for bit, as whole tiles give."""

import pytest
import torch

from vflash_amd import kernels
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu


# On 256 CUs 8192 rows of F = 1024 are one full round of 256x256 tiles, never
# split; 8969 rows are that round and 32 tiles more, split (the last tile row
# holds 9 rows), and the short calls are split entirely.  K 128 is one stage, 640
# runs past the ring; K = 208 (not a multiple of 128) is never split.
@pytest.mark.parametrize("k", [128, 640, 208])
def test_split_tiles_agree_bit_for_bit(dev, k):
    f, whole_rows, rows = 1024, 8192, 8969
    g = torch.Generator(device=dev).manual_seed(k)
    x = torch.randn((rows, k), generator=g, device=dev).to(torch.bfloat16)
    codes, sa = kernels.quantize_rows(x)
    w, sw = quantize_weight_rows(torch.randn((2 * f, k), generator=g, device=dev) * 0.05)
    bias = torch.randn(2 * f, generator=g, device=dev).to(torch.bfloat16)
    h, amax = kernels.fp8_gemm_swiglu(codes, sa, w, sw, rows, bias)
    whole_h, whole_amax = kernels.fp8_gemm_swiglu(codes[:whole_rows], sa[:whole_rows], w, sw, whole_rows, bias)
    assert torch.equal(h[:whole_rows], whole_h) and torch.equal(amax[:whole_rows], whole_amax)
    # The tail of the long call as rows of another whole round.
    last_h, last_amax = kernels.fp8_gemm_swiglu(codes[rows - whole_rows : rows], sa[rows - whole_rows : rows], w,
                                                sw, whole_rows, bias)
    assert torch.equal(h[rows - whole_rows :], last_h) and torch.equal(amax[rows - whole_rows :], last_amax)
    for m in (1, 9, 64, 65, 100, 200, 300):
        part_h, part_amax = kernels.fp8_gemm_swiglu(codes[:m], sa[:m], w, sw, m, bias)
        assert torch.equal(part_h, whole_h[:m]) and torch.equal(part_amax, whole_amax[:m]), m
