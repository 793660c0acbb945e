"""The adapter down-projection's block shapes give one result: calls large enough
for 2x4 and 4x4 blocks of 16 rows x 16 ranks equal 16-row calls (1x1 blocks) bit
for bit, and the fused codes equal the plain quantizer's."""

import pytest
import torch

from vflash_amd import kernels

pytestmark = pytest.mark.gpu


# On 256 CUs: 4100 rows of rank 48 and 100 take 2x4 blocks (partial row and rank
# groups), 4100 rows of rank 500 and 32761 of 48 take 4x4.  K = 80 leaves chunks
# empty, and every K here ends inside a 32-element step.
@pytest.mark.parametrize("m,rank,k", [(4100, 48, 272), (4100, 100, 80), (4100, 500, 80), (32761, 48, 1040)])
def test_blocks_agree_bit_for_bit(dev, m, rank, k):
    g = torch.Generator(device=dev).manual_seed(m + rank)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    x[m - 3, k - 1] = float("nan")
    x[5, 0] = float("inf")
    a = (torch.randn((rank, k), generator=g, device=dev) * 0.05).to(torch.bfloat16)
    t = kernels.lora_down(x, a)
    codes, scales, fused_t = kernels.quantize_rows_lora(x, a)
    plain_codes, plain_scales = kernels.quantize_rows(x)
    assert torch.equal(fused_t.view(torch.int16), t.view(torch.int16))
    assert torch.equal(codes.view(torch.uint8), plain_codes.view(torch.uint8))
    assert torch.equal(scales.view(torch.int32), plain_scales.view(torch.int32))
    for s in (0, 16, 2048, (m - 9) // 16 * 16):
        part = kernels.lora_down(x[s : s + 16], a)
        assert torch.equal(part.view(torch.int16), t[s : s + 16].view(torch.int16)), s
