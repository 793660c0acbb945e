"""The weight-only linear on gfx950: the GEMM that restores the weight in
registers, the restoring pass in front of a plain GEMM, and the calls that stay
with the torch expression."""

import pytest
import torch

from vflash_amd import kernels
from vflash_amd.fp8_linear import RowFP8Execution
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu


def operands(dev, m, k, n, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    codes, scale = quantize_weight_rows(torch.randn((n, k), generator=g, device=dev) * 0.02)
    return x, codes, scale, torch.randn(n, generator=g, device=dev).to(torch.bfloat16)


def check(out, x, codes, scale, bias):
    """One bf16 rounding (half a step: 2^-8 relative, eight significant bits) and a binary32 sum
    of K products in any order (K 2^-24 of the sum of magnitudes; 2^-23 leaves room
    for the accumulator's own alignment)."""
    w = (codes.float() * scale).to(torch.bfloat16).double()
    ref = x.double() @ w.T
    mag = x.double().abs() @ w.abs().T
    if bias is not None:
        ref, mag = ref + bias.double(), mag + bias.double().abs()
    err = (out.double() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + x.shape[1] * 2.0**-23 * mag).all())


# Partial tiles in rows and columns, K tails inside a 64-K stage, each tiling
# (64x64; 128x64 at 200 x 5128; 128x128 at 600 x 5128; 128x256 at 1000 x 7176)
# and the restoring pass (1025 rows).  K = 1296 is 21 stages, the last one partial:
# every slot of each ring (six slots below 128x128, else four) is refilled more than
# twice, and the loop over whole rings ends inside one.
@pytest.mark.parametrize("m,k,n", [(1, 16, 8), (17, 48, 272), (65, 144, 72), (200, 80, 5128),
                                   (600, 208, 5128), (1000, 272, 7176), (1025, 112, 136),
                                   (17, 1296, 272), (200, 1296, 5128), (600, 1296, 5128), (1000, 1296, 7176)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_weight_only_linear(dev, m, k, n, with_bias):
    x, codes, scale, bias = operands(dev, m, k, n, seed=m)
    bias = bias if with_bias else None
    with torch.no_grad():
        fused = kernels.weight_only_linear(x, codes, scale, bias)
        assert fused is not None
        out = RowFP8Execution().linear(x, codes, scale, bias)
    assert torch.equal(out, fused)
    check(out, x, codes, scale, bias)


def test_every_code_is_restored_as_torch_does(dev):
    # Identity activations read the restored weight back; NaN codes included.
    k = 256
    codes = torch.arange(256, device=dev, dtype=torch.uint8).repeat(16, 1).view(torch.float8_e4m3fn)
    scale = torch.logspace(-30, 30, 16, base=2.0, device=dev).reshape(16, 1) * 1.337
    want = (codes.float() * scale).to(torch.bfloat16)
    from vflash_amd._lib import call, ptr, stream_of

    got = torch.empty((16, k), device=dev, dtype=torch.bfloat16)
    call("vflash_restore_rows_bf16", ptr(codes), ptr(scale), k, 16, k, ptr(got), stream_of(dev))
    assert torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    finite = torch.isfinite(want).all(dim=0).to(torch.bfloat16)  # columns without a NaN code
    codes = torch.where(finite.bool(), codes.view(torch.uint8), 0).view(torch.float8_e4m3fn)
    out = kernels.weight_only_linear(torch.eye(k, device=dev, dtype=torch.bfloat16), codes, scale)
    assert torch.equal(out, (codes.float() * scale).to(torch.bfloat16).T)


def test_layouts_and_recorded_calls(dev):
    x, codes, scale, bias = operands(dev, 24, 80, 40)
    ex = RowFP8Execution()
    want = ex.linear(x, codes, scale, bias)
    assert torch.equal(ex.linear(x.reshape(2, 3, 4, 80), codes, scale, bias).reshape(24, 40), want)
    assert torch.equal(ex.linear(x[5], codes, scale, bias), want[5])
    strided = torch.zeros((24, 96), device=dev, dtype=torch.bfloat16)
    strided[:, :80] = x
    strided[:, 80:] = float("nan")
    assert torch.equal(ex.linear(strided[:, :80], codes, scale, bias), want)
    # Outside the kernel's forms: the torch expression, with its own rounding order.
    flat = torch.zeros(24 * 80 + 1, device=dev, dtype=torch.bfloat16)
    flat[1:] = x.reshape(-1)
    unaligned = flat[1:].reshape(24, 80)
    assert kernels.weight_only_linear(unaligned, codes, scale, bias) is None
    check(ex.linear(unaligned, codes, scale, bias), x, codes, scale, bias)
    tracked = x.clone().requires_grad_()
    assert kernels.weight_only_linear(tracked, codes, scale, bias) is None
    ex.linear(tracked, codes, scale, bias).sum().backward()
    w = (codes.float() * scale).to(torch.bfloat16)
    assert torch.allclose(tracked.grad.float(), w.float().sum(0).expand(24, 80), rtol=2.0**-6, atol=1e-3)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        tangent = torch.autograd.forward_ad.unpack_dual(ex.linear(dual, codes, scale, bias)).tangent
    assert tangent is not None
    # Without a bias, which torch's batched form adds after rounding the product.
    batched = torch.vmap(lambda v: ex.linear(v, codes, scale))(x.reshape(4, 6, 80))
    check(batched.reshape(24, 40), x, codes, scale, None)


def test_infinite_scale_and_k_tail(dev):
    # K = 80 leaves 48 zero-filled positions in the last stage: an infinite scale
    # must not turn them into NaN.
    x, codes, scale, _ = operands(dev, 20, 80, 24)
    x = x.abs() + 1
    codes = torch.full((24, 80), 0x38, device=dev, dtype=torch.uint8).view(torch.float8_e4m3fn)  # 1.0
    scale[3] = float("inf")
    out = RowFP8Execution().linear(x, codes, scale)
    assert bool(torch.isinf(out[:, 3]).all()) and bool((out[:, 3] > 0).all())
    assert bool(torch.isfinite(out[:, [i for i in range(24) if i != 3]]).all())


@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
def test_compiled_calls_are_one_graph_of_the_expression(dev, backend):
    x, codes, scale, bias = operands(dev, 24, 80, 40)
    ex = RowFP8Execution()
    want = torch.nn.functional.linear(x, (codes.float() * scale).to(torch.bfloat16), bias)
    with torch.no_grad():
        assert torch.equal(torch.compile(lambda v: ex.linear(v, codes, scale, bias), backend=backend,
                                         fullgraph=True)(x), want)
