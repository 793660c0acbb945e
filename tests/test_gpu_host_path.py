"""The native host path of the W8A8 linear and of the adapter linear against the
Python wrappers (which an execution with a ``measure`` scope takes): the same
bits where it applies, the same results and errors where it does not."""

from contextlib import nullcontext

import pytest
import torch

from vflash_amd import _lib, fused
from vflash_amd.fp8_linear import RowFP8Execution
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu


def executions():
    return (RowFP8Execution("w8a8", activation_quantizer="hip"),
            RowFP8Execution("w8a8", activation_quantizer="hip", measure=lambda _: nullcontext()))


def operands(dev, m, k, n, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    w, s = quantize_weight_rows(torch.randn((n, k), generator=g, device=dev) * 0.02)
    return g, x, w, s, torch.randn(n, generator=g, device=dev).to(torch.bfloat16)


def forms(x):
    """The rows of x as callers hold them: matrix, vector, batch, and layouts that
    the wrappers copy or read with strides."""
    m, k = x.shape
    wide = torch.zeros((m, k + 16), device=x.device, dtype=x.dtype)
    wide[:, :k] = x
    odd = torch.zeros(m * k + 1, device=x.device, dtype=x.dtype)
    odd[1:] = x.reshape(-1)
    return {"matrix": x, "vector": x[0], "batch": x.reshape(1, m, k), "strided": wide[:, :k],
            "unaligned": odd[1:].reshape(m, k),
            "parameter": torch.nn.Parameter(x, requires_grad=False)}


@pytest.mark.parametrize("m,k,n", [(1, 16, 16), (17, 272, 48), (300, 384, 4112)])
@pytest.mark.parametrize("with_bias", [True, False])
def test_linear(dev, m, k, n, with_bias):
    _, x, w, s, b = operands(dev, m, k, n, seed=m)
    native, python = executions()
    bias = b if with_bias else None
    assert _lib.host().w8a8_linear(x, w, s, bias) is not None
    for name, v in forms(x).items():
        got, want = native.linear(v, w, s, bias), python.linear(v, w, s, bias)
        assert got.shape == want.shape and got.stride() == want.stride() and torch.equal(got, want), name
    assert native.calls == python.calls == {"weight_only": 0, "w8a8": 6}


@pytest.mark.parametrize("m,k,n,rank", [(17, 272, 48, 8), (40, 1536, 144, 20), (300, 128, 4112, 128)])
def test_adapter_linear(dev, m, k, n, rank):
    g, x, w, s, b = operands(dev, m, k, n, seed=n)
    down = (torch.randn((rank, k), generator=g, device=dev) * 0.1).to(torch.bfloat16)
    up = (torch.randn((n, rank), generator=g, device=dev) * 0.1).to(torch.bfloat16)
    native, python = executions()
    taken = _lib.host().w8a8_linear_lora(x, w, s, b, down, up, 0.5, 1.375)
    assert (taken is None) == (rank % 8 != 0)
    for name, v in forms(x).items():
        if name == "unaligned":
            continue  # refused by the fused quantizer on either path
        got = fused.fp8_linear_lora(native, v, w, s, b, down, up, scaling=0.5, strength=1.375)
        want = fused.fp8_linear_lora(python, v, w, s, b, down, up, scaling=0.5, strength=1.375)
        assert got.shape == want.shape and torch.equal(got, want), name
    assert native.calls == python.calls
    with pytest.raises(ValueError):
        fused.fp8_linear_lora(native, x, w, s, b, down[:, :-16].contiguous(), up)
    with pytest.raises(ValueError):
        fused.fp8_linear_lora(native, x, w, s, b, down.float(), up)


def test_refusals_are_the_wrappers(dev):
    _, x, w, s, b = operands(dev, 8, 32, 32)
    native, python = executions()
    for bad in ((x.float(), w, s, b.float()), (x[:, :16], w, s, b), (x, w, s.double(), b), (x, w, s[:16], b),
                (x, w, s, b[:16]), (x, w.float(), s, b), (x, w, s.cpu(), b), (x.t().contiguous().t(), w, s, b)):
        for ex in (native, python):
            with pytest.raises(ValueError):
                ex.linear(*bad)
    assert native.calls == python.calls
    assert native.linear(x[:0], w, s, b).shape == (0, 32)
    seen = []
    observed, _ = executions()
    observed.observer = lambda: seen.append(dict(observed.calls))
    observed.linear(x, w, s, b)
    assert seen == [{"weight_only": 0, "w8a8": 0}]


def test_capture_and_streams(dev):
    _, x, w, s, b = operands(dev, 17, 256, 64)
    native, python = executions()
    want = python.linear(x, w, s, b)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        on_side = native.linear(x, w, s, b)
    side.synchronize()
    assert torch.equal(on_side, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = native.linear(x, w, s, b)
    for step in range(3):
        x.add_(1)
        eager = python.linear(x, w, s, b)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), step
