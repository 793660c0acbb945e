"""What still works when a built part of the package is absent, checked on the CPU:
the device and launch checks are answered as a gfx950 device would, and the calls
must not get as far as a launch."""

import pytest
import torch

from vflash_amd import _lib, kernels
from vflash_amd.fp8_linear import RowFP8Execution
from vflash_amd.prepare import quantize_weight_rows


@pytest.fixture
def gfx950(monkeypatch):
    """CPU tensors pass for tensors on the current gfx950 device."""
    monkeypatch.setattr(_lib, "is_gfx950", lambda device: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(kernels, "stream_of", lambda device: 0)


@pytest.fixture
def fresh():
    """The loaders look again, in the test and after it."""
    loaders = [f for f in (_lib.library, getattr(_lib, "available", None), _lib.host) if f is not None]
    for f in loaders:
        f.cache_clear()
    yield
    for f in loaders:
        f.cache_clear()


def operands(m=5, k=32, n=16):
    g = torch.Generator().manual_seed(m)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    w, s = quantize_weight_rows(torch.randn((n, k), generator=g) * 0.02)
    return x, w, s, torch.randn(n, generator=g).to(torch.bfloat16)


def test_weight_only_without_the_library(monkeypatch, tmp_path, gfx950, fresh):
    x, w, s, b = operands()
    monkeypatch.setattr(_lib, "LIBRARY", tmp_path / "libvflash_amd.so")
    want = torch.nn.functional.linear(x, (w.float() * s).to(torch.bfloat16), b)
    with torch.no_grad():
        with pytest.warns(RuntimeWarning, match="not built"):
            assert torch.equal(RowFP8Execution().linear(x, w, s, b), want)
        assert torch.equal(RowFP8Execution().linear(x, w, s, b), want)
    with pytest.raises(RuntimeError, match="not built"):
        RowFP8Execution("w8a8", activation_quantizer="hip").linear(x, w, s, b)
