"""What happens when a built part of the package is absent or older, checked on the CPU:
the device and launch checks are answered as a gfx950 device would, and the calls
must not get as far as a launch."""

import subprocess
import sys

import pytest
import torch

import vflash_amd
from vflash_amd import _lib, build, fp8_linear, fused, kernels
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


def test_weight_only_on_a_torch_that_does_not_name_its_modes(monkeypatch, gfx950):
    monkeypatch.delattr(torch._C, "_len_torch_dispatch_stack")
    monkeypatch.setattr(kernels, "_modes_active", kernels._mode_probe())
    monkeypatch.setattr(kernels, "call", lambda *args: pytest.fail("launched"))
    x, w, s, b = operands()
    want = torch.nn.functional.linear(x, (w.float() * s).to(torch.bfloat16), b)
    with torch.no_grad():
        assert torch.equal(RowFP8Execution().linear(x, w, s, b), want)


@pytest.fixture
def no_host(monkeypatch, fresh):
    """_host.so does not import, as under another Python or torch."""
    monkeypatch.setitem(sys.modules, "vflash_amd._host", None)
    monkeypatch.delattr(vflash_amd, "_host", raising=False)


def test_w8a8_without_the_host_module(monkeypatch, gfx950, no_host):
    x, w, s, b = operands()
    down, up = torch.zeros((8, 32), dtype=torch.bfloat16), torch.zeros((16, 8), dtype=torch.bfloat16)
    launched = []
    monkeypatch.setattr(kernels, "call", lambda name, *args: launched.append(name))
    for module in (fp8_linear, fused):
        monkeypatch.setattr(module, "takes_native_path", lambda execution, value: True)
    ex = RowFP8Execution("w8a8", activation_quantizer="hip")
    with pytest.warns(RuntimeWarning, match="native host path is off"):
        assert ex.linear(x, w, s, b).shape == (5, 16)
    assert fused.fp8_linear_lora(ex, x, w, s, b, down, up).shape == (5, 16)
    assert launched == ["vflash_quantize_rows_e4m3", "vflash_fp8_linear", "vflash_quantize_rows_lora_e4m3",
                        "vflash_fp8_linear_lora"]
    assert ex.calls == {"weight_only": 0, "w8a8": 2}


@pytest.mark.parametrize("absent", ["torch", "torch headers", "Python headers"])
def test_build_without_what_only_the_host_module_needs(monkeypatch, tmp_path, capsys, absent):
    stale = tmp_path / "_host.so"
    stale.write_bytes(b"of another build")
    monkeypatch.setattr(build, "HOST_MODULE", stale)
    monkeypatch.setattr(build.subprocess, "run", lambda *a, **k: pytest.fail("nothing to compile"))
    if absent == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)
    elif absent == "torch headers":
        from torch.utils import cpp_extension

        monkeypatch.setattr(cpp_extension, "include_paths", lambda *a, **k: [str(tmp_path)])
    else:
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build_host() is None
    assert "not built" in capsys.readouterr().err and not stale.exists()


# An older library: one whose argument lists differ, one of the same version that
# lacks entries added since, and a library of something else.
@pytest.mark.parametrize("source,message", [
    ("int vflash_abi_version(void) { return 3; }", "unexpected ABI version"),
    ("int vflash_abi_version(void) { return 4; } int vflash_status_string; int vflash_quantize_rows_e4m3;",
     "older than this package"),
    ("int other;", "unexpected ABI version"),
])
def test_older_library_is_named(monkeypatch, tmp_path, fresh, source, message):
    (tmp_path / "old.c").write_text(source)
    old = tmp_path / "libvflash_amd.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(tmp_path / "old.c"), "-o", str(old)], check=True)
    monkeypatch.setattr(_lib, "LIBRARY", old)
    with pytest.raises(RuntimeError, match=message):
        _lib.library()
