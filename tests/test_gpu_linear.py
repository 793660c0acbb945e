"""W8A8 linear on gfx950 against the oracle (bf16 outputs within 1e-2 relative)."""

import numpy as np
import pytest
import torch

from oracle import fp8 as O
from oracle import fp8_torch as T
from tests.conftest import golden, rel_check, rel_check_device
from vflash_amd import kernels
from vflash_amd.fp8_linear import RowFP8Execution, RowFP8Linear
from vflash_amd.prepare import quantize_weight_rows

pytestmark = pytest.mark.gpu



def tiling(m, n):
    """The GEMM tiling the library picks for an M x N output on 256 CUs (the
    library's own rule, vflash_fp8_gemm_tiling)."""
    return kernels.gemm_tiling(m, n)


# Edge shapes under each tiling: partial row and column tiles, K tails
# (K % 128 != 0 takes the vector-offset DMA everywhere), one K stage.  The first four
# run the few-row kernel, which serves shapes of at most 256 of its workgroups whatever
# the query answers; test_launched_kernels_cpu.py pins what each entry here launches.
EDGES = [
    (1, 16, 16, "64x64"), (17, 48, 272, "64x64"), (300, 144, 48, "64x64"),
    (257, 256, 528, "64x64"),
    (1, 16, 8208, "64x64"), (17, 144, 8208, "64x64"), (65, 256, 4112, "64x64"),
    (257, 48, 2064, "64x64"), (300, 1296, 2064, "64x64"),
    (257, 144, 4112, "128x64"), (300, 256, 4112, "128x64"),
    (520, 144, 4112, "128x128 one round"), (300, 256, 7184, "128x128 one round"),
    (600, 144, 11008, "128x128"), (2100, 256, 3712, "128x128"),
    (257, 144, 13840, "128x192"), (700, 256, 6032, "128x192"),
    (1040, 48, 6160, "256x128"), (1100, 256, 6032, "256x128"),
    (1040, 144, 7184, "256x192"), (1100, 256, 8208, "256x192"),
    (4100, 144, 3088, "256x256"), (4100, 256, 3088, "256x256"), (4097, 128, 3072, "256x256"),
]


def seeded(m, k, n, bias=True, seed=0):
    """The benchmark input recipe: fp32 draws on CPU in the order X, W, bias, then casts."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((m, k), generator=g).to(torch.bfloat16)
    w = torch.randn((n, k), generator=g) * 0.02
    b = (torch.randn(n, generator=g) * 0.01).to(torch.bfloat16) if bias else None
    codes, scale = quantize_weight_rows(w)
    return x, codes, scale, b


def oracle_linear(x, codes, scale, b, rows=None, scalar_product=False):
    xs = x.float().numpy() if rows is None else x.float().numpy()[rows]
    return O.w8a8_linear(
        xs,
        codes.view(torch.uint8).numpy(),
        scale.reshape(-1).numpy(),
        None if b is None else b.float().numpy(),
        scalar_product=scalar_product,
    )


def test_golden_small_case_through_the_c_abi(dev):
    g = golden("gemm_small.npz")
    m = g["x"].shape[0]
    a = torch.from_numpy(g["a_codes"]).view(torch.float8_e4m3fn).to(dev)
    sa = torch.from_numpy(g["sa"]).to(dev)
    w = torch.from_numpy(g["w_codes"]).view(torch.float8_e4m3fn).to(dev)
    sw = torch.from_numpy(g["sw"]).to(dev)
    bias = torch.from_numpy(g["bias"]).to(torch.bfloat16).to(dev)
    out = kernels.fp8_gemm(a, sa, w, sw, m, bias).float().cpu().numpy()
    _, exact = rel_check(out, g["expected"])
    assert exact > 0.95  # the exact-sum reference differs only by rare ties of fp32 sums
    nob = kernels.fp8_gemm(a, sa, w, sw, m).float().cpu().numpy()
    rel_check(nob, g["scaled"])


def test_small_linear_4096x3072x3072(dev):
    # X bf16 [4096, 3072] N(0,1); W N(0, 0.02) -> e4m3 [3072, 3072]; bias N(0, 0.01); seed 0.
    x, codes, scale, b = seeded(4096, 3072, 3072)
    ex = RowFP8Execution("w8a8", activation_quantizer="triton")
    out = ex.linear(x.to(dev), codes.to(dev), scale.to(dev), b.to(dev))
    assert out.dtype == torch.bfloat16 and out.shape == (4096, 3072)
    worst, exact = rel_check(out.float().cpu().numpy(), oracle_linear(x, codes, scale, b))
    assert exact > 0.9
    assert ex.calls == {"weight_only": 0, "w8a8": 1}


@pytest.mark.parametrize("m,k,n,tiles", EDGES)
def test_edges_under_every_tiling(dev, m, k, n, tiles):
    assert tiling(m, n) == tiles
    x, codes, scale, b = seeded(m, k, n, seed=m + k + n)
    codes_d, scale_d = codes.to(dev), scale.to(dev)
    a, sa = kernels.quantize_rows(x.to(dev))
    rows = np.r_[0:8, m // 2:m // 2 + 8, max(m - 24, 0):m] if m > 512 else None
    out = kernels.fp8_gemm(a, sa, codes_d, scale_d, m, b.to(dev))
    got = out.float().cpu().numpy()
    rel_check(got if rows is None else got[rows], oracle_linear(x, codes, scale, b, rows))
    out = kernels.fp8_gemm(a, sa, codes_d, scale_d, m, None)
    got = out.float().cpu().numpy()
    rel_check(got if rows is None else got[rows], oracle_linear(x, codes, scale, None, rows))
    # The gate-residual epilogue under the same tiling (one K stage, K tails, partial
    # tiles), on the kernel's own projection: bf16(residual + bf16(gate * y)) exactly.
    g = torch.Generator().manual_seed(m + n)
    gate = torch.rand(n, generator=g).to(torch.bfloat16).to(dev)
    res = torch.randn((m, n), generator=g).to(torch.bfloat16).to(dev)
    y = kernels.fp8_gemm(a, sa, codes_d, scale_d, m, b.to(dev))
    gated = kernels.fp8_gemm_gate_residual(a, sa, codes_d, scale_d, m, gate, res, b.to(dev))
    want = T.gate_residual(res, gate.reshape(1, n).expand(m, n), y).to(torch.bfloat16)
    assert torch.equal(gated, want)


def test_three_dimensional_input_and_torch_quantizer(dev):
    x, codes, scale, b = seeded(2 * 3 * 40, 256, 64)
    x3 = x.reshape(2, 120, 256)
    ex = RowFP8Execution("w8a8", activation_quantizer="torch")
    out = ex.linear(x3.to(dev), codes.to(dev), scale.to(dev), b.to(dev))
    assert out.shape == (2, 120, 64)
    # The portable quantizer is torch's expression on this device: amax / 448.0
    # is a product with RN(1/448) in torch's GPU kernels.
    rel_check(out.reshape(-1, 64).float().cpu().numpy(),
              oracle_linear(x, codes, scale, b, scalar_product=True))


def test_module_forward_and_measure_scopes(dev):
    x, codes, scale, b = seeded(64, 128, 32)
    scopes = []

    class Scope:
        def __init__(self, name):
            self.name = name

        def __enter__(self):
            scopes.append(self.name)

        def __exit__(self, *exc):
            return False

    ex = RowFP8Execution("w8a8", activation_quantizer="triton", measure=Scope)
    original = torch.nn.Linear(128, 32, dtype=torch.bfloat16)
    original.bias.data.copy_(b)
    module = RowFP8Linear(original, ex)
    module.load_state_dict(
        {"weight": codes.to(dev), "row_scale": scale.to(dev), "bias": original.bias.to(dev)},
        assign=True,
    )
    out = module(x.to(dev))
    rel_check(out.float().cpu().numpy(), oracle_linear(x, codes, scale, b))
    assert scopes == ["linear.activation_quantize", "linear.fp8_gemm"]


def test_metric_shape_sampled_rows(dev):
    # M=32760, K=5120, N=13824: every row is computed, sampled rows are checked,
    # including the 248-row partial last tile.
    x, codes, scale, b = seeded(32760, 5120, 13824)
    ex = RowFP8Execution("w8a8", activation_quantizer="triton")
    out = ex.linear(x.to(dev), codes.to(dev), scale.to(dev), b.to(dev))
    rows = np.r_[0:32, 4096:4128, 32512:32520, 32728:32760]
    got = out.float().cpu().numpy()[rows]
    rel_check(got, oracle_linear(x, codes, scale, b, rows=rows))
    assert bool(torch.isfinite(out.float()).all())


def test_metric_shape_every_element(dev):
    # M=32760, K=5120, N=13824: all 453 million outputs against the oracle's
    # chain restated in torch (oracle/fp8_torch.py: binary64 sums of the decoded
    # products, the two bf16 roundings) within the GEMM tolerance, and the
    # activation codes and scales of every row bit-exact against the restated
    # oracle quantizer.  The MFMA's binary32 accumulation puts about 1 % of the
    # outputs one bf16 step from the exact sum's rounding (the same accumulation
    # as the reference's own _scaled_mm call, tests/test_gpu_vendor.py); the
    # identical fraction is printed and bounded below.
    from oracle import fp8_torch as T

    m = 32760
    x, codes, scale, b = seeded(m, 5120, 13824)
    xd, cd, sd, bd = x.to(dev), codes.to(dev), scale.to(dev), b.to(dev)
    ex = RowFP8Execution("w8a8", activation_quantizer="triton")
    out = ex.linear(xd, cd, sd, bd)
    a, sa = kernels.quantize_rows(xd)
    ra, rs = T.quantize_rows(xd)
    assert torch.equal(a.view(torch.uint8), ra) and torch.equal(sa.reshape(-1), rs)
    ref = T.add_bias(T.scaled_mm(ra[:m], rs[:m], cd, sd), bd)
    worst, exact = rel_check_device(out, ref)
    print(f"[metric shape] every element: identical {exact:.6f}, worst {worst:.3g}")
    assert exact > 0.95
