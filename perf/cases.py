"""The work that users of this package have it do, as cases that can be timed.

Every case is one call sequence through the public entry points, over the sizes of
the package's own configurations, tests and benchmark: the H3 denoiser's linears
(hidden 5376, inner 7168, FFN 14336), the 5120-wide configuration, the skinny audio
widths, row tiles with their remainders, and the default weight-only mode.

kind         entry points
linear       ``RowFP8Execution("w8a8").linear``
lora         ``fused.fp8_linear_lora``
qkv          ``fused.qkv_linear`` (planes, or chunked views; with or without the adapter pack)
ffn          ``fused.fp8_ffn`` (GELU-tanh or SwiGLU; optionally behind the fused producer)
producer     ``producers.rmsnorm_modulate_quantize``
nvfp4        ``NVFP4Execution.linear`` (W4A4 or W4A8)
weight_only  ``RowFP8Execution().linear``
"""

import math

import torch

from vflash_amd import fused
from vflash_amd.fp8_linear import RowFP8Execution
from vflash_amd.nvfp4_linear import NVFP4Execution, NVFP4Weight
from vflash_amd.prepare import quantize_nvfp4_weight, quantize_weight_rows
from vflash_amd.producers import rmsnorm_modulate_quantize

BF16 = torch.bfloat16
EPS = 1e-6


def listed():
    return [
        # The remainder of a row-tiled forward (1024-row tiles leave a few rows):
        # the smallest call, where launches and weight reads count.
        dict(name="linear_tail_17x5120x5120", kind="linear", m=17, k=5120, n=5120, bias=True),
        # One FP8 linear of the small configuration.
        dict(name="linear_4096x3072x3072", kind="linear", m=4096, k=3072, n=3072, bias=True),
        # The headline linear: all tokens of a 21x30x52 latent through the FFN up-projection.
        dict(name="linear_32760x5120x13824", kind="linear", m=32760, k=5120, n=13824, bias=True),
        # An audio-stream linear with its rank-32 adapter.
        dict(name="lora_256x1536x4608_r32", kind="lora", m=256, k=1536, n=4608, rank=32),
        # The merged Q/K/V projection of one 1024-row tile, with the three rank-128
        # adapters of the production pipeline, written as planes.
        dict(name="qkv_1024x5376x7168_r128", kind="qkv", m=1024, k=5376, inner=7168, rank=128, planes=True),
        # The GELU feed-forward on one GPU's share of an eight-way token split.
        dict(name="ffn_gelu_4095x5120x13824", kind="ffn", m=4095, h=5120, f=13824, act="gelu_tanh",
             norm=False),
        # The H3 feed-forward on the live text and audio rows of an audio pass.
        dict(name="ffn_swiglu_777x5376x14336", kind="ffn", m=777, h=5376, f=14336, act="swiglu", norm=False),
        # The H3 feed-forward half of a block on every token: norm, modulation and
        # quantization, SwiGLU input, output with gate-residual.  The largest call.
        dict(name="ffn_block_32760x5376x14336", kind="ffn", m=32760, h=5376, f=14336, act="swiglu", norm=True),
        # An NVFP4 (W4A4) projection of the H3 block on a few hundred rows.
        dict(name="nvfp4_w4a4_300x5376x7168", kind="nvfp4", m=300, k=5376, n=7168, act="nvfp4"),
        # The same arithmetic on every token at the configuration's widths.
        dict(name="nvfp4_w4a4_32760x5120x13824", kind="nvfp4", m=32760, k=5120, n=13824, act="nvfp4"),
        # NVFP4 weights with per-token E4M3 activations, one 1024-row tile.
        dict(name="nvfp4_w4a8_1024x5120x13824", kind="nvfp4", m=1024, k=5120, n=13824, act="e4m3"),
        # The default mode: text tokens through a linear restored from its codes.
        dict(name="weight_only_512x5120x5120", kind="weight_only", m=512, k=5120, n=5120, bias=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _width(rng, lo, hi, q):
    """A width in [lo, hi], a multiple of q: half of them the package's own, half any."""
    own = [v for v in (1536, 3072, 4608, 5120, 5376, 6144, 7168, 13824, 14336) if lo <= v <= hi and v % q == 0]
    if own and rng.random() < 0.5:
        return rng.choice(own)
    return max(q, round(_log(rng, lo, hi) / q) * q)


def draw(rng):
    kind = rng.choice(["linear", "linear", "lora", "qkv", "ffn", "ffn", "producer", "nvfp4", "nvfp4", "weight_only"])
    m = int(_log(rng, 1, 32760))
    if kind == "linear":
        return dict(kind=kind, m=m, k=_width(rng, 512, 14336, 16), n=_width(rng, 512, 14336, 16),
                    bias=rng.random() < 0.7)
    if kind == "lora":
        return dict(kind=kind, m=int(_log(rng, 16, 4096)), k=_width(rng, 1024, 7168, 16),
                    n=_width(rng, 1024, 7168, 16), rank=rng.choice([16, 32, 128, rng.randint(1, 128)]))
    if kind == "qkv":
        return dict(kind=kind, m=m, k=_width(rng, 1024, 5376, 16), inner=_width(rng, 1024, 7168, 32),
                    rank=rng.choice([0, 16, 128]), planes=rng.random() < 0.5)
    if kind == "ffn":
        return dict(kind=kind, m=m, h=_width(rng, 1024, 5376, 16), f=_width(rng, 2048, 14336, 128),
                    act=rng.choice(["gelu_tanh", "swiglu"]), norm=rng.random() < 0.3)
    if kind == "producer":
        return dict(kind=kind, m=m, k=_width(rng, 1024, 7168, 16))
    if kind == "nvfp4":
        return dict(kind=kind, m=min(m, 16384), k=_width(rng, 1024, 7168, 64), n=_width(rng, 1024, 14336, 128),
                    act=rng.choice(["nvfp4", "e4m3"]))
    return dict(kind=kind, m=int(_log(rng, 16, 4096)), k=_width(rng, 1024, 5376, 16),
                n=_width(rng, 1024, 7168, 16), bias=rng.random() < 0.5)


class _Inputs:
    """Seeded tensors on the GPU, with the configurations' distributions."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=BF16):
        return torch.empty(shape, device="cuda").normal_(0.0, std, generator=self.g).to(dtype)

    def uniform(self, *shape):
        return torch.empty(shape, device="cuda").uniform_(0.0, 1.0, generator=self.g).to(BF16)

    def fp8(self, n, k):
        return quantize_weight_rows(self.normal(n, k, std=0.02, dtype=torch.float32))


def _index(m, rows=8):
    """The adaLN row of each token of a packed sequence: runs of tokens share a row."""
    return (torch.arange(m, device="cuda") * rows) // m


def prepare(case, seed):
    kind, i = case["kind"], _Inputs(seed)
    s = {"case": dict(case)}
    m = case["m"]
    if kind in ("linear", "weight_only"):
        n, k = case["n"], case["k"]
        s["ex"] = (RowFP8Execution("w8a8", activation_quantizer="hip") if kind == "linear" else RowFP8Execution())
        s["x"] = i.normal(m, k)
        s["w"], s["s"] = i.fp8(n, k)
        s["b"] = i.normal(n, std=0.01) if case["bias"] else None
    elif kind == "lora":
        n, k, r = case["n"], case["k"], case["rank"]
        s["ex"] = RowFP8Execution("w8a8", activation_quantizer="hip")
        s["x"] = i.normal(m, k)
        s["w"], s["s"] = i.fp8(n, k)
        s["b"] = i.normal(n, std=0.01)
        s["down"], s["up"] = i.normal(r, k, std=0.01), i.normal(n, r, std=0.01)
    elif kind == "qkv":
        n, k, r = 3 * case["inner"], case["k"], case["rank"]
        s["ex"] = RowFP8Execution("w8a8", activation_quantizer="hip")
        s["x"] = i.normal(1, m, k)
        s["w"], s["s"] = i.fp8(n, k)
        s["parts"] = [fused.LowRankResidual(i.normal(r, k, std=0.01), i.normal(case["inner"], r, std=0.01), f)
                      for f in (1.0, 0.5, 0.75)] if r else []
        s["pack"] = fused.stack_adapters(s["parts"], k, n) if r else ()
    elif kind == "ffn":
        h, f = case["h"], case["f"]
        s["ex"] = RowFP8Execution("w8a8", activation_quantizer="hip")
        s["x"], s["res"] = i.normal(1, m, h), i.normal(1, m, h)
        s["wu"], s["su"] = i.fp8(2 * f if case["act"] == "swiglu" else f, h)
        s["wd"], s["sd"] = i.fp8(h, f)
        s["bu"], s["bd"] = i.normal(s["wu"].shape[0], std=0.01), i.normal(h, std=0.01)
        s["table"] = i.uniform(8, 6, h)
        s["index"] = _index(m)
        s["norm"] = i.uniform(h)
    elif kind == "producer":
        s["x"] = i.normal(1, m, case["k"])
        s["table"] = i.uniform(8, 6, case["k"])
        s["index"] = _index(m)
        s["norm"] = i.uniform(case["k"])
    else:
        n, k = case["n"], case["k"]
        s["ex"] = NVFP4Execution(activations=case["act"])
        s["x"] = i.normal(m, k)
        # The calibrated global scale of the activations: 448 * 6 over the largest of them.
        s["weight"] = NVFP4Weight(*quantize_nvfp4_weight(i.normal(n, k, std=0.02, dtype=torch.float32),
                                                         input_scale=2688.0 / 5.5))
        s["b"] = i.normal(n, std=0.01)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind in ("linear", "weight_only"):
        return s["ex"].linear(s["x"], s["w"], s["s"], s["b"])
    if kind == "lora":
        return fused.fp8_linear_lora(s["ex"], s["x"], s["w"], s["s"], s["b"], s["down"], s["up"], scaling=0.5)
    if kind == "qkv":
        return fused.qkv_linear(s["ex"], s["x"], s["w"], s["s"], planes=c["planes"], residuals=s["pack"])
    if kind == "producer":
        q = rmsnorm_modulate_quantize(s["x"], s["norm"], s["table"][:, 1, :], s["table"][:, 0, :], eps=EPS,
                                      index=s["index"])
        return q.codes, q.scales
    if kind == "ffn":
        x = s["x"]
        if c["norm"]:
            x = rmsnorm_modulate_quantize(x, s["norm"], s["table"][:, 4, :], s["table"][:, 3, :], eps=EPS,
                                          index=s["index"])
        return fused.fp8_ffn(s["ex"], x, s["wu"], s["su"], s["bu"], s["wd"], s["sd"], s["bd"],
                             s["table"][:, 5, :], s["res"], activation=c["act"], gate_index=s["index"])
    return s["ex"].linear(s["x"], s["weight"], s["b"])


def work(case):
    kind, m = case["kind"], case["m"]
    if kind in ("linear", "lora", "weight_only"):
        n, k, r = case["n"], case["k"], case.get("rank", 0)
        return {"bytes": 2 * m * k + n * k + 6 * n + 2 * m * n + 2 * r * (k + n), "flops": 2 * m * (n * k + r * (n + k))}
    if kind == "qkv":
        n, k, r = 3 * case["inner"], case["k"], case["rank"]
        return {"bytes": 2 * m * k + n * k + 4 * n + 2 * m * n + 2 * r * (3 * k + n),
                "flops": 2 * m * (n * k + r * (n + 3 * k))}
    if kind == "producer":
        return {"bytes": m * (3 * case["k"] + 4), "flops": 8 * m * case["k"]}
    if kind == "ffn":
        h, f = case["h"], case["f"]
        up = 2 * f if case["act"] == "swiglu" else f
        return {"bytes": 6 * m * h + (up + f) * h + 6 * (up + h), "flops": 2 * m * h * (up + f)}
    n, k = case["n"], case["k"]
    return {"bytes": 2 * m * k + n * k // 2 + n * k // 16 + 2 * n + 2 * m * n, "flops": 2 * m * n * k}


# Relative errors (2-norm), three to four times the measured distance of the entry
# points' outputs from exact(): 0.0017 with one rounding to bfloat16 per output, 0.0023
# with two (the bias), 0.0029 with an adapter, 0.0034 for an FFN, where a code of its
# second quantization can also fall to the neighbour.  The producer's outputs are E4M3
# codes and row scales: 0.0001, the few codes at a rounding boundary.
def tolerance(case):
    return {"rel": {"ffn": 1e-2, "producer": 5e-4}.get(case["kind"], 8e-3)}


def _e4m3_rows(x):
    """Codes (as float64 values) and scales of the per-token E4M3 quantization."""
    x = x.float()
    amax = x.abs().amax(dim=1, keepdim=True)
    scale = torch.where(amax > 0, torch.clamp((amax.double() / 448.0).float(), min=torch.finfo(torch.float32).tiny),
                        torch.ones_like(amax))
    q = torch.clamp(x / scale, -448.0, 448.0).to(torch.float8_e4m3fn)
    return q.double(), scale.double()


E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _nvfp4_weight(w):
    n, half = w.packed.shape
    table = torch.tensor(E2M1, dtype=torch.float64, device=w.packed.device)
    q = torch.stack([table[(w.packed & 15).long()], table[(w.packed >> 4).long()]], dim=-1).reshape(n, 2 * half)
    sf = w.scales.view(torch.float8_e4m3fn).double().reshape(n // 128, half // 32, 32, 4, 4)
    sf = sf.permute(0, 3, 2, 1, 4).reshape(n, half // 8)
    return (q.reshape(n, half // 8, 16) * sf.unsqueeze(-1)).reshape(n, 2 * half)


def _nvfp4_rows(x, gsf):
    """The activations as W4A4 sees them: E2M1 value times E4M3 block scale."""
    m, k = x.shape
    b = x.float().reshape(m, k // 16, 16)
    sf = torch.clamp(gsf * (b.abs().amax(dim=-1) * torch.tensor(1.0 / 6.0, device=x.device)), max=448.0)
    sf = sf.to(torch.float8_e4m3fn).float()
    one = torch.ones_like(sf)
    scale = torch.where(sf != 0, one / (sf * (torch.ones_like(gsf) / gsf)), torch.zeros_like(sf))
    v = torch.clamp(b * scale.unsqueeze(-1), -6.0, 6.0)
    a = v.abs()
    q = torch.zeros_like(a)
    for edge, low, step in ((0.25, 1, .5), (0.75, 0, .5), (1.25, 1, .5), (1.75, 0, .5), (2.5, 1, 1.), (3.5, 0, 1.),
                            (5.0, 1, 2.)):
        q = q + step * ((a > edge) if low else (a >= edge))
    return (torch.copysign(q, v).double() * sf.double().unsqueeze(-1)).reshape(m, k)


def _modulated(s, shift, scale):
    """bf16 output of RMSNorm and adaLN modulation, each rounding of the contract from 64 bits."""
    x = s["x"].reshape(-1, s["x"].shape[-1]).double()
    n = (x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + EPS) * s["norm"].double()).to(BF16).double()
    t = s["table"][s["index"]]
    y = (n * (1.0 + t[:, scale].double()).to(BF16).double()).to(BF16).double()
    return (y + t[:, shift].double()).to(BF16)


def exact(case, seed):
    """What run() returns, with every sum and product in 64 bits; tensors that the
    contract stores in bfloat16 or E4M3 on the way are rounded there."""
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "producer":
        q, scale = _e4m3_rows(_modulated(s, 0, 1))
        pad = -q.shape[0] % 16
        return (torch.cat([q, torch.zeros((pad, q.shape[1]), dtype=q.dtype, device=q.device)]),
                torch.cat([scale, torch.ones((pad, 1), dtype=scale.dtype, device=q.device)]))
    if kind == "ffn":
        q, a = _e4m3_rows(_modulated(s, 3, 4) if case["norm"] else s["x"].reshape(-1, case["h"]))
        y = (q @ s["wu"].double().T) * a * s["su"].double().T
        y = (y.to(BF16).double() + s["bu"].double()).to(BF16).double()
        if case["act"] == "swiglu":
            v, g = y.chunk(2, dim=1)
            y = v * torch.nn.functional.silu(g).to(BF16).double()
        else:
            y = torch.nn.functional.gelu(y, approximate="tanh")
        q, a = _e4m3_rows(y.to(BF16))
        z = (q @ s["wd"].double().T) * a * s["sd"].double().T + s["bd"].double()
        return (s["res"].double() + s["table"][:, 5][s["index"]].double() * z).reshape(s["res"].shape)
    x = s["x"].reshape(-1, s["x"].shape[-1])
    if kind == "nvfp4":
        w = s["weight"]
        if case["act"] == "nvfp4":
            y = (_nvfp4_rows(x, w.input_scale) @ _nvfp4_weight(w).T) * (w.alpha.double() / w.input_scale.double())
        else:
            q, a = _e4m3_rows(x)
            y = (q @ _nvfp4_weight(w).T) * a * w.alpha.double()
        return y + s["b"].double()
    if kind == "weight_only":
        w = (s["w"].double() * s["s"].double()).to(BF16).double()
        y = x.double() @ w.T
        return y if s["b"] is None else y + s["b"].double()
    q, a = _e4m3_rows(x)
    y = (q @ s["w"].double().T) * a * s["s"].double().T
    if kind == "linear":
        return y if s["b"] is None else y + s["b"].double()
    if kind == "lora":
        t = (x.double() @ s["down"].double().T).to(BF16).double()
        return y + s["b"].double() + 0.5 * (t @ s["up"].double().T)
    if s["parts"]:
        y = y + torch.cat([((x.double() @ r.down.double().T).to(BF16).double() @ r.up.double().T) * r.scaling
                           for r in s["parts"]], dim=1)
    return tuple(v.reshape(*s["x"].shape[:-1], -1) for v in y.chunk(3, dim=1))
