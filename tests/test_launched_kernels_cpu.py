"""The kernels that the GPU tests say they reach: what the library launches for their
shapes on 256 compute units, read from the launches themselves (tests/launches.py),
so that a changed dispatch rule cannot leave a test aimed at another kernel."""

import re

import pytest

from tests import (test_gpu_adapters, test_gpu_few_rows, test_gpu_fused, test_gpu_graph, test_gpu_linear,
                   test_gpu_lora_blocks, test_gpu_nvfp4_tilings, test_gpu_tail_tiles, test_gpu_weight_only)
from tests.launches import LIBRARY, launches

pytestmark = pytest.mark.skipif(not LIBRARY.exists(), reason="the library is not built")
P = "@4096"
FEW_ROWS = r"fp8_gemm_skinny<\d,[12],[68]>"
TILINGS = {"256x256": r"256,256,", "256x192": r"256,192,", "256x128": r"256,128,", "128x192": r"128,192,",
           "128x128": r"128,128,2,", "128x128 one round": r"128,128,3,", "128x64": r"128,64,", "64x64": r"64,64,"}


def up16(v):
    return -(-v // 16) * 16


def tiled(name):
    return r"fp8_gemm_pipe<\d," + TILINGS[name]


def head(m, k, n):
    return [P, P, k, P, P, k, m, n, k, None]


def linear(m, k, n):
    return "vflash_fp8_linear", [*head(m, k, n), P, n, None]


def gate(m, k, n):
    return "vflash_fp8_linear_gate_residual", [*head(m, k, n), P, n, 1, m, None, 0, P, n, P, n, None]


def adapter(m, k, n, rank):
    return "vflash_fp8_linear_lora", [*head(m, k, n), P, up16(rank), P, -(-rank // 8) * 8, rank, 0.5, 1.0, P, n, None]


def adapter_gate(m, k, n, rank):
    return "vflash_fp8_linear_lora_gate_residual", [
        *head(m, k, n), P, n, 1, m, None, 0, P, n, P, up16(rank), P, -(-rank // 8) * 8, rank, 0.5, 1.0, P, n, None]


def branches(m, k, inner, rank):
    return "vflash_fp8_linear_lora_branches", [
        *head(m, k, 3 * inner), P, 3 * up16(rank), up16(rank), P, -(-rank // 8) * 8, rank, 3, [1.0, 0.5, 0.3], 1.0, P,
        3 * inner, 0, 0, None]


def swiglu(m, k, f):
    return "vflash_fp8_linear_swiglu", [*head(m, k, 2 * f), P, f, P, None]


def check(tmp_path, expected):
    """``expected``: (call, pattern of its one kernel) pairs."""
    for (call, pattern), (status, run) in zip(expected, launches(tmp_path, [call for call, _ in expected])):
        assert status == 0 and len(run) == 1, call
        assert re.match(pattern, run[0][0]), (call, run[0][0], pattern)


def table(test, names):
    """The parameter table of a test."""
    (rows,) = [m.args[1] for m in test.pytestmark if m.name == "parametrize" and m.args[0] == names]
    return rows


def test_linear_edges(tmp_path):
    few = test_gpu_linear.EDGES[:4]
    expected = [(entry(m, k, n), FEW_ROWS if (m, k, n, name) in few else tiled(name))
                for m, k, n, name in test_gpu_linear.EDGES for entry in (linear, gate)]
    assert {name for _, _, _, name in test_gpu_linear.EDGES[4:]} == set(TILINGS)
    check(tmp_path, expected)


def test_tail_tiles(tmp_path):
    shapes = table(test_gpu_tail_tiles.test_linear_tail_tiles_match_untailed_operands, "m,n")
    names = ["256x256"] * 3 + ["256x192", "256x128", "128x192", "128x128", "128x128 one round", "128x64", "64x64"]
    patterns = [tiled(name) for name in names] + [FEW_ROWS]
    assert len(shapes) == len(patterns)
    check(tmp_path, [(linear(m, 384, n), p) for (m, n), p in zip(shapes, patterns)])


def test_adapter_epilogues(tmp_path):
    shapes = table(test_gpu_fused.test_lora_epilogue_under_each_tiling, "m,n,k")
    names = ["64x64", "128x64", "128x128", "128x192", "256x128", "256x192", "256x256"]
    patterns = [FEW_ROWS, *map(tiled, names)]
    assert len(shapes) == len(patterns)
    check(tmp_path, [(adapter(m, k, n, 48), p) for (m, n, k), p in zip(shapes, patterns)])
    shapes = table(test_gpu_adapters.test_adapted_gate_residual_on_the_kernels_operands, "m,k,n,rank,scaling,token_gate")
    assert len(shapes) == len(patterns)
    check(tmp_path, [(adapter_gate(m, k, n, rank), p) for (m, k, n, rank, _, _), p in zip(shapes, patterns)])


def test_adapter_branches(tmp_path):
    # Waves inside one branch, except in 256x192 tiles, whose shape is in test_gpu_lora_tiles.py.
    shapes = table(test_gpu_adapters.test_qkv_branches_on_the_kernels_operands, "m,hidden,inner,ranks,scalings")
    calls = [branches(m, k, inner, max(ranks)) for m, k, inner, ranks, _ in shapes]
    for (_, _, inner, _, _), (status, ((kernel, _, _),)) in zip(shapes, launches(tmp_path, calls)):
        columns = re.match(r"fp8_gemm_pipe<3,\d+,(\d+),", kernel)
        assert status == 0 and (re.match(FEW_ROWS, kernel) or inner % (int(columns.group(1)) // 2) == 0), kernel
    check(tmp_path, [(branches(1000, 256, 7168, 100), tiled("256x192")),
                     (adapter(1000, 256, 7168, 100), tiled("256x128"))])


def test_operand_layouts_and_graphs(tmp_path):
    shapes = table(test_gpu_fused.test_gate_residual_operand_layouts_give_the_same_bits, "m,h,k")
    patterns = [FEW_ROWS, tiled("64x64"), r"fp8_gemm_mixed<2,128,128,", tiled("256x192")]
    check(tmp_path, [(gate(m, k, h), p) for (m, h, k), p in zip(shapes, patterns)])
    shapes = table(test_gpu_graph.test_w8a8_linear_replays_from_a_graph, "m,k,n")
    check(tmp_path, [(linear(*s), tiled(name)) for s, name in zip(shapes, ("256x128", "128x192"))])


def test_few_rows(tmp_path):
    widths = table(test_gpu_few_rows.test_few_rows_match_the_tiled_kernel, "n")
    assert widths == [48, 1008, 5136]
    rows32, rows64 = r"fp8_gemm_skinny<\d,1,8>", r"fp8_gemm_skinny<\d,2,6>"
    patterns = {48: [rows32] * 5, 1008: [rows32] * 4 + [rows64], 5136: [rows32] * 2 + [rows64] * 2 + [tiled("128x64")]}
    expected = [(linear(9000 if n == 48 else 2000, 144, n), "fp8_gemm_pipe") for n in widths]
    for n in widths:
        for m, p in zip((1, 17, 40, 64, 300), patterns[n]):
            expected += [(call, p) for call in (linear(m, 144, n), gate(m, 144, n), adapter(m, 144, n, 24),
                                                adapter_gate(m, 144, n, 24))]
    check(tmp_path, expected)


def test_split_last_rounds(tmp_path):
    # test_gpu_mixed_tiles.py, test_gpu_swiglu_tiles.py and test_gpu_tiled.py.
    whole, split = r"fp8_gemm_pipe<4,256,256,", r"fp8_gemm_mixed<4,64,256,"
    expected = [(entry(8269, k, 6288), rf"fp8_gemm_mixed<\d,256,128,") for k in (128, 640) for entry in (linear, gate)]
    expected += [(entry(4095, k, 5120), rf"fp8_gemm_mixed<\d,128,128,") for k in (128, 640) for entry in (linear, gate)]
    expected += [(entry(1024, 128, n), "fp8_gemm_pipe") for n in (6288, 5120) for entry in (linear, gate)]
    expected += [(swiglu(m, k, 1024), split) for k in (128, 640) for m in (8969, 1, 9, 64, 65, 100, 200, 300)]
    expected += [(swiglu(m, 208, 1024), whole) for m in (8969, 9, 300)] + [(swiglu(8192, 640, 1024), whole)]
    expected += [(linear(17, 5120, n), tiled("64x64")) for n in (13824, 15360)]
    expected += [(linear(17, k, n), FEW_ROWS) for k, n in ((5120, 5120), (13824, 5120), (1536, 6144))]
    expected += [(linear(1024, 5120, 5120), tiled("128x192")), (linear(1024, 1536, 6144), tiled("128x192"))]
    expected += [(linear(16384, 5120, 15360), tiled("256x256"))]
    expected += [(linear(m, 5120, n), r"fp8_gemm_mixed<0,256,128,") for m, n in ((16384, 13824), (32785, 15360))]
    check(tmp_path, expected)


def test_adapter_blocks_and_shared_rows(tmp_path):
    def down(m, k, rank):
        return "vflash_lora_down", [P, m, k, k, P, rank, P, up16(rank), None]

    def gelu(m, k):
        return "vflash_gelu_quantize_rows_e4m3", [P, m, k, k, None, 0, P, P, up16(m), None]

    shapes = table(test_gpu_lora_blocks.test_blocks_agree_bit_for_bit, "m,rank,k")
    expected = [(down(m, k, rank), rf"lora_down_blocks<0,{b}>") for (m, rank, k), b in
                zip(shapes, ("2,4", "2,4", "4,4", "4,4"))]
    expected += [(down(16, k, rank), r"lora_down_blocks<0,1,1>") for _, rank, k in shapes]
    expected += [(gelu(m, 4104), rf"gelu_quant_rows<\d+,{waves}>") for m, waves in
                 ((1, 4), (17, 4), (700, 4), (1095, 2), (1500, 2), (3000, 1), (4095, 2))]
    check(tmp_path, expected)


def test_nvfp4_tilings(tmp_path):
    # Both activation kinds take each tiling, 256x256 (the reference side) included.
    assert table(test_gpu_nvfp4_tilings.test_tilings_agree_bit_for_bit, "k") == [64, 320, 640]
    n, expected = 1152, []
    for m, tile in ((1, "64,64"), (17, "64,64"), (65, "64,64"), (300, "64,64"), (1000, "64,128"), (2047, "128,128"),
                    (4001, "256,128"), (8192, "256,256")):
        for k in (64, 320, 640):
            expected += [(("vflash_nvfp4_w4a4_linear", [P, k // 2, P, P, P, P, m, n, k, None, P, n, None]),
                          rf"nvfp4_gemm_pipe<1,{tile},"),
                         (("vflash_nvfp4_linear", [P, P, k, P, P, P, m, n, k, None, P, n, None]),
                          rf"nvfp4_gemm_pipe<0,{tile},")]
    check(tmp_path, expected)


def test_weight_only_tilings(tmp_path):
    shapes = table(test_gpu_weight_only.test_weight_only_linear, "m,k,n")
    tiles = ["64,64"] * 3 + ["128,64", "128,128", "128,256", None, "64,64", "128,64", "128,128", "128,256"]
    assert len(shapes) == len(tiles)
    check(tmp_path, [(("vflash_w8a16_linear", [P, k, P, P, k, m, n, k, None, P, n, None]), rf"w8a16_gemm_pipe<{tile},")
                     for (m, k, n), tile in zip(shapes, tiles) if tile])
