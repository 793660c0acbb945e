"""Calls of very many rows stay inside HIP's grid limit (a grid dimension below 2^32
work-items) and start a workgroup for every row."""

import pytest

from tests.launches import LIBRARY, launches

pytestmark = pytest.mark.skipif(not LIBRARY.exists(), reason="the library is not built")
P = "@4096"


# Four rows per workgroup reach 2^26 rows.  Rows that a whole workgroup shares (few
# rows, or above 4096 columns) must get as far: 2^24 rows of 4104 columns fit the
# memory of one GPU.
def test_row_quantizer(tmp_path):
    cases = [(m, k) for k in (512, 4096, 4104, 8192, 16384)
             for m in (1, 17, 2048, 2049, 2**22, 2**22 + 1, 2**24 - 16, 2**24, 2**24 + 1, 2**26 - 16)]
    padded = [(m + 15) // 16 * 16 for m, _ in cases]
    results = launches(tmp_path, [("vflash_quantize_rows_e4m3", [P, m, k, k, P, P, p, None])
                                  for (m, k), p in zip(cases, padded)])
    for (m, k), rows, (status, run) in zip(cases, padded, results):
        assert status == 0 and len(run) == 1, (m, k)
        kernel, (x, y, z), threads = run[0]
        assert x * y * (1 if kernel.endswith(",4>") else 4) >= rows and z == 1 and threads == 256, (m, k, kernel)


@pytest.mark.parametrize("n", [1, 5120, 2**22, 2**22 + 1, 2**24 - 1, 2**24, 2**26 + 3, 2**31 - 1])
def test_restored_weight(tmp_path, n):
    (status, run), = launches(tmp_path, [("vflash_restore_rows_bf16", [P, P, 16, n, 16, P, None])])
    assert status == 0 and len(run) == 1
    _, (x, y, _), _ = run[0]
    assert x * y >= n


# At 2^30 columns a call of few rows needs more tiles than a grid holds: refused as an
# argument from 2^29 on, before the runtime would.
@pytest.mark.parametrize("m,n,want", [(1, 2**24, 0), (64, 2**29 - 8, 0), (256, 2**29 - 8, 0), (1024, 2**24, 0),
                                      (1, 2**29, -1), (1, 2**31, -1)])
def test_weight_only_gemm(tmp_path, m, n, want):
    (status, run), = launches(tmp_path, [("vflash_w8a16_linear", [P, 16, P, P, 16, m, n, 16, None, P, n, None])])
    assert status == want and len(run) == (want == 0)
