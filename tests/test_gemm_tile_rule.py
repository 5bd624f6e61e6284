"""Which rows of an int8 GEMM take 256 x 256 tiles (``rk_int8_gemm_large_rows``), at the shapes on
both sides of the rule's lines. Each line was measured on MI355X; the wrong side of it cost
8-28% (2900 x 4096 x 512 13.7 us in small tiles, 17.8 in large ones).
"""

from __future__ import annotations

import pytest

from local_ai_training import _native as nat

SHAPES = [
    # a short contraction under 256 large tiles: small tiles, whatever the output's width
    (2900, 4096, 256, 0), (2900, 4096, 512, 0), (3600, 4096, 768, 0), (2048, 6144, 512, 0),
    (2304, 5632, 960, 0), (1300, 8192, 512, 0), (1400, 8192, 256, 0),
    # at most 768 small tiles (one round, three to a CU): small up to K 3071
    (2816, 4096, 2048, 0), (3072, 4096, 2560, 0), (1848, 5888, 1664, 0), (6144, 2048, 2048, 0),
    (6144, 2048, 3072, 6144), (3072, 4096, 5632, 3072), (5632, 2048, 5632, 0),
    # more than 768: large from K 1024
    (6656, 2048, 1024, 6656), (3328, 4096, 1024, 3328), (3328, 4096, 1008, 0),
    # 256 large tiles and more: K 256 for wide outputs, K 1024 for narrow ones
    (4096, 4096, 256, 4096), (8192, 2048, 1024, 8192), (8192, 2048, 960, 0),
    # rows past whole rounds go to small tiles where that pays for the second launch
    (5003, 8192, 256, 5003), (5003, 8192, 512, 5003), (5003, 8192, 1024, 4096),
    (8300, 8192, 256, 8192), (3108, 6144, 2048, 2560),
    (2900, 6144, 256, 2560), (9000, 2048, 2048, 8192), (3600, 8192, 960, 3600),
]


@pytest.mark.parametrize("m,n,k,rows", SHAPES)
def test_forward_form(m, n, k, rows):
    assert nat.load_library().rk_int8_gemm_large_rows(m, n, k, 0) == rows


@pytest.mark.parametrize("m,n,k,rows", [(6656, 2048, 1024, 0), (6656, 2048, 1280, 6656),
                                        (3840, 4096, 1088, 0), (8192, 2048, 1024, 8192),
                                        (16, 65536, 4096, 0), (512, 512, 512, 0)])
def test_grad_input_form(m, n, k, rows):
    assert nat.load_library().rk_int8_gemm_large_rows(m, n, k, 1) == rows
