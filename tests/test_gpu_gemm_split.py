"""Outputs whose rows are split between whole rounds of large tiles and small tiles, and grids of
fewer than 256 large tiles on both sides of the rule that takes them.

The int32 sums are exact, so every output must equal bf16((acc * ls) * rs) in float32, bit for
bit, plus the residual's float32 add: row, scale, output and residual offsets of the second
launch, the last row of either part, and both operand forms with and without a ragged K.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K): two launches (pipe and ring kernels, one row past the first part, ragged K), then
# one launch of 220 large tiles, of 768 small ones, of 224 large ones
SHAPES = [(3108, 6144, 1024), (2561, 6144, 1024), (2817, 5632, 1072), (8449, 2048, 1024),
          (4225, 4096, 1088), (5003, 2768, 1040), (2900, 4096, 1024),
          (3400, 4096, 1088)]


def operands(cuda, m, n, k, seed):
    gen = torch.Generator(device=cuda).manual_seed(seed)
    a = torch.randint(-127, 128, (m, k), generator=gen, device=cuda, dtype=torch.int8)
    packed = torch.randint(0, 7, (n, k), generator=gen, device=cuda, dtype=torch.uint8)
    packed |= torch.randint(0, 15, (n, k), generator=gen, device=cuda, dtype=torch.uint8) << 4
    ls = torch.rand(m, generator=gen, device=cuda) + 0.5
    rs = torch.rand(n, generator=gen, device=cuda) + 0.5
    return a, packed, ls, rs, (packed & 15).double() - 3


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_forward(cuda, m, n, k):
    from local_ai_training.int8_matmul import (packed_int8_mm, packed_int8_mm_residual,
                                               residual_supported)

    a, packed, ls, rs, code = operands(cuda, m, n, k, m)
    acc = (a.double() @ code.t().contiguous()).float()
    expect = ((acc * ls[:, None]) * rs[None, :]).bfloat16()
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(packed_int8_mm(a, packed, 3, ls, rs, dtype), expect.to(dtype))
    residual = torch.randn(m, n, device=cuda)
    if residual_supported(a, packed, residual):
        got = packed_int8_mm_residual(a, packed, 3, ls, rs, residual)
        assert torch.equal(got, residual + expect.float())


@pytest.mark.parametrize("m,n,k", [(3108, 5632, 1024), (2561, 6144, 1088), (8449, 2048, 1024),
                                   (7000, 2048, 1024), (7000, 2048, 1280)])
def test_grad_input(cuda, m, n, k):
    from local_ai_training.int8_matmul import packed_int8_mm_t

    a, packed, ls, _, code = operands(cuda, m, k, n, n)
    a = torch.randint(-127, 128, (m, k), device=cuda, dtype=torch.int8)
    expect = ((a.double() @ code).float() * ls[:, None]).bfloat16()
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(packed_int8_mm_t(a, packed, 3, ls, None, dtype), expect.to(dtype))
