"""The tiled int8 GEMMs at K % 16 == 0 with a ragged last 64-byte k-step, on the GPU.

The int32 sums are exact, so the output must equal bf16((acc * ls) * rs) in float32, bit for
bit. Shapes: every tail length (16, 32, 48 bytes), tile edges of the 128 x 128 and 256 x 256
ring kernels and of the persistent kernel (N >= 4096), operands whose rows are wider than K
(the bytes past K are set to values that would change the sums if they were read), and 17
token rows (the smallest count the tiled kernels take).
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K, bytes of row padding past K)
SHAPES = [
    (17, 8, 16, 0), (17, 8, 16, 48), (128, 128, 80, 0), (129, 136, 112, 16), (300, 264, 272, 32),
    (1000, 1040, 2768, 0), (257, 2768, 1040, 48), (16385, 264, 1072, 0), (4096, 4104, 1072, 16),
    (4100, 4104, 272, 0), (4100, 4104, 304, 16),
]


@pytest.mark.parametrize("m,n,k,pad", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_tail_gemm_is_exact(cuda, m, n, k, pad, dtype):
    from local_ai_training.int8_matmul import int8_mm_nt, packed_int8_mm

    max_code = 7
    gen = torch.Generator(device=cuda).manual_seed(m + n + k)

    def ints(low, high, *shape, dtype=torch.int8):
        return torch.randint(low, high, shape, generator=gen, device=cuda, dtype=dtype)

    a = ints(-127, 128, m, k + pad)[:, :k]
    nibble = ints(0, 2 * max_code + 1, n, k + pad, dtype=torch.uint8)
    packed = (nibble | (ints(0, 15, n, k + pad, dtype=torch.uint8) << 4))[:, :k]
    code = ((packed & 15).to(torch.int16) - max_code).to(torch.int8)
    ls = torch.rand(m, generator=gen, device=cuda) + 0.5
    rs = torch.rand(n, generator=gen, device=cuda) + 0.5
    acc = (a.double() @ code.double().t().contiguous()).float()
    expect = ((acc * ls[:, None]) * rs[None, :]).bfloat16().to(dtype)
    assert torch.equal(packed_int8_mm(a, packed, max_code, ls, rs, dtype), expect)
    wide = torch.full((n, k + pad), 127, device=cuda, dtype=torch.int8)
    wide[:, :k] = code
    assert torch.equal(int8_mm_nt(a, wide[:, :k], ls, rs, dtype), expect)
    assert torch.equal(int8_mm_nt(a, wide[:, :k], ls, None, dtype),
                       (acc * ls[:, None]).bfloat16().to(dtype))
