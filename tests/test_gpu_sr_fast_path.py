"""Stochastic row quantization where its division-free path hands over to the exact one.

The kernel rounds floor(x * (1/s) + u) and redoes a group of values through the IEEE division
only when one lies within 2^-14 of an integer; the result must be floor(RN(RN(x / s) + u)) for
every value, as the oracle computes it. Rows are made of values at and a few ulps around whole
and half steps, where that decision is taken most often, at the row lengths of each kernel form
(one wavefront with 1, 2 and 4 vectors per lane, four wavefronts, the re-reading form) and one
ragged length per form; scales run from the smallest to the largest a row can have.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import quant as oquant

pytestmark = pytest.mark.gpu


def rows_near_steps(m, k, seed, largest):
    rng = np.random.default_rng(seed)
    amax = np.float32(largest) * (0.5 + 0.5 * rng.random((m, 1))).astype(np.float32)
    step = (amax / np.float32(127)).astype(np.float32)
    x = (rng.integers(-254, 255, (m, k)) * np.float32(0.5) * step).astype(np.float32)
    ulps = rng.integers(-3, 4, (m, k)).astype(np.int32)
    x = np.where(x == 0, x, (x.view(np.int32) + ulps).view(np.float32))
    x[:, 0] = amax[:, 0]
    x[m // 2, 1:] = 0.0  # a row of one value
    return np.clip(x, -amax, amax)


@pytest.mark.parametrize("k", [8, 200, 256, 512, 1000, 2048, 2500, 4096, 6144, 9000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sr_equals_the_exact_quotient(cuda, k, dtype):
    from local_ai_training.ops import ratchet

    for seed, largest in ((3, 1.0), (4, 1e-36), (5, 3e38)):
        x = torch.from_numpy(rows_near_steps(37, k, seed, largest)).to(dtype).to(cuda)
        q, s = ratchet().quantize_rows(x, None, True, 1234567 + seed)
        qr, sr = oquant.quantize_rows_sr(x.float().cpu().numpy(), None, 1234567 + seed)
        assert np.array_equal(s.cpu().numpy(), sr)
        assert np.array_equal(q.cpu().numpy(), qr)


def test_non_finite_values(cuda):
    from local_ai_training.ops import ratchet

    x = torch.randn(3, 512, generator=torch.Generator().manual_seed(1))
    x[0, 5], x[1, 7], x[2, 9] = float("nan"), float("inf"), -float("inf")
    q, s = ratchet().quantize_rows(x.to(cuda), None, True, 11)
    clean = x.clone()
    clean[0, 5] = 0.0
    want, want_s = oquant.quantize_rows_sr(clean[:1].numpy(), None, 11)
    got = q.cpu().numpy()
    assert got[0, 5] == -127 and s[0].item() == want_s[0]  # the maximum skips a NaN
    assert np.array_equal(np.delete(got[0], 5), np.delete(want[0], 5))
    # an infinite step: finite values take floor(u) = 0, the infinite one is a NaN quotient
    for row, col in ((1, 7), (2, 9)):
        assert got[row, col] == -127 and not np.delete(got[row], col).any()


def test_bf16_copy_of_float32_rows(cuda):
    from local_ai_training.ops import ratchet

    x = torch.randn(19, 1030, generator=torch.Generator().manual_seed(2)).to(cuda)
    for k, pad in ((1030, 0), (1024, 0), (1024, 3), (40, 4)):
        out = torch.full((19, k + pad), 7.0, device=cuda, dtype=torch.bfloat16)
        ratchet().quantize_rows(x[:, :k].contiguous(), None, True, 3, x_bf16=out[:, :k])
        assert torch.equal(out[:, :k], x[:, :k].bfloat16())
        assert bool((out[:, k:] == 7.0).all())
