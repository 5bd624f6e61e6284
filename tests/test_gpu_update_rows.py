"""The update at row counts around its blocks of four and eight rows, around the counts that take
blocks of eight (768, streamed rows 2048) and past one row per wavefront of the largest grid
(16384): packed bytes, move counts and row rms, bit for bit.

Every source and width class (in registers, rows of up to 512, 2048 and 6144 columns, float32 512
and 2048; streamed beyond) is compared with the oracle at small row counts. Past 16384 rows
the narrow classes are compared with it too; the wide ones, where it would take minutes, with
the same rows updated in two calls, on the other side of the line or the grid.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import update as oupd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 5, 7, 8, 9, 17, 16384, 16391])
@pytest.mark.parametrize("source,k", [("bf16", 64), ("bf16", 520), ("f32", 72), ("f32", 264),
                                      ("splits", 64), ("splits", 1032), ("one split", 520)])
def test_row_counts(cuda, rows, source, k):
    from local_ai_training.ops import ratchet

    if rows > 100 and k > 100:
        pytest.skip("the oracle's time; the narrow rows walk the same loop")
    rng = np.random.default_rng(rows + k)
    packed = (rng.integers(0, 7, (rows, k)) | (rng.integers(0, 15, (rows, k)) << 4)).astype(np.uint8)
    parts = rng.standard_normal(({"splits": 3}.get(source, 1), rows, k)).astype(np.float32)
    grad = torch.from_numpy(parts[0])
    if source != "f32":  # split partials are added in order, then rounded
        for part in parts[1:]:
            grad = grad + torch.from_numpy(part)
        grad = grad.bfloat16()
    counts = torch.zeros(4, dtype=torch.int64, device=cuda)
    rms = torch.empty(rows, device=cuda)
    state = torch.from_numpy(packed).to(cuda)
    rule = (3, 8, 0.5, 1.5, 1e-8, None, 0.0, counts, rms, None, None, None)
    if "split" in source:
        ratchet().update_from_partials(state, torch.from_numpy(parts).to(cuda), *rule, None)
    else:
        ratchet().update_from_grad(state, grad.to(cuda), *rule)
    want = oupd.update_from_gradient(packed, grad.float().numpy(), 3, 8, 0.5, 1.5, 1e-8,
                                     vec=oupd.vec_for_dtype("f32" if source == "f32" else "bf16"))
    assert np.array_equal(state.cpu().numpy(), want["packed"])
    assert counts.tolist() == want["counts"].tolist()
    assert np.array_equal(rms.cpu().numpy().view(np.uint32), want["row_rms"].view(np.uint32))


# (source, columns): every class that test_row_counts does not reach
WIDE = [("f32", 1032), ("f32", 2312), ("bf16", 2056), ("bf16", 6664), ("splits", 2056),
        ("splits", 6664), ("one split", 64), ("one split", 2056), ("one split", 6664)]


@pytest.mark.parametrize("rows", [1, 5, 9, 17])
@pytest.mark.parametrize("source,k", WIDE)
def test_wide_rows(cuda, rows, source, k):
    test_row_counts(cuda, rows, source, k)


@pytest.mark.parametrize("rows,cut", [(16391, 8201), (2048, 2047), (768, 767)])
@pytest.mark.parametrize("source,k", [("bf16", 64), ("bf16", 520), ("f32", 264), ("splits", 64),
                                      ("splits", 1032), ("one split", 520), *WIDE])
def test_rows_in_one_call_and_in_two(cuda, source, k, rows, cut):
    from local_ai_training.ops import ratchet

    gen = torch.Generator(cuda).manual_seed(k)
    code = torch.randint(0, 7, (rows, k), generator=gen, device=cuda, dtype=torch.uint8)
    pressure = torch.randint(0, 15, (rows, k), generator=gen, device=cuda, dtype=torch.uint8)
    packed = code | (pressure << 4)
    splits = {"splits": 3}.get(source, 1)
    parts = torch.randn(splits, rows, k, generator=gen, device=cuda)

    def run(first, last):
        counts = torch.zeros(4, dtype=torch.int64, device=cuda)
        rms = torch.empty(last - first, device=cuda)
        state = packed[first:last].clone()
        rule = (3, 8, 0.5, 1.5, 1e-8, None, 0.0, counts, rms, None, None, None)
        if "split" in source:
            ratchet().update_from_partials(state, parts[:, first:last].contiguous(), *rule, None)
        else:
            grad = parts[0, first:last]
            ratchet().update_from_grad(state, grad.bfloat16() if source == "bf16" else grad, *rule)
        return state, counts, rms

    state, counts, rms = run(0, rows)
    low, high = run(0, cut), run(cut, rows)
    assert torch.equal(state, torch.cat([low[0], high[0]])) and not torch.equal(state, packed)
    assert torch.equal(counts, low[1] + high[1])
    assert torch.equal(rms.view(torch.int32), torch.cat([low[2], high[2]]).view(torch.int32))
