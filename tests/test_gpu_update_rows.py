"""The update at row counts around its blocks of four and eight rows and past one row per
wavefront of the largest grid (16384), for every source and width class, against the oracle:
packed bytes, move counts and row rms, bit for bit.
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
