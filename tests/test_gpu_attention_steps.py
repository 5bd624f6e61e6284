"""The keys that share one update of the attention forward's running max: 32 at head size 128, 64
at 64. Probabilities are rounded to bf16 relative to the running max after their update, and
what was summed before is rescaled in float32, so this count is part of the result's rounding.

The first U keys score 0 and the next U score s > 0; only the first key has a value. With updates
of U keys its probability is 1 exactly and the rescale by exp(-s) is float32, so the output is
the exact quotient rounded once to bf16 (float32 exp2, sums and quotient: under 2^-20 relative).
With more keys per update the probability exp(-s) itself is rounded to bf16 first, a second
error of up to 2^-9 that leaves many elements more than half a bf16 step off.
"""

from __future__ import annotations

import math

import pytest
import torch

from local_ai_training.ops import ratchet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,u", [(64, 64), (128, 32)])
def test_keys_per_update_of_the_running_max(cuda, d, u):
    s, scale = 2 * u, 1.0 / math.sqrt(d)
    q, k, v = (torch.zeros(1, 1, s, d) for _ in range(3))
    q[0, 0, :, 0] = torch.linspace(1, 30, s)
    k[0, 0, u:, 0] = 1.0
    v[0, 0, 0] = torch.randn(d, generator=torch.Generator().manual_seed(d))
    q, k, v = (t.bfloat16() for t in (q, k, v))
    out, _ = ratchet().attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    e = torch.exp(q[0, 0, u:, 0].double() * scale)
    later = torch.arange(1, u + 1, dtype=torch.float64)  # later keys that each query sees
    exact = v[0, 0, 0].double()[None, :] / (u + later * e)[:, None]
    half_step = torch.exp2(torch.floor(torch.log2(exact.abs())) - 8)
    error = (out[0, 0, u:].double().cpu() - exact).abs()
    assert bool((error <= half_step + 2.0 ** -20 * exact.abs()).all())
