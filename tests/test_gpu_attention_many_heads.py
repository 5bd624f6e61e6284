"""More (batch, head) pairs than one launch holds blocks (2^24): the forward takes them in several
launches. With one position the output is the value itself, bit for bit, and the log-sum-exp
the one score, so every pair of both launches is compared."""

from __future__ import annotations

import pytest
import torch

from local_ai_training.attention import attention_supported, causal_attention
from local_ai_training.ops import ratchet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,heads", [(2**24 - 1, 1), (2**24 + 3, 1), (2**23 + 5, 3)])
def test_heads_past_one_launch(cuda, batch, heads):
    print(f"attention forward {batch}x{heads}x1x64", flush=True)
    v = torch.randn(batch, 1, heads, 64, device=cuda, dtype=torch.bfloat16).transpose(1, 2)
    one = torch.ones(1, 1, 1, 64, device=cuda, dtype=torch.bfloat16).expand(batch, heads, 1, 64)
    assert attention_supported(one, one, v)
    with torch.no_grad():
        assert torch.equal(causal_attention(one, one, v), v)
    _, lse = ratchet().attention_forward(one, one, v, 0.125)
    assert float((lse - 8.0).abs().max()) <= 4e-6  # float32: log2, the product with ln 2
