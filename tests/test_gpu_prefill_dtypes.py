"""Prefill takes the int8 layers' bf16 results directly where only their values matter.

Without gradients the qkv projection (into a bf16 cache) and the feed-forward expansion hand on
their bf16 results; widened and narrowed again they are the same values, so logits, keys and
values equal those of the float32 hand-over bit for bit, the output dtypes stay, and the
cache's unwritten positions are zero.
"""

from __future__ import annotations

import pytest
import torch

from local_ai_training.model import FeedForward, KVCache, ModelConfig, build_seeded_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cache_dtype", [torch.bfloat16, torch.float32, None])
@pytest.mark.parametrize("prompt", [(1,), (33,), (64,), (20, 13)])
def test_prefill_equals_the_float32_hand_over(cuda, monkeypatch, cache_dtype, prompt):
    config = ModelConfig(vocab_size=256, block_size=64, n_layer=2, n_head=4, n_embd=256,
                         ffn_hidden=640, matmul_mode="int8")
    model = build_seeded_model(config, max_code=3, seed=4).to(cuda).eval()
    tokens = torch.randint(0, 256, (3, sum(prompt)), generator=torch.Generator().manual_seed(1))

    def run():
        cache = model.new_cache(3, dtype=cache_dtype)
        logits = [model.prefill(part.to(cuda), cache) for part in tokens.split(prompt, dim=1)]
        return logits, cache

    logits, cache = run()
    monkeypatch.setattr(KVCache, "stores_bf16", lambda self, layer: False)
    monkeypatch.setattr(FeedForward, "bf16_expand", False)
    want, kept = run()
    for a, b in zip(logits + cache.keys + cache.values, want + kept.keys + kept.values):
        assert a.dtype == b.dtype and torch.equal(a, b)
    for t in cache.keys + cache.values:
        assert not t[:, :, sum(prompt):].any()
