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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch,heads,head,length", [(3, 4, 64, 1), (2, 5, 128, 40), (1, 2, 8, 7)])
def test_append_writes_what_torch_copies_write(cuda, monkeypatch, dtype, batch, heads, head,
                                               length):
    """Two prompts one after the other, strided keys and values, every position compared."""
    import local_ai_training.model as model_mod

    gen = torch.Generator(device=cuda).manual_seed(length)
    rows = torch.randn(batch, 2 * length + 3, 3 * heads * head, generator=gen, device=cuda).to(dtype)

    def run():
        cache = KVCache(1, batch, heads, head, 2 * length + 9, cuda, dtype=dtype)
        for first, last in ((0, length), (length, 2 * length + 3)):
            _, k, v = (t.unflatten(-1, (heads, head)).transpose(1, 2)
                       for t in rows[:, first:last].chunk(3, dim=-1))
            # a fresh buffer must not show what its memory held before
            torch.full((batch, heads, 2 * length + 9, head), 5.0, device=cuda, dtype=dtype)
            with torch.no_grad():
                cache.append(0, k, v)
            cache.length = last
        return cache.keys[0], cache.values[0]

    got = run()
    monkeypatch.setattr(model_mod, "_hip_append_supported",
                        lambda cache, layer, k, v: False)
    for a, b in zip(got, run()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("buffers", ["none", "strided", "float32 values"])
def test_append_beside_its_own_buffers(cuda, buffers):
    """A first prompt behind position 0 leaves zeros before it; buffers that the caller set are
    written as torch's copies write them."""
    cache = KVCache(1, 2, 3, 64, 24, cuda, dtype=torch.bfloat16)
    cache.length = 5
    if buffers != "none":
        cache.keys[0] = torch.zeros(2, 24, 3, 64, device=cuda, dtype=torch.bfloat16).transpose(1, 2)
        cache.values[0] = torch.zeros(2, 3, 24, 64, device=cuda, dtype=torch.bfloat16)
    if buffers == "float32 values":
        cache.keys[0], cache.values[0] = cache.keys[0].contiguous(), cache.values[0].float()
    k, v = torch.randn(2, 2, 3, 7, 64, device=cuda).bfloat16()
    torch.full((4, 2, 3, 24, 64), 5.0, device=cuda, dtype=torch.bfloat16)
    with torch.no_grad():
        cache.append(0, k, v)
    for got, new in ((cache.keys[0], k), (cache.values[0], v)):
        want = torch.zeros(2, 3, 24, 64, device=cuda)
        want[:, :, 5:12] = new.float()
        assert torch.equal(got.float(), want)


def test_append_refuses_what_does_not_fit(cuda):
    from local_ai_training.ops import ratchet

    keys = torch.zeros(1, 2, 10, 64, device=cuda, dtype=torch.bfloat16)
    k = torch.ones(1, 2, 4, 64, device=cuda, dtype=torch.bfloat16)
    for start, clear_to in ((7, 0), (-1, 0), (0, 11)):
        with pytest.raises(RuntimeError, match="past the cache"):
            ratchet().kv_append(k, k, keys, keys.clone(), start, clear_to)
    with pytest.raises(RuntimeError, match="16-byte"):
        ratchet().kv_append(k[..., :60], k[..., :60], keys[..., :60].contiguous(),
                            keys[..., :60].contiguous(), 0, 0)
    with pytest.raises(ValueError, match="full"):
        KVCache(1, 1, 2, 64, 3, cuda).append(0, k, k)
    assert not keys.any()


def test_append_opcheck(cuda):
    from local_ai_training.ops import ratchet

    keys = torch.randn(2, 2, 12, 64, device=cuda, dtype=torch.bfloat16)
    k = torch.randn(2, 2, 5, 64, device=cuda, dtype=torch.bfloat16)
    torch.library.opcheck(ratchet().kv_append, (k, k * 2, keys, keys.clone(), 3, 12))


@pytest.mark.parametrize("expansion", ["int8", "fp32", "nn.Linear"])
def test_feed_forward_without_gradients_takes_any_expansion(cuda, monkeypatch, expansion):
    """The bf16 hand-over asks an int8 expansion only; another layer in its place is called
    with its inputs alone and its float32 result goes on as it is."""
    config = ModelConfig(vocab_size=64, block_size=16, n_layer=1, n_head=2, n_embd=128,
                         ffn_hidden=256, matmul_mode="int8")
    layer = build_seeded_model(config, max_code=3, seed=1).to(cuda).eval().blocks[0].feed_forward
    if expansion == "nn.Linear":
        layer.expand = torch.nn.Linear(128, 256, bias=False, device=cuda)
    else:
        layer.expand.matmul_mode = expansion
    x = torch.randn(2, 7, 128, device=cuda, generator=torch.Generator(cuda).manual_seed(3))
    with torch.no_grad():
        got = layer(x)
        monkeypatch.setattr(FeedForward, "bf16_expand", False)
        assert got.dtype == torch.float32 and torch.equal(got, layer(x))


@pytest.mark.parametrize("device", ["cuda", "cuda:0", torch.device("cuda"), 0])
def test_append_to_a_cache_on_a_device_of_any_form(cuda, device):
    cache = KVCache(1, 2, 3, 64, 10, device, dtype=torch.bfloat16)
    k, v = torch.randn(2, 2, 3, 7, 64, device=cuda).bfloat16()
    with torch.no_grad():
        cache.append(0, k, v)
    for got, new in ((cache.keys[0], k), (cache.values[0], v)):
        assert got.device == k.device and torch.equal(got[:, :, :7], new)
        assert not got[:, :, 7:].any()
