"""Causal self-attention of the training step on HIP kernels.

The reference attends with ``F.scaled_dot_product_attention(q, k, v, is_causal=True)``
(``model.py:117-123``). Here the forward is ``rk_attention_forward`` (flash form on the bf16
MFMA, ``csrc/rk_attention.hip``), which writes the output and the per-query log-sum-exp in
the form torch's memory-efficient attention forward does; the backward is
``rk_attention_backward`` (``csrc/rk_attention_bwd.hip``) at head size 128 where that is the
faster one (``_backward_fits``): 165 us at B 8, H 16, S 1024 against 293 us for torch's
memory-efficient backward, which adds its float32 dq by atomics in an order that varies from
1024 positions on. Both are equally far from float64 (relative errors of dq, dk, dv 2.48e-3,
2.46e-3, 2.30e-3 there, the same to three digits at 96 to 2048 positions and for scores of three
times the size). Elsewhere, and at head size 64, it is torch's memory-efficient backward, called
on the forward's two tensors. The same two HIP kernels at head size 64 took 70 us against 131 at
B 32, H 8, S 512; they are not in use, for no lack of accuracy: they round differently, and the
stochastic rounding and the update's thresholds downstream turn on last bits.

Supported: bfloat16 GPU q, k, v [B, H, S, D] with D 64 or 128, unit feature stride,
16-byte aligned storage and strides that are multiples of 8 elements, no attention mask,
no dropout, the default scale. Anything else goes to ``F.scaled_dot_product_attention``.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F
from torch import Tensor

from .ops import ratchet

_NO_DROPOUT_SEED: dict[int, tuple[Tensor, Tensor]] = {}


def _philox_placeholders() -> tuple[Tensor, Tensor]:
    """The (seed, offset) pair the memory-efficient backward takes; unused without dropout."""
    key = 0
    if key not in _NO_DROPOUT_SEED:
        _NO_DROPOUT_SEED[key] = (torch.zeros((), dtype=torch.int64),
                                 torch.zeros((), dtype=torch.int64))
    return _NO_DROPOUT_SEED[key]


def _extent_fits(shape: tuple[int, ...], stride: tuple[int, ...]) -> bool:
    """The kernel's 32-bit buffer offsets: one (batch, head)'s rows up to S + 128 (the last
    key block's padding) within 2^31 bytes of bf16, at most 2^31 - 1 (batch, head) pairs, and
    fewer than 2^24 blocks of 128 positions in a head (the same limits ``rk_attention_forward``
    checks before launching)."""
    b, h, s, d = shape
    return (((s + 128) * stride[2] + d) * 2 < 2**31 and b * h <= 0x7FFFFFFF
            and s <= 128 * (2**24 - 1))


def attention_supported(q: Tensor, k: Tensor, v: Tensor) -> bool:
    if not (q.is_cuda and q.dtype == torch.bfloat16 and q.dim() == 4):
        return False
    if k.shape != q.shape or v.shape != q.shape or k.dtype != q.dtype or v.dtype != q.dtype:
        return False
    if q.shape[-1] not in (64, 128):
        return False
    for t in (q, k, v):
        if t.stride(-1) != 1 or t.data_ptr() % 16 or any(s % 8 for s in t.stride()[:3]):
            return False
        if not _extent_fits(tuple(t.shape), t.stride()):
            return False
    return True


def _backward_fits(tensors: tuple[Tensor, ...]) -> bool:
    """What ``rk_attention_backward`` takes (head size 128, and the limits of its 32-bit offsets:
    one head's rows up to the padded length within 2^31 bytes of bf16, and all rows' two float32
    statistics), where it is the faster one.

    torch's kernel walks a head of up to 128 positions in one block; the HIP pair is two
    launches of 128-row blocks. Device time in us, torch / HIP: 16 heads in all S 48 8.9 / 14.7,
    S 128 14.7 / 23.3, S 160 36.9 / 24.7; 64 heads S 112 20.7 / 23.5, S 128 25.9 / 24.0; 128 heads
    S 48 13.4 / 15.2, S 64 22.4 / 15.9; 256 heads S 16 9.0 / 11.6, S 32 18.9 / 12.9; 1024 heads
    S 12 22.0 / 22.7, S 24 63.2 / 25.8. So up to 128 positions HIP takes 24 or more with at least
    8192 positions over all heads."""
    b, h, s, d = tensors[0].shape
    padded = -(-s // 128) * 128
    return (d == 128 and (s > 128 or s >= 24 and b * h * s >= 8192)
            and 8 * b * h * padded < 2**31
            and ((padded + 64) * max(t.stride(2) for t in tensors) + d) * 2 < 2**31)


class CausalAttentionFn(torch.autograd.Function):
    """o = causal softmax(q k^T / sqrt(D)) v: HIP forward, HIP backward at head size 128."""

    @staticmethod
    def forward(ctx, q: Tensor, k: Tensor, v: Tensor) -> Tensor:
        scale = 1.0 / math.sqrt(q.shape[-1])
        out, lse = ratchet().attention_forward(q, k, v, scale)
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, grad_out: Tensor):
        q, k, v, out, lse = ctx.saved_tensors
        # create_graph: torch's operator, which knows that its results depend on q, k and v
        # (and refuses their derivative), batched gradients included
        if not torch.is_grad_enabled() and _backward_fits((q, k, v, out, grad_out)):
            return ratchet().attention_backward(grad_out, q, k, v, out, lse, ctx.scale)
        seed, offset = _philox_placeholders()
        dq, dk, dv, _ = torch.ops.aten._scaled_dot_product_efficient_attention_backward(
            grad_out, q, k, v, None, out, lse, seed, offset, 0.0, [True, True, True, False], True)
        return dq, dk, dv


def causal_attention(q: Tensor, k: Tensor, v: Tensor) -> Tensor:
    """``F.scaled_dot_product_attention(q, k, v, is_causal=True)``: the HIP forward where it
    applies, torch's otherwise."""
    if attention_supported(q, k, v):
        return CausalAttentionFn.apply(q, k, v)
    return F.scaled_dot_product_attention(q, k, v, is_causal=True)
