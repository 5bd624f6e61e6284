"""The HIP causal-attention backward (``rk_attention_backward``) against float64 autograd.

Tolerance, element by element. With E the error of ds_ij = p_ij (g_i . v_j - delta_i):
* p and ds enter their products rounded to bf16 (2^-9 relative), and every result is rounded once;
* delta_i carries the rounding of the bf16 o, 2^-9 of sum_d |g_id o_id|;
* the float32 sums g . v and g . o of D terms carry at most D 2^-24 of their absolute sums each;
* the float32 scores and log-sum-exp (products of up to 150 here) move p by less than 2^-12 of it.
So E <= 2^-9 |ds| + p (2^-9 |g|.|o| + 2^-17 (|g|.|v| + |g|.|o|)) + 2^-12 |ds|, and dq, dk and dv are
within scale E |k|, scale E^T |q| and (2^-9 + 2^-12) p^T |g|, plus 2^-9 of themselves. The test
allows twice that.

Lengths: one position, the edges of the 32-row tiles and the 128-row blocks, a ragged long one
and the training window.
"""

from __future__ import annotations

import math

import pytest
import torch

from local_ai_training.attention import CausalAttentionFn, causal_attention
from local_ai_training.ops import ratchet

pytestmark = pytest.mark.gpu

D = 128  # the head size it takes


def inputs(cuda, b, h, s, d, seed=0, scale=1.0):
    gen = torch.Generator().manual_seed(seed + 1000 * s + d)
    qkv = (torch.randn(b, s, 3 * h * d, generator=gen) * scale).to(torch.bfloat16).to(cuda)
    q, k, v = (t.view(b, s, h, d).transpose(1, 2) for t in qkv.chunk(3, dim=-1))
    g = torch.randn(b, s, h, d, generator=gen).to(torch.bfloat16).to(cuda).transpose(1, 2)
    return q, k, v, g


def reference(q, k, v, g):
    """float64 gradients, and the bound on each element (module docstring)."""
    q, k, v, g = (t.detach().double().contiguous() for t in (q, k, v, g))

    def transposed(t):
        return t.transpose(-1, -2).contiguous()

    s, d = q.shape[2:]
    scale = 1.0 / math.sqrt(d)
    mask = torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1)
    p = (q @ transposed(k) * scale).masked_fill(mask, -math.inf).softmax(dim=-1)
    o = p @ v
    ds = p * (g @ transposed(v) - (g * o).sum(dim=-1, keepdim=True))
    go = (g * o).abs().sum(dim=-1, keepdim=True)
    e = (2.0 ** -9 + 2.0 ** -12) * ds.abs() + p * (
        2.0 ** -9 * go + 2.0 ** -17 * (g.abs() @ transposed(v.abs()) + go))
    grads = (scale * ds @ k, scale * transposed(ds) @ q, transposed(p) @ g)
    terms = (scale * e @ k.abs(), scale * transposed(e) @ q.abs(),
             (2.0 ** -9 + 2.0 ** -12) * transposed(p) @ g.abs())
    return [(grad, 2.0 * (term + 2.0 ** -9 * grad.abs())) for grad, term in zip(grads, terms)]


def hip(q, k, v, g):
    scale = 1.0 / math.sqrt(q.shape[-1])
    o, lse = ratchet().attention_forward(q, k, v, scale)
    return ratchet().attention_backward(g, q, k, v, o, lse, scale)


def check(got, operands):
    for mine, (ref, bound) in zip(got, reference(*operands)):
        assert mine.dtype == torch.bfloat16 and bool(torch.isfinite(mine).all())
        assert bool(((mine.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("s", [1, 31, 32, 33, 64, 65, 127, 128, 129, 191, 300, 517, 1024])
def test_gradients_against_float64(cuda, s):
    print(f"attention backward S={s}", flush=True)
    q, k, v, g = inputs(cuda, 2, 3, s, D)
    check(hip(q, k, v, g), (q, k, v, g))


def test_large_scores_and_the_layouts_it_takes(cuda):
    q, k, v, g = inputs(cuda, 1, 2, 200, D, scale=3.0)
    check(hip(q, k, v, g), (q, k, v, g))
    got = hip(*(t.contiguous() for t in (q, k, v, g)))
    for a, b in zip(got, hip(q, k, v, g)):
        assert torch.equal(a, b)  # the same sums whatever the strides
        assert a.transpose(1, 2).is_contiguous()
    # a gradient without unit feature stride or 16-byte rows is copied
    wide = torch.zeros(1, 2, 200, D + 4, device=cuda, dtype=torch.bfloat16)
    wide[..., :D] = g
    for odd in (wide[..., :D], g.transpose(2, 3).contiguous().transpose(2, 3)):
        for a, b in zip(hip(q, k, v, odd), got):
            assert torch.equal(a, b)


def test_runs_repeat_and_rows_past_the_end_do_not_count(cuda):
    # positions past S of a longer buffer hold values that would change every sum
    q, k, v, g = (t.contiguous() for t in inputs(cuda, 2, 2, 160, D))
    for t in (q, k, v, g):
        t[:, :, 130:] = 60000.0
    cut = [t[:, :, :130] for t in (q, k, v, g)]
    first = hip(*cut)
    check(first, cut)
    for a, b in zip(first, hip(*(t.clone() for t in cut))):
        assert torch.equal(a, b)


def test_expanded_gradient_and_double_backward(cuda):
    q, k, v, _ = inputs(cuda, 1, 2, 140, D)  # a length that takes the HIP kernels
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    got = torch.autograd.grad(causal_attention(*leaves).sum(), leaves)
    check(got, (q, k, v, torch.ones_like(q)))
    first = torch.autograd.grad(CausalAttentionFn.apply(*leaves).float().square().sum(), leaves,
                                create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(first[0].float().sum(), leaves)


def test_opcheck(cuda):
    q, k, v, g = inputs(cuda, 2, 2, 40, D)
    o, lse = ratchet().attention_forward(q, k, v, 0.125)
    torch.library.opcheck(ratchet().attention_backward, (g, q, k, v, o, lse, 0.125))


@pytest.mark.parametrize("s,d", [(140, 128), (40, 128), (40, 64)])
def test_a_second_derivative_is_refused_whatever_requires_grad(cuda, s, d):
    """The gradients depend on q, k and v also where the output's gradient is a constant: a
    penalty on them must raise, not leave its share out."""
    leaves = [t.detach().requires_grad_() for t in inputs(cuda, 1, 2, s, d)[:3]]
    out = causal_attention(*leaves)
    first = torch.autograd.grad(out.float().sum(), leaves, create_graph=True)
    check([a.detach() for a in first], (*(t.detach() for t in leaves), torch.ones_like(out)))
    for a in first:
        assert a.requires_grad
        with pytest.raises(RuntimeError):
            torch.autograd.grad(out.float().sum() + a.float().square().sum(), leaves,
                                retain_graph=True)


@pytest.mark.parametrize("create_graph", [False, True])
@pytest.mark.parametrize("s,d", [(140, 128), (40, 128), (40, 64)])
def test_batched_gradients(cuda, s, d, create_graph):
    leaves = [t.detach().requires_grad_() for t in inputs(cuda, 2, 2, s, d)[:3]]
    out = causal_attention(*leaves)
    grads = torch.randn(3, *out.shape, device=cuda).bfloat16()
    got = torch.autograd.grad(out, leaves, grads, retain_graph=True, create_graph=create_graph,
                              is_grads_batched=True)
    one = [torch.autograd.grad(out, leaves, g, retain_graph=True, create_graph=create_graph)
           for g in grads]
    for mine, single in zip(got, zip(*one)):
        assert mine.requires_grad == create_graph and torch.equal(mine, torch.stack(single))
