"""Which attention backward a call takes: shapes on both sides of every line of the rule (each line
was measured; the wrong side cost up to 2x in device time at few short heads)."""

from __future__ import annotations

import pytest
import torch

from local_ai_training.attention import _backward_fits


@pytest.mark.parametrize("b,h,s,d,hip", [
    (8, 16, 1024, 128, True), (1, 1, 129, 128, True), (1, 16, 160, 128, True),
    (1, 16, 128, 128, False), (1, 4, 96, 128, False), (1, 1, 1, 128, False),
    (4, 16, 128, 128, True), (4, 16, 127, 128, False), (8, 16, 64, 128, True),
    (8, 16, 63, 128, False), (64, 16, 24, 128, True), (512, 16, 23, 128, False),
    (512, 16, 8, 128, False), (32, 8, 512, 64, False),
])
def test_rule(b, h, s, d, hip):
    q = torch.empty(b, s, h, d, dtype=torch.bfloat16, device="meta").transpose(1, 2)
    assert _backward_fits((q, q, q, q, q)) is hip


def test_limits_of_the_offsets():
    wide = torch.empty_strided((1, 1, 4096, 128), (0, 0, 2**18, 1), dtype=torch.bfloat16,
                               device="meta")
    many = torch.empty(2**20, 1, 256, 128, dtype=torch.bfloat16, device="meta")
    assert not _backward_fits((wide,) * 5) and not _backward_fits((many,) * 5)
