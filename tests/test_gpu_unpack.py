"""``unpack`` of the packed state at every alignment: 16-byte vectors where all three pointers
allow them (from 2^17 bytes on), with a tail of n % 16 bytes, and byte by byte otherwise. Exact."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4096, 100_003, 2**17 - 1, 2**17, 2**17 + 15])
@pytest.mark.parametrize("offset", [0, 1, 16])
def test_unpack_matches_the_nibbles(cuda, n, offset):
    from local_ai_training import _native as nat

    gen = torch.Generator(device=cuda).manual_seed(n)
    packed = torch.randint(0, 256, (n + offset,), generator=gen, device=cuda,
                           dtype=torch.uint8)[offset:]
    for max_code in (1, 7):
        code = torch.full((n + 32,), 99, device=cuda, dtype=torch.int8)
        pressure = code.clone()
        for c, p in ((code, pressure), (code, None), (None, pressure)):
            nat.call("rk_unpack", packed.data_ptr(), ctypes.c_int64(n), max_code, nat.ptr(c),
                     nat.ptr(p), nat.stream_handle(packed.device))
        wide = packed.to(torch.int16)
        assert torch.equal(code[:n], ((wide & 15) - max_code).to(torch.int8))
        assert torch.equal(pressure[:n], ((wide >> 4) - 7).to(torch.int8))
        assert bool((code[n:] == 99).all()) and bool((pressure[n:] == 99).all())
