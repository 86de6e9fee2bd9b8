"""Workspace sizes: one sized for a call's longest sequence serves every shorter
one (and fewer heads, and no lists), as a caller that allocates once relies on."""
from __future__ import annotations

import ctypes

import pytest

from fftsparse_amd import _lib
from fftsparse_amd._lib import AttnArgs


def attn_bytes(L, bs, D=128, Hq=32, Hk=8, listed=True, Lq=None):
    args = AttnArgs(dtype=1, B=1, Hq=Hq, Hk=Hk, Lq=Lq or L, Lk=L, D=D, bs=bs, q_sl=D, k_sl=D, v_sl=D,
                    blk_cnt=4096 if listed else None, blk_bits=4096 if listed else None)
    return _lib.load().fs_bsattn_work_bytes(ctypes.byref(args))


# around every length at which the attention takes another form, and between
LENGTHS = sorted({n + d for n in (1, 64, 960, 4096, 6144, 12288, 24576, 32768, 40960, 49152, 81920, 131072)
                  for d in (-1, 0, 1, 17, 129) if n + d > 0} | set(range(500, 140000, 2777)))


@pytest.mark.parametrize("bs", [16, 32, 64, 128])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hk", [(32, 8), (32, 32), (4, 1)])
def test_attention_workspace_grows_with_the_length(bs, D, Hq, Hk):
    n = [attn_bytes(L, bs, D, Hq, Hk) for L in LENGTHS]
    assert n == sorted(n)
    assert n[0] > 0
    for L, listed in zip(LENGTHS, n):
        assert attn_bytes(L, bs, D, Hq, Hk, listed=False) <= listed
        assert attn_bytes(L, bs, D, Hk, Hk) <= listed              # fewer query heads
    # fewer queries than keys
    for Lq in (1, 1000, 40000):
        n = [attn_bytes(L, bs, D, Hq, Hk, Lq=Lq) for L in LENGTHS]
        assert n == sorted(n)


@pytest.mark.parametrize("bs", [16, 128])
@pytest.mark.parametrize("tau", [0.0, 0.1])
def test_flexprefill_workspace_grows_with_length_and_heads(bs, tau):
    lib = _lib.load()
    lengths = [L for L in LENGTHS if bs < L <= 8192 * bs] + list(range(60000, 70000, 509))
    for Hq in (1, 4, 28, 32, 70, 512, 1024):
        n = [lib.fs_flex_work_bytes(Hq, 1, L, bs, tau) for L in sorted(lengths)]
        assert n == sorted(n)
    for L in (300, 4100, 33000, 65537):
        n = [lib.fs_flex_work_bytes(Hq, 1, L, bs, tau) for Hq in range(1, 1100, 3)]
        assert n == sorted(n)
