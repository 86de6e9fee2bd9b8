"""What a caller of the attention may rely on besides its result: the two halves
of the call (prepare stages V, run reads what was staged), an output that takes
V's place, and any stride of V."""
from __future__ import annotations

import pytest
import torch

from fftsparse_amd import AttentionCall, block_sparse_attention
from fftsparse_amd.attn import bits_from_mask

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _qkv(L, Hq, Hk, D=128, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(1, h, L, D, generator=g).to(dtype).to(DEV) for h in (Hq, Hk, Hk)]


def _lists(Hq, L, bs, density, seed=0):
    n = -(-L // bs)
    mask = torch.rand(Hq, n, n, generator=torch.Generator().manual_seed(seed)) < density
    return [t.to(DEV) for t in bits_from_mask(mask)]


@pytest.mark.parametrize("L,bs,listed", [(700, 128, False), (333, 32, False), (1500, 128, True), (1000, 64, True),
                                         (900, 32, True)])
def test_run_reads_v_as_it_was_prepared(L, bs, listed):
    q, k, v = _qkv(L, 4, 2, seed=L)
    lists = _lists(4, L, bs, 0.6) if listed else (None, None)
    ref = block_sparse_attention(q, k, v, *lists, block_size=bs)
    call = AttentionCall(q, k, v, *lists, block_size=bs)
    call.prepare()
    v.fill_(float("nan"))
    assert torch.equal(call.run(), ref)


@pytest.mark.parametrize("listed", [False, True])
def test_prepare_serves_every_query_head_count(listed):
    """2 and 64 query heads on the same 2 KV heads and workspace: few and many uses of V."""
    L, Hk = 2100, 2
    q, k, v = _qkv(L, 64, Hk, seed=3)
    lists = [_lists(h, L, 128, 0.5) if listed else (None, None) for h in (Hk, 64)]
    few = AttentionCall(q[:, :Hk], k, v, *lists[0])
    many = AttentionCall(q, k, v, *lists[1])
    ref = block_sparse_attention(q, k, v, *lists[1])
    many.work.zero_()
    few.args.work = many.args.work
    few.prepare()
    assert torch.equal(many.run(), ref)


@pytest.mark.parametrize("L,bs,listed", [(700, 128, False), (2000, 128, False), (3000, 128, True), (2500, 64, True),
                                         (1500, 32, True)])
def test_output_may_take_the_place_of_v(L, bs, listed):
    q, k, v = _qkv(L, 16, 16, seed=L)
    lists = _lists(16, L, bs, 0.7) if listed else (None, None)
    ref = block_sparse_attention(q, k, v, *lists, block_size=bs)
    for shift in (0, 64 * 128):                      # v's own storage, and rows that meet it in part
        buf = torch.zeros(shift + v.numel(), dtype=v.dtype, device=DEV)
        buf[shift:] = v.transpose(1, 2).reshape(-1)
        out = buf[:v.numel()].view(1, L, 16, 128)
        got = block_sparse_attention(q, k, buf[shift:].view(1, L, 16, 128).transpose(1, 2), *lists, block_size=bs,
                                     out=out)
        assert torch.equal(got, ref)


@pytest.mark.parametrize("step", [-1, 0])
@pytest.mark.parametrize("listed", [False, True])
def test_v_rows_in_descending_order_or_repeated(listed, step):
    """Row strides of V that a C caller may give (torch has no negative ones)."""
    L, H, D = 300, 2, 128
    q, k, v = _qkv(L, H, H, seed=9)
    lists = _lists(H, L, 64, 0.7) if listed else (None, None)
    ref = block_sparse_attention(q, k, (v.flip(2) if step else v[:, :, :1].expand(-1, -1, L, -1)).contiguous(), *lists,
                                 block_size=64)
    call = AttentionCall(q, k, v, *lists, block_size=64)
    if step:
        call.args.v += 2 * (L - 1) * D               # each head's last row first
    call.args.v_sl = step * D
    assert torch.equal(call(), ref)
