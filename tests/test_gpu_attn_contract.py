"""What a caller of the attention may rely on besides its result: the two halves
of the call (prepare stages V, run reads what was staged), an output that takes
V's place, any stride of V, and large values."""
from __future__ import annotations

import math

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


@pytest.mark.parametrize("D,bs,listed", [(64, 128, False), (64, 128, True), (64, 32, True), (64, 16, True),
                                         (128, 128, False), (128, 32, True), (128, 16, True), (128, 128, True)])
def test_large_values_under_rising_scores(D, bs, listed):
    """Scores that rise along the keys by a factor of 2^55 in weight, values near 2^100: the output is
    a mean of values, and the sums behind it stay finite too."""
    L, H = 1000, 2
    u = torch.nn.functional.normalize(torch.randn(D, generator=torch.Generator().manual_seed(D)), dim=0)
    rise = torch.arange(L) / L * 55.0 * math.log(2.0) * D ** 0.5 / 8.0
    q = (8.0 * u).expand(1, H, L, D).bfloat16().contiguous()
    k = (rise[:, None] * u).expand(1, H, L, D).bfloat16().contiguous()
    v = torch.randn(1, H, L, D, generator=torch.Generator().manual_seed(1)).bfloat16() * 2.0 ** 100
    n = -(-L // bs)
    lists = bits_from_mask(torch.ones(H, n, n, dtype=torch.bool)) if listed else (None, None)
    out = block_sparse_attention(q.to(DEV), k.to(DEV), v.to(DEV), *(x.to(DEV) if listed else x for x in lists),
                                 block_size=bs).double().cpu()
    s = (q.double() @ k.double().transpose(-1, -2)) * D ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    ref = (torch.softmax(s, -1) @ (v.double() * 2.0 ** -100)).transpose(1, 2)
    assert out.isfinite().all()
    assert (out * 2.0 ** -100 - ref).abs().max() < 2e-2
