"""Attention that reads V as it is stored against attention through the V^T
pre-pass.  Both read the same values and add the same products in the same
order, so their outputs are equal bit for bit; a V view whose row stride
passes the direct form's 32-bit offsets takes the pre-pass, which gives the
same call both ways."""
from __future__ import annotations

import pytest
import torch

from fftsparse_amd import block_sparse_attention
from fftsparse_amd.attn import bits_from_mask

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
FAR = 1 << 23                                        # row stride (elements) that the direct form does not take


def _far(v):
    """v's values in a view of row stride FAR (one KV head after another inside a row's gap)."""
    B, Hk, L, D = v.shape
    buf = torch.empty(L * FAR, dtype=v.dtype, device=v.device)
    out = buf.as_strided((B, Hk, L, D), (Hk * D, D, FAR, 1))
    out.copy_(v)
    return out


@pytest.mark.parametrize("Lk,Lq,bs,D,dtype,causal,listed", [
    (1, 1, 128, 128, torch.bfloat16, True, False), (64, 64, 64, 128, torch.bfloat16, True, True),
    (65, 65, 128, 128, torch.bfloat16, False, True), (100, 100, 64, 64, torch.float16, False, True),
    (500, 500, 128, 128, torch.float16, True, True), (447, 300, 128, 64, torch.bfloat16, True, True),
    (129, 129, 64, 128, torch.bfloat16, True, False), (500, 500, 32, 64, torch.bfloat16, True, False),
    (333, 77, 16, 128, torch.float16, True, False),
])
def test_direct_equals_transposed(Lk, Lq, bs, D, dtype, causal, listed):
    B, Hq, Hk = (1, 4, 2) if listed else (2, 4, 2)
    g = torch.Generator().manual_seed(Lk * D + bs)
    q, k, v = (torch.randn(B, h, n, D, generator=g).to(dtype).to(DEV) for h, n in ((Hq, Lq), (Hk, Lk), (Hk, Lk)))
    kw = dict(block_size=bs, is_causal=causal)
    if listed:
        mask = torch.rand(Hq, -(-Lq // bs), -(-Lk // bs), generator=g) < 0.6
        kw["blk_cnt"], kw["blk_bits"] = (t.to(DEV) for t in bits_from_mask(mask))
    a, b = block_sparse_attention(q, k, v, **kw), block_sparse_attention(q, k, _far(v), **kw)
    assert torch.equal(a, b)
    # an infinite last value row reaches the rows that attend to it, as through V^T
    v[:, :, -1, 3] = float("inf")
    a, b = block_sparse_attention(q, k, v, **kw), block_sparse_attention(q, k, _far(v), **kw)
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("L,B", [(320, 1), (900, 1), (960, 4), (1100, 1)])
def test_dense_by_64_queries(L, B):
    """Dense calls below and above the workgroup counts at which they take 64 queries a workgroup."""
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(B, h, L, 128, generator=g).to(torch.bfloat16).to(DEV) for h in (16, 4, 4))
    o = block_sparse_attention(q, k, v).float().cpu()
    kf, vf = (t.float().cpu().repeat_interleave(4, 1) for t in (k, v))
    s = (q.float().cpu() @ kf.transpose(-1, -2)) * 128 ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    ref = (torch.softmax(s, -1) @ vf).transpose(1, 2)
    assert (o - ref).abs().max() < 2e-2


@pytest.mark.parametrize("growth", [30.0, 3000.0, -3000.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq", [2, 32])
def test_head_dim_64_running_max(growth, dtype, Hq):
    """Head dim 64 takes its exponentials against the running max with no row
    max: scores that rise or fall along the keys, far past the range of a 16-bit
    probability, direct (2 heads) and through V^T (32 heads on one KV head)."""
    L, D = 1600, 64
    g = torch.Generator().manual_seed(12)
    u = torch.randn(D, generator=g)
    u /= u.norm()
    q = torch.randn(1, Hq, L, D, generator=g) + 10.0 * u
    k = torch.randn(1, 1, L, D, generator=g) + (torch.arange(L, dtype=torch.float32) / L * growth)[:, None] * u
    v = torch.randn(1, 1, L, D, generator=g)
    q, k, v = (x.to(dtype) for x in (q, k, v))
    s = (q.float() @ k.float().transpose(-1, -2)) * D ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    ref = (torch.softmax(s, -1) @ v.float()).transpose(1, 2)
    qd, kd, vd = (x.to(DEV) for x in (q, k, v))
    assert (block_sparse_attention(qd, kd, vd).float().cpu() - ref).abs().max() < 2e-2
    for bs in (128, 64, 32):
        n = -(-L // bs)
        mask = torch.ones(Hq, n, n, dtype=torch.bool).tril()
        cnt, bits = (t.to(DEV) for t in bits_from_mask(mask))
        assert (block_sparse_attention(qd, kd, vd, cnt, bits, block_size=bs).float().cpu() - ref).abs().max() < 2e-2
