"""Attention that reads V as it is stored against attention through the V^T
pre-pass.  Both read the same values and add the same products in the same
order, so their outputs are equal bit for bit: a whole call against its two
halves, which always take the pre-pass, and against a V view whose row stride
passes the direct form's 32-bit offsets, which takes it too.  And the dense
calls by 64 and by 128 queries a workgroup."""
from __future__ import annotations

import pytest
import torch

from fftsparse_amd import AttentionCall, block_sparse_attention
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
    for value in (None, float("inf")):
        if value is not None:
            v[:, :, -1, 3] = value                   # reaches the rows that attend to it, as through V^T
        a = block_sparse_attention(q, k, v, **kw)
        call = AttentionCall(q, k, v, **kw)
        call.prepare()
        for b in [call.run()] + ([block_sparse_attention(q, k, _far(v), **kw)] if Lk <= 65 else []):
            assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())
            assert value is not None or not a.isnan().any()


@pytest.mark.parametrize("L,B", [(320, 1), (900, 1), (960, 4), (1100, 1)])
def test_dense_by_64_queries(L, B):
    """Dense calls of few workgroups (48, 128, 512 and 144 of 128 queries), which take 64 queries each."""
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(B, h, L, 128, generator=g).to(torch.bfloat16).to(DEV) for h in (16, 4, 4))
    o = block_sparse_attention(q, k, v).float().cpu()
    kf, vf = (t.float().cpu().repeat_interleave(4, 1) for t in (k, v))
    s = (q.float().cpu() @ kf.transpose(-1, -2)) * 128 ** -0.5
    s.masked_fill_(torch.ones(L, L, dtype=torch.bool).triu(1), float("-inf"))
    ref = (torch.softmax(s, -1) @ vf).transpose(1, 2)
    assert (o - ref).abs().max() < 2e-2


def _dense_reference(q, k, v, causal):
    """fp32 attention, head by head (products of matrices only)."""
    B, Hq, Lq, D = q.shape
    Hk, Lk = k.shape[1:3]
    out = torch.empty(B, Lq, Hq, D, device=DEV)
    hidden = torch.arange(Lk, device=DEV)[None] > torch.arange(Lq, device=DEV)[:, None] + Lk - Lq
    for b in range(B):
        for h in range(Hq):
            kt = k[b, h // (Hq // Hk)].float().T.contiguous()
            s = q[b, h].float() @ kt * D ** -0.5
            if causal:
                s.masked_fill_(hidden, float("-inf"))
            out[b, :, h] = torch.softmax(s, -1) @ v[b, h // (Hq // Hk)].float()
    return out


@pytest.mark.parametrize("B,Hq,Hk,Lq,Lk,bs,D,dtype,causal,rise", [
    (4, 32, 8, 1200, 1200, 128, 128, torch.bfloat16, True, 0.0),       # V in place, 1280 workgroups
    (1, 32, 4, 4097, 4097, 128, 128, torch.bfloat16, True, 0.0),       # through V^T, one query past a block
    (4, 32, 8, 512, 512, 128, 128, torch.float16, True, 0.0),          # 512 workgroups of short sequences
    (2, 32, 8, 1111, 1111, 128, 64, torch.bfloat16, True, 30.0),       # head dim 64: no row max, scores that rise
    (2, 32, 8, 1111, 1111, 32, 64, torch.float16, True, 3000.0),
    (1, 32, 2, 2100, 2100, 128, 64, torch.bfloat16, False, 30.0),      # through V^T, not causal
    (1, 40, 8, 2100, 2333, 128, 128, torch.bfloat16, True, 30.0),      # fewer queries than keys
    (1, 40, 2, 1900, 2333, 16, 128, torch.float16, False, -30.0),
])
def test_dense_by_128_queries(B, Hq, Hk, Lq, Lk, bs, D, dtype, causal, rise):
    """Dense calls of more workgroups of 128 queries than take 64 each, whatever the block size but 64."""
    groups = B * Hq * -(-Lq // 128)
    assert groups > 512 or (groups > 384 and Lk < 960)
    print(f"[case] dense by 128: B={B} {Hq}/{Hk} Lq={Lq} Lk={Lk} D={D} {dtype} causal={causal}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(Lq + D)
    u = torch.nn.functional.normalize(torch.randn(D, generator=g, device=DEV), dim=0)
    q = torch.randn(B, Hq, Lq, D, generator=g, device=DEV) + (10.0 * u if rise else 0.0)
    k = torch.randn(B, Hk, Lk, D, generator=g, device=DEV)
    k += (torch.arange(Lk, device=DEV) / Lk * rise)[:, None] * u
    v = torch.randn(B, Hk, Lk, D, generator=g, device=DEV)
    q, k, v = (x.to(dtype) for x in (q, k, v))
    out = block_sparse_attention(q, k, v, block_size=bs, is_causal=causal).float()
    assert (out - _dense_reference(q, k, v, causal)).abs().max() < 2e-2


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
