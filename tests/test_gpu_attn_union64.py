"""Attention over 16- and 32-token block lists in groups of 64 and of 128 queries:
lengths at the edges of a group, entries selected by one row of a group only,
rows that select nothing, and the length at which the group size changes."""
import pytest
import torch

import fftsparse_amd
from fftsparse_amd.attn import bits_from_mask

pytestmark = pytest.mark.gpu


def reference(q, k, v, mask, bs, rows):
    """fp32 attention of the given query rows; a row that selects no key is 0."""
    G = q.shape[1] // k.shape[1]
    L, D = q.shape[2:]
    kf, vf = k[0].float().repeat_interleave(G, 0), v[0].float().repeat_interleave(G, 0)
    s = torch.stack([q[0, h, rows].float() @ kf[h].T.contiguous() for h in range(q.shape[1])]) / D ** 0.5
    j = torch.arange(L, device=q.device)
    keep = mask[:, rows // bs][:, :, j // bs] & (j[None] <= rows[:, None])[None]
    p = torch.nan_to_num(torch.softmax(s.masked_fill(~keep, float("-inf")), -1))
    return torch.stack([p[h] @ vf[h] for h in range(q.shape[1])])


@pytest.mark.parametrize("L,bs,D,density,dtype", [
    (64, 32, 128, 0.6, torch.bfloat16),           # one group
    (65, 16, 128, 0.6, torch.float16),            # one row past a group
    (127, 16, 64, 0.5, torch.bfloat16),           # head dim 64: groups of 128
    (129, 16, 128, 0.5, torch.bfloat16),
    (700, 32, 128, 0.05, torch.float16),          # entries of one row, empty rows
    (1999, 16, 128, 0.02, torch.bfloat16),
    (1025, 32, 128, 1.0, torch.bfloat16),
    (40960, 32, 128, 0.02, torch.bfloat16),       # the last length in groups of 64
    (40961, 32, 128, 0.02, torch.bfloat16),       # the first in groups of 128
    (32769, 16, 128, 0.01, torch.bfloat16),       # likewise at 16-token blocks
])
def test_union_groups(L, bs, D, density, dtype):
    print(f"[case] union groups L={L} bs={bs} D={D} density={density} {dtype}", flush=True)
    Hq, Hk = 4, 2
    g = torch.Generator(device="cuda").manual_seed(L + bs)
    q, k, v = (torch.randn(1, h, L, D, generator=g, device="cuda").to(dtype) for h in (Hq, Hk, Hk))
    N = -(-L // bs)
    mask = torch.rand(Hq, N, N, generator=g, device="cuda") < density
    mask[:, 1::5] = False                          # rows that select nothing
    cnt, bits = bits_from_mask(mask)
    out = fftsparse_amd.block_sparse_attention(q, k, v, cnt, bits, block_size=bs)
    out = out.view(L, Hq, D).transpose(0, 1).float()
    rows = torch.arange(L, device="cuda")
    if L > 4096:
        rows = torch.cat([rows[:130], rows[::613], rows[-130:]])
    ref = reference(q, k, v, mask, bs, rows)
    got = out[:, rows]
    # P and the output are rounded to the 16-bit type: each entry of P to 2^-9 (bf16)
    # of itself, so a row errs by 2^-9 max |V| (about 5) at most, and its store by 2^-9 |out|
    eps = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    assert (got - ref).abs().max().item() <= 2 * eps * v.float().abs().max().item()
    empty = ~mask.any(-1)[:, rows // bs]
    assert (got[empty] == 0).all()


@pytest.mark.parametrize("Lk,bs", [(41003, 32), (32790, 16)])
@pytest.mark.parametrize("Lq,causal,density,dtype", [
    (700, True, 0.3, torch.float16), (333, False, 0.05, torch.bfloat16), (130, False, 1.0, torch.float16),
    (260, True, 1.0, torch.bfloat16),
])
def test_groups_of_128_at_head_dim_128(Lk, bs, Lq, causal, density, dtype):
    """Past the lengths of groups of 64: fewer queries than keys, not causal, full lists, both types."""
    print(f"[case] groups of 128 Lk={Lk} bs={bs} Lq={Lq} causal={causal} density={density} {dtype}", flush=True)
    Hq, D = 2, 128
    g = torch.Generator(device="cuda").manual_seed(Lq + bs)
    q, k, v = (torch.randn(1, h, n, D, generator=g, device="cuda").to(dtype) for h, n in ((Hq, Lq), (1, Lk), (1, Lk)))
    mask = torch.rand(Hq, -(-Lq // bs), -(-Lk // bs), generator=g, device="cuda") < density
    mask[:, 1::5] = False
    cnt, bits = bits_from_mask(mask)
    out = fftsparse_amd.block_sparse_attention(q, k, v, cnt, bits, block_size=bs, is_causal=causal)
    i, j = torch.arange(Lq, device="cuda"), torch.arange(Lk, device="cuda")
    for h in range(Hq):
        s = q[0, h].float() @ k[0, 0].float().T.contiguous() * D ** -0.5
        keep = mask[h][i // bs][:, j // bs]
        if causal:
            keep &= j[None] <= i[:, None] + Lk - Lq
        p = torch.nan_to_num(torch.softmax(s.masked_fill(~keep, float("-inf")), -1))
        eps = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
        assert (out[0, :, h].float() - p @ v[0, 0].float()).abs().max() <= 2 * eps * v.float().abs().max()
        assert (out[0, ~keep.any(-1), h] == 0).all()


@pytest.mark.parametrize("bs,D", [(32, 128), (16, 128), (32, 64), (16, 64)])
def test_rows_that_begin_late_or_far_below_zero(bs, D):
    """Rows whose first listed block comes after others' of the group (their first tiles hold no
    key of theirs), with scores of -800 to -2300: from a start above them they would all be 0."""
    L, H = 600, 2
    n = -(-L // bs)
    q = torch.full((1, H, L, D), 10.0, dtype=torch.bfloat16, device="cuda")
    k = (-10.0 * (2.0 - torch.arange(L, device="cuda") / L))[None, None, :, None].expand(1, 1, L, D).bfloat16()
    v = torch.randn(1, 1, L, D, generator=torch.Generator().manual_seed(bs)).bfloat16().cuda()
    r, c = torch.meshgrid(torch.arange(n), torch.arange(n), indexing="ij")
    mask = ((c >= r - r % 3) & (c <= r)).repeat(H, 1, 1)      # rows of a group begin 0, 1 or 2 blocks back
    mask[1] &= (c == r)                                       # and the second head's at their own block
    mask[:, 1::7] = False
    cnt, bits = (t.cuda() for t in bits_from_mask(mask))
    out = fftsparse_amd.block_sparse_attention(q, k.contiguous(), v, cnt, bits, block_size=bs)
    j = torch.arange(L)
    keep = mask[:, j // bs][:, :, j // bs] & (j[None] <= j[:, None])[None]
    s = (q[0].double().cpu() @ k[0].double().cpu().expand(H, -1, -1).transpose(1, 2)) / D ** 0.5
    p = torch.nan_to_num(torch.softmax(s.masked_fill(~keep, float("-inf")), -1))
    ref = p @ v[0].double().cpu().expand(H, -1, -1)
    assert (out.view(L, H, D).transpose(0, 1).double().cpu() - ref).abs().max() <= 2.0 ** -8 * v.abs().max().item()
