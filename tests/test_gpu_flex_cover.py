"""The sparse heads' block-level attention and cover of FlexPrefill, every head
made sparse (tau above any divergence), at the block counts where its tiles of
32 rows and keys end: one partial tile, whole tiles, one row past a tile, rows of
no multiple of four blocks, and lengths that end inside a block; and the last
block's passes at the chunk counts of short and long sequences.  Blocks equal the
oracle's for >= 99.9% of the causal decisions (a tie of rounded scores at the
cut's boundary may fall otherwise)."""
from __future__ import annotations

import pytest
import torch

from fftsparse_amd.flex import flex_select
from fftsparse_amd.synth import make_qkv
from oracle import flex as oflex

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("L,bs,Hq,Hk,dtype,tau", [
    (70, 16, 2, 1, torch.bfloat16, 10.0), (512, 16, 4, 2, torch.float16, 10.0), (1056, 32, 2, 1, torch.bfloat16, 10.0),
    (1000, 32, 4, 1, torch.bfloat16, 10.0), (2047, 64, 2, 2, torch.bfloat16, 10.0), (4100, 128, 2, 1, torch.float16, 10.0),
    (2090, 16, 2, 1, torch.bfloat16, 10.0), (4300, 32, 1, 1, torch.bfloat16, 0.0), (4300, 128, 70, 1, torch.bfloat16, 0.0),
])
def test_cover_and_profiles_against_oracle(L, bs, Hq, Hk, dtype, tau):
    q, k, _ = make_qkv(L, Hq, Hk, dtype=dtype, seed=L + bs)
    qt, kt = q.transpose(1, 2), k.transpose(1, 2)
    ref = oflex.active_blocks(qt, kt, bs, 0.9, tau)
    sel = flex_select(qt.to(DEV), kt.to(DEV), gamma=0.9, tau=tau, block_size=bs)
    assert bool(sel.head_info[:, 2].all()) == (tau > 0)
    got = sel.dense_mask().cpu()
    n = got.shape[1]
    tri = torch.ones(n, n, dtype=torch.bool).tril()
    assert not bool((got & ~tri).any())
    assert (sel.vertical.cpu() - ref.vertical_t).abs().sum(-1).max() < 2e-5
    assert (sel.slash.cpu() - ref.slash_t).abs().sum(-1).max() < 2e-5
    same = (got == ref.mask)[:, tri].float().mean().item()
    print(f"L={L} bs={bs} Hq={Hq}: equal {same:.6f} of {Hq * int(tri.sum())} decisions", flush=True)
    assert same >= 0.999


@pytest.mark.parametrize("dims", [(0, 1), (0, 8), (0, 64)])
@pytest.mark.parametrize("row,key", [(9, 4), (4, 4), (9, 9)])
def test_score_past_the_float_range_spoils_its_whole_row(dims, row, key):
    """A block score that leaves the float range (two dims of a query block and of a key block whose
    products cancel) makes every probability of its row nan: the cover takes none of it, wherever in
    the row the score lies, and the other rows as ever."""
    n, bs, H = 12, 16, 1
    q, k, _ = make_qkv(n * bs, H, H, dtype=torch.bfloat16, seed=bs)
    qt, kt = q.transpose(1, 2).contiguous(), k.transpose(1, 2).contiguous()
    qt[..., list(dims)] = 0.0
    kt[..., list(dims)] = 0.0
    qt[:, row * bs:(row + 1) * bs, :, list(dims)] = 1e30
    kt[:, key * bs:(key + 1) * bs, :, dims[0]] = 1e30
    kt[:, key * bs:(key + 1) * bs, :, dims[1]] = -1e30
    sel = flex_select(qt.to(DEV), kt.to(DEV), gamma=0.9, tau=10.0, block_size=bs)
    assert int(sel.head_info[0, 2]) == 1
    got = sel.dense_mask().cpu()[0]
    assert torch.nonzero(got[row]).flatten().tolist() == [0, row]
    assert got.sum() > 2 * n
