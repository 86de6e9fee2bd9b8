"""The diffuse heads' rows of fs_select (score panel on MFMA, per-row top-k) at
the sizes where the panel's shape changes: one 64-block word and its
remainders, 16, 8, 4 and 2 rows per panel (N up to 1024, 2048, 4096, 8192), the
last partial panel, head dims that fill part of an MFMA step, more heads than
one decision group holds, and q_b / k_b that allow no 16-byte loads.  Every
head is made diffuse (stripe_threshold 0); the bar is the selection tests':
exact or excused block decisions >= 99.9% of all causal decisions."""
from __future__ import annotations

import math

import pytest
import torch

from fftsparse_amd import _lib, select_blocks
from fftsparse_amd._lib import SelectArgs
from fftsparse_amd.synth import make_qkv
from oracle import v7
from tests.helpers import MATCH_MIN, block_match

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("N,Hq,Hk,D,dtype", [
    (12, 2, 1, 128, torch.bfloat16), (64, 2, 1, 128, torch.bfloat16), (65, 2, 1, 64, torch.float16),
    (300, 3, 1, 128, torch.float32), (130, 2, 2, 24, torch.float32), (130, 2, 2, 40, torch.bfloat16),
    (200, 70, 1, 64, torch.bfloat16), (140, 2, 1, 256, torch.bfloat16),
    (1024, 1, 1, 128, torch.bfloat16), (1033, 1, 1, 128, torch.bfloat16), (2061, 1, 1, 64, torch.float16),
    (4099, 1, 1, 32, torch.bfloat16),
])
def test_diffuse_rows_against_oracle(N, Hq, Hk, D, dtype):
    bs = 8
    L = N * bs - 3                                   # the last block is partial
    q, k, _ = make_qkv(L, Hq, Hk, D=D, dtype=dtype, seed=N)
    kw = dict(block_size=bs, stripe_threshold=0.0, qk_topk_ratio=0.3, sink_ratio=0.01, recent_ratio=0.0,
              local_span_ratio=0.02, corr_threshold=0.9, column_topk_ratio=0.2)
    ref = v7.select_mask(q, k, **kw)
    assert not bool(ref.is_stripe.any())
    sel = select_blocks(q.to(DEV), k.to(DEV), **kw)
    got = sel.dense_mask().cpu()
    assert torch.equal(sel.blk_cnt.cpu(), got.sum(-1, dtype=torch.int32))
    frac, exact, unexc = block_match(got, ref.mask, ref.excusable)
    print(f"N={N} D={D} {dtype}: match={frac:.6f} exact={exact:.6f} unexcused={unexc}", flush=True)
    assert frac >= MATCH_MIN


def _topk_rows(q_b, k_b, N, D, dtype, ratio=0.3):
    """fs_select's diffuse rows alone (no sink, window, columns or last row)."""
    H = q_b.shape[0]
    cnt = torch.empty(H, N, dtype=torch.int32, device=DEV)
    bits = torch.empty(H, N, (N + 63) // 64, dtype=torch.int64, device=DEV)
    keep = torch.zeros(H, N, dtype=torch.uint8, device=DEV)
    _lib.call("fs_select", SelectArgs(
        q_b=q_b.data_ptr(), k_b=k_b.data_ptr(), dtype=_lib.FS_DTYPE[dtype], Hq=H, Hk=H, N=N, Nk=N, D=D, mask_causal=1,
        keep_sink=0, keep_recent=0, local_window=0, remote_start=1, dyn_mode=1, stripe_all_diffuse=1,
        keep_tau=keep.data_ptr(), qk_topk_ratio=ratio, col_mode=0, blk_cnt=cnt.data_ptr(), blk_bits=bits.data_ptr()),
        DEV)
    return cnt, bits


@pytest.mark.parametrize("D", [128, 20])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_that_allow_no_wide_loads(D, dtype):
    """Block means at an odd element, or rows that are no multiple of 16 bytes,
    select what aligned copies padded with zeros select (the same products, in
    the same order, so the same bits; 1/sqrt(D) differs, and only scales)."""
    N, H = 150, 2
    g = torch.Generator().manual_seed(D)
    x = [torch.randn(H, N, D, generator=g).to(dtype) for _ in range(2)]
    pad = -D % 8
    wide = [torch.nn.functional.pad(t, (0, pad)).to(DEV).contiguous() for t in x]
    odd = []
    for t in x:
        buf = torch.empty(t.numel() + 1, dtype=dtype, device=DEV)
        buf[1:] = t.flatten().to(DEV)
        odd.append(buf[1:].view(H, N, D))
    assert odd[0].data_ptr() % 16 != 0
    ca, ba = _topk_rows(*wide, N, D + pad, dtype)
    cb, bb = _topk_rows(*odd, N, D, dtype)
    assert torch.equal(ca, cb) and torch.equal(ba, bb)
    k = [max(1, math.trunc(float(torch.tensor(float(i + 1)) * torch.tensor(0.3)))) for i in range(N)]
    assert ca.cpu().tolist() == [k] * H


def test_ties_at_the_threshold_go_to_the_lower_block():
    N, H, D = 200, 1, 64
    q = torch.ones(H, N, D, dtype=torch.bfloat16, device=DEV)
    k = torch.ones(H, N, D, dtype=torch.bfloat16, device=DEV)
    k[:, 5] = 2.0                                    # one larger score; every other one ties
    cnt, bits = _topk_rows(q, k, N, D, torch.bfloat16)
    from fftsparse_amd.attn import mask_from_bits
    m = mask_from_bits(bits, N)[0].cpu()
    for i in range(N):
        want = max(1, math.trunc(float(torch.tensor(float(i + 1)) * torch.tensor(0.3))))
        order = sorted(range(i + 1), key=lambda j: (j != 5, j))[:want]
        assert sorted(order) == torch.nonzero(m[i]).flatten().tolist()


@pytest.mark.parametrize("diffuse", [True, False])
@pytest.mark.parametrize("window", [2**31 - 1, 2**31 - 150, 199])
def test_window_wider_than_the_sequence(diffuse, window):
    """A local window that no sequence is long for selects every block up to the diagonal."""
    N = 200
    q_b = torch.randn(1, N, 64, generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
    cnt = torch.empty(1, N, dtype=torch.int32, device=DEV)
    bits = torch.empty(1, N, (N + 63) // 64, dtype=torch.int64, device=DEV)
    keep = torch.zeros(1, N, dtype=torch.uint8, device=DEV)
    var = torch.zeros(1, 1, device=DEV)
    _lib.call("fs_select", SelectArgs(
        q_b=q_b.data_ptr(), k_b=q_b.data_ptr(), dtype=_lib.FS_DTYPE[torch.bfloat16], Hq=1, Hk=1, N=N, Nk=N, D=64,
        mask_causal=1, keep_sink=0, keep_recent=0, local_window=window, remote_start=1, dyn_mode=1,
        stripe_all_diffuse=int(diffuse), diag_var=var.data_ptr(), n_samples=1, stripe_threshold=1.0,
        keep_tau=keep.data_ptr(), qk_topk_ratio=0.1, col_mode=0, blk_cnt=cnt.data_ptr(), blk_bits=bits.data_ptr()),
        DEV)
    assert cnt[0].cpu().tolist() == list(range(1, N + 1))
