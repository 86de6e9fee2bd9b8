"""What a user of fftsparse_amd has it do, as cases that can be timed and compared.

Every case is one call of a public entry point on tensors that a prefill has in
hand on the GPU: the FFTSparse v7 prefill at the lengths the reference reports
(8K to 128K) and below its dense limit, its other block size, head dim and data
type, the prefill with the rotary embedding fused into the block pooling, the
fixed mask, the two comparison selectors (XAttention, FlexPrefill), and the
selection alone in fp32.  Head counts are those of the benchmark configurations
(32 / 8, 28 / 4, 4 / 1).

The inputs follow the recipe of ``fftsparse_amd.synth`` (Gaussian Q/K/V, RoPE,
attention sinks, vertical stripes, a periodic pair), with what captured Q/K
show besides: queries that lean towards the sinks and stripes, and, in one
query head of four, a topic per segment of tokens, which makes it one of the
heads without diagonal structure ("diffuse").
"""
from __future__ import annotations

import math

import numpy as np
import torch

import fftsparse_amd
from fftsparse_amd import fix_mask, flex, xattn
from fftsparse_amd.hf import PRODUCTION_KWARGS

# The settings of the reference's efficiency runs, threshold 0.9, without the block size.
V7 = {k: v for k, v in PRODUCTION_KWARGS.items() if k != "block_size"}
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# Largest Hq * L * L for which exact() forms the attention in 64 bits (about 10 seconds).
EXACT_SCORES = 28 * 65536 * 65536


def _case(name, path, L, Hq, Hk, *, D=128, bs=128, dtype="bf16", B=1, layout="blhd", threshold=0.9, stride=8, tau=0.1):
    c = dict(path=path, L=L, Hq=Hq, Hk=Hk, D=D, bs=bs, dtype=dtype, B=B, layout=layout, threshold=threshold,
             stride=stride, tau=tau)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a prompt below ten blocks: the dense path, where launches and one wave of workgroups count
        _case("short-1k", "v7", 1000, 32, 8),
        # several such prompts at once
        _case("short-batch4", "v7", 1200, 32, 8, B=4, layout="bhld"),
        # the reference's shortest reported length, called as the reference calls it: K/V repeated to the query heads
        _case("v7-8k-repeated", "v7", 8192, 32, 32, layout="bhld"),
        # the benchmark's 32K layer, in the layout of a model's projections
        _case("v7-32k", "v7", 32768, 32, 8),
        # 64-token blocks (28 / 4 heads), a length that is no multiple of anything
        _case("v7-60k-block64", "v7", 60001, 28, 4, bs=64, layout="bhld"),
        # head dim 64 in fp16, ragged
        _case("v7-20k-d64-f16", "v7", 20333, 32, 8, D=64, dtype="f16"),
        # the headline: one 128K layer
        _case("v7-128k", "v7", 131072, 32, 8, layout="bhld"),
        # the patched model's prefill: rotary embedding and pooling in one pass, then the selection and the attention
        _case("rope-24k", "rope", 24571, 32, 8),
        # the fixed sink / recent / local mask
        _case("fixed-16k", "fixed", 16384, 32, 8),
        # the comparison selectors at the benchmark's settings
        _case("xattn-32k", "xattn", 32768, 32, 8, layout="bhld"),
        _case("flex-32k", "flex", 32768, 32, 8, bs=32, threshold=0.95),
        # the block mask alone from fp32 states (the smallest benchmark configuration): launches and latency
        _case("select-8k-f32", "select", 8192, 4, 1, dtype="f32", layout="bhld"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["v7", "v7", "v7", "short", "rope", "fixed", "xattn", "flex", "select"])
    Hq, Hk = rng.choice([(32, 8), (32, 8), (28, 4), (32, 32), (16, 2)])
    layout = rng.choice(["blhd", "bhld"])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if path == "short":
        return _case(None, "v7", _log(rng, 128, 1279), Hq, Hk, dtype=dtype, B=rng.choice([1, 1, 2, 4]), layout=layout)
    if path == "v7":
        D = rng.choice([128, 128, 128, 64])
        bs = rng.choice([128, 128, 128, 64])
        return _case(None, "v7", _log(rng, 4096, 98304), Hq, Hk, D=D, bs=bs, dtype=dtype, layout=layout,
                     threshold=rng.choice([0.9, 0.9, 0.8, 0.95]))
    if path == "rope":
        return _case(None, "rope", _log(rng, 4096, 65536), Hq, Hk, dtype=dtype, layout="blhd")
    if path == "fixed":
        return _case(None, "fixed", _log(rng, 2048, 32768), Hq, Hk, dtype=dtype, layout=layout)
    if path == "xattn":
        return _case(None, "xattn", _log(rng, 4096, 40000), Hq, Hk, dtype=dtype, layout=layout,
                     threshold=rng.choice([0.8, 0.9]), stride=rng.choice([8, 8, 16, 4]))
    if path == "flex":
        return _case(None, "flex", _log(rng, 4096, 40000), Hq, Hk, bs=rng.choice([32, 32, 64, 128, 16]), dtype=dtype,
                     layout="blhd", threshold=rng.choice([0.9, 0.95]), tau=rng.choice([0.1, 0.0]))
    return _case(None, "select", _log(rng, 4096, 131072), *rng.choice([(4, 1), (32, 8)]), dtype=rng.choice(["f32", "bf16"]),
                 layout=layout)


# ---- inputs -----------------------------------------------------------------

def _cos_sin(L, D, device, theta=500000.0):
    inv = 1.0 / (theta ** (torch.arange(0, D, 2, device=device, dtype=torch.float64) / D))
    ang = torch.arange(L, device=device, dtype=torch.float64)[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], -1)
    return ang.cos().float(), ang.sin().float()


def _unit(g, *shape):
    x = torch.randn(*shape, generator=g, device="cuda")
    return x / x.norm(dim=-1, keepdim=True)


def _states(case, seed):
    """q [B,Hq,L,D], k and v [B,Hk,L,D] in the case's dtype and layout; K/V heads
    beyond the eight of the model's are repeated ones, as repeat_kv makes them."""
    B, L, Hq, Hk, D = (case[n] for n in ("B", "L", "Hq", "Hk", "D"))
    G = max(1, Hq // 8) if Hk == Hq and Hq > 8 else Hq // Hk          # query heads per KV head of the model
    Hkv = Hq // G
    dt = DTYPES[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    cos, sin = _cos_sin(L, D, "cuda")
    n_str = max(1, round(0.01 * L))
    seg, topics = 512, 16
    n_seg = -(-L // seg)
    out = ([], [], [])
    for _ in range(B):
        u = _unit(g, Hkv, D)                                           # sink / stripe direction
        ea = _unit(g, Hkv, D)
        eb = torch.randn(Hkv, D, generator=g, device="cuda")
        eb = eb - (eb * ea).sum(-1, keepdim=True) * ea
        eb = eb / eb.norm(dim=-1, keepdim=True)
        ts = _unit(g, Hkv, topics, D)
        kz = torch.randint(topics, (Hkv, n_seg), generator=g, device="cuda")
        qz = torch.randint(topics, (Hq, n_seg), generator=g, device="cuda")
        pos = torch.randperm(L, generator=g, device="cuda")[:n_str]
        ang = 2.0 * math.pi * torch.arange(L, device="cuda") / (512 if L >= 100000 else 256)
        heads = torch.arange(Hq, device="cuda")
        lean = 1.0 + 3.0 * torch.rand(Hq, generator=g, device="cuda")
        token_seg = torch.arange(L, device="cuda") // seg

        def rope(x):
            if case["path"] == "rope":                                 # the path applies it
                return x
            h = D // 2
            return x * cos + torch.cat([-x[..., h:], x[..., :h]], -1) * sin

        q = rope(torch.randn(Hq, L, D, generator=g, device="cuda"))
        q += (lean[:, None] * u[heads // G])[:, None, :]
        for h in range(3, Hq, 4):                                      # the diffuse heads
            q[h] += 6.0 * ts[h // G][qz[h]][token_seg]
        k = rope(torch.randn(Hkv, L, D, generator=g, device="cuda"))
        for h in range(Hkv):
            k[h] += 6.0 * ts[h][kz[h]][token_seg]
        k += 2.0 * (torch.cos(ang)[None, :, None] * ea[:, None, :] + torch.sin(ang)[None, :, None] * eb[:, None, :])
        k[:, pos] += 12.0 * u[:, None, :]
        k[:, :4] += 24.0 * u[:, None, :]
        v = torch.randn(Hkv, L, D, generator=g, device="cuda")
        for o, x, n in zip(out, (q, k, v), (Hq, Hk, Hk)):
            x = x.to(dt)
            o.append(x if x.shape[0] == n else x.repeat_interleave(n // x.shape[0], 0))
    res = []
    for xs in out:
        x = xs[0][None] if B == 1 else torch.stack(xs)
        if case["layout"] == "blhd":                                   # a projection's output, seen per head
            x = x.transpose(1, 2).contiguous().transpose(1, 2)
        res.append(x)
    return res


def prepare(case, seed):
    q, k, v = _states(case, seed)
    s = {"case": case, "q": q, "k": k, "v": v}
    if case["path"] == "rope":
        cos, sin = _cos_sin(case["L"], case["D"], "cuda")
        s["cos"], s["sin"] = cos.to(q.dtype), sin.to(q.dtype)
    return s


# ---- one pass ---------------------------------------------------------------

def run(s):
    c, q, k, v = s["case"], s["q"], s["k"], s["v"]
    kw = dict(V7, block_size=c["bs"], corr_threshold=c["threshold"])
    if c["path"] == "v7":
        return fftsparse_amd.myattn_prefill(q, k, v, 0, **kw)
    if c["path"] == "rope":
        # what the patched attention forward does: the rotated K goes into the cache
        qr, kr, q_b, k_b = fftsparse_amd.rope_pool(q, k, s["cos"], s["sin"], block_size=c["bs"])
        sel = fftsparse_amd.select_blocks(qr, kr, pooled=(q_b, k_b), **kw)
        o = fftsparse_amd.block_sparse_attention(qr, kr, v, sel.blk_cnt, sel.blk_bits, block_size=c["bs"])
        return o, kr
    if c["path"] == "fixed":
        return fix_mask.myattn_prefill(q, k, v, 0, block_size=c["bs"])
    if c["path"] == "xattn":
        return xattn.Xattention_prefill(q, k, v, c["stride"], threshold=c["threshold"])
    if c["path"] == "flex":
        return flex.Flexprefill_prefill(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), gamma=c["threshold"],
                                        tau=c["tau"], block_size=c["bs"])
    sel = fftsparse_amd.select_blocks(q, k, **kw)
    return {"cnt": sel.blk_cnt, "bits": sel.blk_bits, "corr_sum": sel.corr_sum, "col_mean": sel.col_mean,
            "last_scores": sel.last_scores, "mean_var": sel.mean_var}


# ---- work and tolerance -----------------------------------------------------

def _dense(c):
    return c["path"] == "v7" and c["L"] < 10 * c["bs"]


def _share(c):
    """About the share of the causal blocks that is selected on these inputs (measured)."""
    if _dense(c):
        return 1.0
    if c["path"] == "flex":
        return 0.55 if c["bs"] < 64 else 0.9
    return {"v7": 0.28, "rope": 0.24, "fixed": 0.28, "xattn": 0.8, "select": 0.0}[c["path"]]


def work(case):
    B, L, Hq, Hk, D, bs = (case[n] for n in ("B", "L", "Hq", "Hk", "D", "bs"))
    e = 4 if case["dtype"] == "f32" else 2
    N = -(-L // bs)
    if case["path"] == "select":
        return {"bytes": e * L * D * (Hq + Hk) + Hq * N * (N / 8 + 4), "flops": Hq * D * N * N + L * D * (Hq + Hk)}
    scores = Hq * L * L / 2
    flops = 4 * D * B * scores * _share(case)
    if case["path"] == "xattn":
        flops += 2 * D * scores / case["stride"]
    elif case["path"] == "flex":
        flops += 2 * D * Hq * bs * L
    return {"bytes": 2 * B * L * D * (2 * Hq + 2 * Hk + (Hk if case["path"] == "rope" else 0)), "flops": flops}


def tolerance(case):
    # 16-bit outputs of an attention with 16-bit probabilities; a selection that
    # decides one near-tie otherwise moves 64 or 128 rows of one head
    if _dense(case) or case["path"] == "fixed":
        return {"rel": 8e-3, "max": 0.1}
    if case["path"] == "select":
        # fp32 sums over up to 1024 block means (last scores rounded to the data
        # type); lags, columns and rows that tie to rounding
        return {"rel": 1e-5 if case["dtype"] == "f32" else 2e-3, "max": 2e-2, "differ": 5e-3}
    return {"rel": 8e-3, "max": 0.8}


# ---- 64 bits ----------------------------------------------------------------

def _attention64(q, k, v, mask, bs, causal=True):
    """[B, L, Hq, D] in 64 bits over the blocks of mask [Hq, N, N] (None: all)."""
    B, Hq, L, D = q.shape
    G = Hq // k.shape[1]
    out = torch.empty(B, L, Hq, D, dtype=torch.float64, device=q.device)
    step = 1024
    for b in range(B):
        for h in range(Hq):
            kt = k[b, h // G].double().T.contiguous()
            vd = v[b, h // G].double()
            for t0 in range(0, L, step):
                t1 = min(L, t0 + step)
                end = t1 if causal else L
                s = (q[b, h, t0:t1].double() / math.sqrt(D)) @ kt[:, :end]
                keep = torch.ones(t1 - t0, end, dtype=torch.bool, device=q.device)
                if mask is not None:
                    rows = torch.arange(t0, t1, device=q.device) // bs
                    cols = torch.arange(end, device=q.device) // bs
                    keep = mask[h][rows][:, cols]
                if causal:
                    keep = keep & (torch.arange(end, device=q.device)[None] <= torch.arange(t0, t1, device=q.device)[:, None])
                s.masked_fill_(~keep, -math.inf)
                out[b, t0:t1, h] = torch.softmax(s, -1) @ vd[:end]
    return out


def _means(x, bs):
    """Block means [H, N, D] of [H, L, D], the last block's over bs rows too, as the dtype holds them."""
    H, L, D = x.shape
    N = -(-L // bs)
    p = torch.zeros(H, N * bs, D, dtype=x.dtype, device=x.device)
    p[:, :L] = x
    m = torch.stack([p[h].double().view(N, bs, D).sum(1) / bs for h in range(H)])
    return m.to(x.dtype).double()


def _top(x, n):
    """[..., M] bool: the n largest of each row, ties to the lower index."""
    order = torch.sort(x, dim=-1, descending=True, stable=True).indices[..., :n]
    return torch.zeros(x.shape, dtype=torch.bool, device=x.device).scatter_(-1, order, True)


def _v7_mask64(q, k, bs, threshold):
    """The v7 block mask [Hq, N, N] and its statistics, from q [Hq,L,D], k [Hk,L,D]."""
    Hq, L, D = q.shape
    G = Hq // k.shape[0]
    N = -(-L // bs)
    dev = q.device
    sink = max(1, int(N * V7["sink_ratio"]))
    recent = max(1, int(N * V7["recent_ratio"]))
    lw = max(2, int(N * V7["local_span_ratio"])) // 2
    qb, kb = _means(q, bs), _means(k, bs).repeat_interleave(G, 0)
    S = torch.stack([qb[h] @ kb[h].T.contiguous() for h in range(Hq)])
    i = torch.arange(N, device=dev)
    lag = i[:, None] - i[None, :]
    causal = lag >= 0
    # lag sums and their post-processing
    sums = torch.zeros(Hq, N, dtype=torch.float64, device=dev)
    sums.scatter_add_(1, lag.clamp(min=0).flatten().expand(Hq, -1), (S * causal).flatten(1))
    corr = sums / (N - i).clamp(min=1)
    ex, st = lw + 1, N - sink - 5
    corr[:, :ex] = 0
    corr[:, st:] = 0
    if ex < st:
        w = torch.log10((N - i[ex:st]).double())
        corr[:, ex:st] = (corr[:, ex:st] - corr[:, ex:st].amin(-1, keepdim=True)) * (w / max(math.log10(N - ex), 1e-6))
    rs = max(lw, recent - 1) + 1
    far = corr[:, rs:]
    keep = torch.zeros(Hq, N, dtype=torch.bool, device=dev)
    keep[:, rs:] = far / far.amax(-1, keepdim=True).clamp(min=1e-6) >= float(np.float32(threshold))
    # diagonals: stripe or diffuse
    avail = max(1, (N + rs) // 2 - rs + 1)
    count = max(V7["min_diag_samples"], min(int(avail * V7["diag_sample_ratio"]), V7["max_diag_samples"]))
    count = min(count, avail)
    taus = [rs] if count <= 1 else (torch.linspace(0, avail - 1, count).long() + rs).tolist()
    s = S / math.sqrt(D)
    var = []
    for t in taus:
        d = torch.diagonal(s, offset=-t, dim1=1, dim2=2)[:, :-1]
        var.append(d.diff(dim=-1).var(-1) / d.abs().mean(-1).clamp(min=1e-6))
    mean_var = torch.stack(var, -1).mean(-1)
    stripe = mean_var <= float(np.float32(V7["stripe_threshold"])) if rs < N - 1 else torch.zeros_like(mean_var, dtype=torch.bool)
    # columns, last row
    rows = s * causal
    rows[:, N - 1] = 0
    col = rows.sum(1) / (N - 1 - i).clamp(min=1)
    c0, c1 = max(1, int(N * 0.1)), N - max(1, int(N * 0.2))
    ratio = V7["column_topk_ratio"] * min(1.0, math.sqrt(128.0 / N))
    cols = torch.zeros(Hq, N, dtype=torch.bool, device=dev)
    cols[:, c0:c1] = _top(col[:, c0:c1], min(max(1, int((c1 - c0) * ratio)), c1 - c0))
    last = S[:, N - 1].to(q.dtype).double()
    prior = (i[None, :] < sink) | (i[None, :] >= N - recent) | (lag.abs() <= lw)
    mask = prior.expand(Hq, N, N).clone()
    mask[:, N - 1] |= _top(last, min(128, N))
    lags = keep[:, lag.clamp(min=0)] & (lag >= rs) & (i[None, :] >= sink)
    mask |= stripe[:, None, None] & (lags | cols[:, None, :])
    for h in torch.nonzero(~stripe).flatten().tolist():
        x = s[h].masked_fill(~causal, -math.inf)
        order = torch.sort(x, dim=-1, descending=True, stable=True).indices
        n = ((i + 1).float() * float(np.float32(V7["qk_topk_ratio"]))).long().clamp(min=1)
        mask[h] |= torch.zeros_like(x, dtype=torch.bool).scatter_(1, order, i[None, :] < n[:, None])
    return mask & causal, dict(corr_sum=sums, col_mean=col, last_scores=last, mean_var=mean_var)


def _xattn_mask64(q, k, stride, threshold):
    """The XAttention block mask [Hq, N, N] (antidiagonal scores, 128-token blocks)."""
    Hq, L, D = q.shape
    G = Hq // k.shape[0]
    N = -(-L // 128)
    n = N * 128 // stride
    rb = 128 // stride
    mask = torch.zeros(Hq, N, N, dtype=torch.bool, device=q.device)

    def rows(x, flip):
        p = torch.zeros(N * 128, D, dtype=torch.float64, device=x.device)
        p[:L] = x
        p = p.view(n, stride, D)
        return (p.flip(1) if flip else p).reshape(n, stride * D)

    i = torch.arange(N, device=q.device)
    for h in range(Hq):
        a, b = rows(q[h], True), rows(k[h // G], False).T.contiguous()
        sums = torch.zeros(N, N, dtype=torch.float64, device=q.device)
        for r0 in range(0, n, 16 * rb):
            r1 = min(n, r0 + 16 * rb)
            x = (a[r0:r1] @ b[:, :r1]).to(q.dtype).double() / (math.sqrt(D) * stride)
            r = torch.arange(r0, r1, device=q.device)
            p = torch.softmax(x.masked_fill_(torch.arange(r1, device=q.device)[None] > r[:, None], -math.inf), -1)
            p[r >= -(-L // stride)] = 0
            sums[r0 // rb:r1 // rb, :r1 // rb] = p.view((r1 - r0) // rb, rb, r1 // rb, rb).sum((1, 3))
        sums = sums.to(q.dtype).double()
        forced = (i[None] == 0) | (i[None] == i[:, None])
        rest = sums.masked_fill(forced, 0.0)
        val, order = torch.sort(rest.masked_fill(i[None] > i[:, None], -1.0), dim=-1, descending=True, stable=True)
        val = val.clamp(min=0)
        before = (sums * forced).sum(-1, keepdim=True) + val.cumsum(-1) - val
        take = before < sums.sum(-1, keepdim=True) * threshold
        mask[h] = torch.zeros_like(mask[h]).scatter_(1, order, take) | forced
    return mask & (i[None, :] <= i[:, None])


def _flex_mask64(q, k, bs, gamma, tau):
    """The FlexPrefill block mask [Hq, N, N]."""
    Hq, L, D = q.shape
    G = Hq // k.shape[0]
    N = -(-L // bs)
    dev = q.device
    i = torch.arange(N, device=dev)
    tri = torch.ones(N, N, dtype=torch.bool, device=dev).tril()
    size = torch.tensor([min(bs, L - j * bs) for j in range(N)], dtype=torch.float64, device=dev)[:, None]
    mask = torch.zeros(Hq, N, N, dtype=torch.bool, device=dev)

    def pool(x):
        p = torch.zeros(N * bs, *x.shape[1:], dtype=torch.float64, device=dev)
        p[:L] = x
        return p.view(N, bs, *x.shape[1:]).sum(1)

    def cover(x):
        return int((torch.sort(x, descending=True).values.cumsum(0) <= gamma).sum()) + 1

    for h in range(Hq):
        kd = k[h // G].double()
        last = (q[h, L - bs:] / math.sqrt(D)).double()
        s = (last @ kd.T.contiguous()).to(q.dtype).double()
        s[:, L - bs:].masked_fill_(~torch.ones(bs, bs, dtype=torch.bool, device=dev).tril(), -math.inf)
        p = torch.softmax(s, -1)
        vert, slash = p.mean(0), torch.zeros(L, dtype=torch.float64, device=dev)
        for r in range(bs):
            slash[bs - 1 - r:] += p[r, :L - (bs - 1 - r)]
        slash /= bs
        nv, ns = (min(max(cover(x) // 128 + 1, 1), N) for x in (vert, slash))
        pv, ps = pool(vert), pool(slash)
        kb = (pool(kd) / size).to(q.dtype).double()
        a = torch.softmax((kb @ last.mean(0).to(q.dtype).double()).to(q.dtype).double(), 0)
        m = (a + pv) / 2
        js = torch.sqrt(0.5 * (a * torch.log(a / m)).sum() + 0.5 * (pv * torch.log(pv / m)).sum())
        if js < tau:
            nv = ns = 1
            qb = (pool(q[h].double()) / bs).to(q.dtype)
            pad = N * bs - L
            if pad:
                qb[-1] = (qb[-1] * bs).to(q.dtype) / (bs - pad)
            t = ((qb / math.sqrt(D)).double() @ kb.T.contiguous()).to(q.dtype).double().masked_fill_(~tri, -math.inf)
            flat = torch.softmax(t, -1).flatten()
            val, order = torch.sort(flat, descending=True, stable=True)
            mask[h].view(-1)[order[val.cumsum(0) <= gamma * N]] = True
        pv[0] = math.inf
        ps[-1] = math.inf
        mask[h] |= _top(pv, nv)[None, :]
        offs = _top(ps, ns).flip(0)                                    # offset s is entry N - 1 - s
        mask[h] |= offs[(i[:, None] - i[None, :]).clamp(min=0)]
        mask[h, 0, 0] = True
    return mask & tri


def _rope64(x, cos, sin):
    """The rotated states as the dtype holds them: each product and the sum rounded once."""
    h = x.shape[-1] // 2
    a = (x.double() * cos.double()).to(x.dtype).double()
    b = (torch.cat([-x[..., h:], x[..., :h]], -1).double() * sin.double()).to(x.dtype).double()
    return (a + b).to(x.dtype)


def exact(case, seed):
    c = case
    if c["path"] != "select" and c["B"] * c["Hq"] * c["L"] * c["L"] > EXACT_SCORES:
        return None
    s = prepare(c, seed)
    q, k, v, bs = s["q"], s["k"], s["v"], c["bs"]
    if _dense(c):
        return _attention64(q, k, v, None, bs).flatten(2)
    if c["path"] == "select":
        st = _v7_mask64(q[0], k[0], bs, c["threshold"])[1]
        return {"cnt": None, "bits": None, **st}
    if c["path"] == "rope":
        q, k = _rope64(q, s["cos"], s["sin"]), _rope64(k, s["cos"], s["sin"])
    if c["path"] in ("v7", "rope"):
        mask = _v7_mask64(q[0], k[0], bs, c["threshold"])[0]
    elif c["path"] == "fixed":
        N = -(-c["L"] // bs)
        i = torch.arange(N, device=q.device)
        n = max(1, int(N * 0.1))
        mask = (i[None] < n) | (i[None] >= N - n) | ((i[:, None] - i[None]).abs() <= max(2, int(N * 0.1)) // 2)
        mask = mask.expand(c["Hq"], N, N)
    elif c["path"] == "xattn":
        mask = _xattn_mask64(q[0], k[0], c["stride"], c["threshold"])
    else:
        mask = _flex_mask64(q[0], k[0], bs, c["threshold"], c["tau"])
    o = _attention64(q, k, v, mask, bs)
    if c["path"] == "rope":
        return o, k.double()
    if c["path"] == "xattn":
        return o.transpose(1, 2)
    return o if c["path"] == "flex" else o.flatten(2)
