"""Prompt portions of the windowed paged attention (csrc/kernels/attn_window_pipe.hip) at the edges
of row blocks, key runs, windows, kept tokens, pages and head sizes, against float64.

Bound: weights rounded to bf16 in numerator and sum (relative 2^-9 each), the gate through a
1-ulp reciprocal, the result rounded once: |error| <= 4 * 2^-9 * sum(p |v|) / den + f32 noise
(a soft cap moves scores by up to 2^-20 of the cap)."""
import math

import pytest
import torch

from loqa_hub_amd import ops
from loqa_hub_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(feeds, pasts, H, G, D, Dv, window, keep=0, cap=0.0, slopes=False, sink=False, gate=False, blk=16, scale=None,
           out_pad=0, seed=0):
    g = torch.Generator().manual_seed(seed)
    B, T, lens = len(feeds), sum(feeds), [f + p for f, p in zip(feeds, pasts)]
    per = [-(-n // blk) for n in lens]
    scale = D ** -0.5 if scale is None else scale
    q = torch.randn(T, H * D, generator=g).bfloat16().to(DEV)
    kc = torch.full((sum(per) + 2, blk, G * D), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((sum(per) + 2, blk, G * Dv), float("nan"), dtype=torch.bfloat16)
    ids = torch.randperm(sum(per) + 2, generator=g).int()
    bt = torch.zeros(B, max(per), dtype=torch.int32)
    ks, vs, at = [], [], 0
    for b, n in enumerate(lens):
        k, v = torch.randn(n, G * D, generator=g).bfloat16(), torch.randn(n, G * Dv, generator=g).bfloat16()
        bt[b, :per[b]] = ids[at:at + per[b]]
        at += per[b]
        rows = (bt[b, :per[b]].long()[:, None] * blk + torch.arange(blk)).reshape(-1)[:n]
        kc.view(-1, G * D)[rows], vc.view(-1, G * Dv)[rows] = k, v
        ks.append(k.to(DEV).double().view(n, G, D))
        vs.append(v.to(DEV).double().view(n, G, Dv))
    cu = torch.tensor([0] + feeds).cumsum(0).int().to(DEV)
    pos = torch.cat([torch.arange(p, p + f) for f, p in zip(feeds, pasts)]).int().to(DEV)
    sk = torch.randn(H, generator=g).to(DEV) if sink else None
    sl = (torch.rand(H, generator=g) * 0.02).to(DEV) if slopes else None
    gt = torch.randn(T, H * Dv, generator=g).bfloat16().to(DEV) if gate else None
    o = torch.empty(T, H * Dv + out_pad, dtype=torch.bfloat16, device=DEV)[:, :H * Dv]
    seqmix.window_attention(q, kc.to(DEV), vc.to(DEV), cu, torch.tensor(lens, dtype=torch.int32, device=DEV), bt.to(DEV), pos,
                            scale, cap, window, keep, gt, H, G, D, Dv, max_q=max(feeds), max_ctx=max(lens), matrix_cores=True,
                            sink=sk, slopes=sl, out=o)
    for b, (f, n) in enumerate(zip(feeds, lens)):
        rows = slice(int(cu[b]), int(cu[b]) + f)
        k = ks[b].repeat_interleave(H // G, 1).permute(1, 2, 0).contiguous()
        v = vs[b].repeat_interleave(H // G, 1).transpose(0, 1).contiguous()
        s = torch.bmm(q[rows].double().view(f, H, D).transpose(0, 1), k) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        away = pos[rows, None] - torch.arange(n, device=DEV)[None]
        if sl is not None:
            s = s - sl.double()[:, None, None] * away
        seen = away >= 0
        if window:
            seen &= (away < window) | (torch.arange(n, device=DEV)[None] < keep)
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sk is not None:
            top = torch.maximum(top, sk.double()[:, None, None])
        p = (s - top).exp()
        p = p / (p.sum(-1, keepdim=True) + ((sk.double()[:, None, None] - top).exp() if sk is not None else 0.0))
        want, size = torch.bmm(p, v), torch.bmm(p, v.abs())
        if gt is not None:
            w = torch.sigmoid(gt[rows].double()).view(f, H, Dv).transpose(0, 1)
            want, size = want * w, size * w
        got = o[rows].double().view(f, H, Dv).transpose(0, 1)
        assert ((got - want).abs() <= 4 * 2.0 ** -9 * size + 1e-5).all(), (b, f, n)


@pytest.mark.parametrize("window,keep", [(0, 0), (1, 0), (64, 0), (100, 5), (100, 70), (300, 300), (65, 64)])
@pytest.mark.parametrize("D,Dv", [(64, 64), (64, 128), (128, 64), (128, 128), (96, 72), (40, 256)])
def test_windows(D, Dv, window, keep):
    _check([1, 33, 64, 130, 257], [300, 0, 513, 31, 64], 4, 2, D, Dv, window, keep, sink=True, gate=True, seed=window)


@pytest.mark.parametrize("blk", [1, 8, 16, 24, 64, 256])
def test_pages(blk):
    _check([70, 3, 200], [700, 90, 5], 4, 2, 128, 128, 128, 3, blk=blk, seed=blk)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,T,H", [(1, 300, 4), (2, 520, 40), (3, 900, 40)])
def test_every_block_height(D, B, T, H):
    _check([T] * B, [7] * B, H, 4, D, D, 200, 4, seed=T)


@pytest.mark.parametrize("D,Dv", [(64, 64), (128, 128), (72, 48), (128, 40)])
def test_transformed_scores(D, Dv):
    _check([90, 40], [100, 0], 4, 2, D, Dv, 0, cap=20.0, seed=1)
    _check([90, 40], [100, 0], 4, 2, D, Dv, 77, 2, slopes=True, sink=True, seed=2)
    _check([90, 40], [100, 0], 4, 2, D, Dv, 77, 2, cap=5.0, slopes=True, gate=True, seed=3)
    _check([50], [10], 4, 2, D, Dv, 0, scale=-0.1, seed=4)


def test_other_places_take_the_other_kernel():
    _check([60], [40], 4, 2, 64, 64, 0, out_pad=4, seed=5)
    _check([60, 300], [40, 0], 4, 2, 192, 64, 100, 3, seed=6)


def _us(call):
    for _ in range(3):
        call()
    us = []
    for _ in range(8):                # the fastest of eight, the host ahead
        at = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda._sleep(500000)
        at[0].record()
        for _ in range(10):
            call()
        at[1].record()
        torch.cuda.synchronize()
        us.append(at[0].elapsed_time(at[1]))
    return min(us)


@pytest.mark.parametrize("cap", [0.0, 20.0])
def test_many_short_feeds(cap):
    # more of them than CUs do not take a second round: a ninth feed, 0.9 to 1.0 of the time (1.7 to 1.9 with two key runs)
    _check([20, 37, 64, 20, 1, 64, 20, 20, 20], [0, 100, 0, 0, 3, 64, 0, 0, 0], 32, 8, 64, 64, 300, cap=cap, seed=6)

    def call(B, n=40, H=32, D=64):
        q, kc = torch.randn(B * n, H * D, device=DEV).bfloat16(), torch.randn(3 * B, 16, 8 * D, device=DEV).bfloat16()
        bt, cu = torch.arange(3 * B, dtype=torch.int32, device=DEV).view(B, 3), torch.arange(0, B * n + 1, n, dtype=torch.int32, device=DEV)
        ctx, pos = torch.full((B,), n, dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV).repeat(B)
        return lambda: seqmix.window_attention(q, kc, kc, cu, ctx, bt, pos, 0.125, cap, 300, 0, None, H, 8, D, D, max_q=n, max_ctx=n)
    assert _us(call(9)) < 1.4 * _us(call(8))


@pytest.mark.parametrize("feeds,pasts,H,window,keep", [([33], [2100], 8, 0, 0), ([1, 64, 40], [4000, 450, 700], 4, 0, 0), ([100, 7], [1200, 1500], 8, 0, 0),
                                                       ([130], [3000], 8, 1030, 70), ([64], [1500], 16, 1100, 200)])
def test_parts_of_the_keys(feeds, pasts, H, window, keep):
    """One to eight parts of a block's keys in workgroups of their own; parts that end among the kept tokens' tiles."""
    keys = min(max(f + p for f, p in zip(feeds, pasts)), window + 64 + keep if window else 1 << 30)
    assert ops.attn_parts(max(feeds), H * len(feeds), keys) > 1
    _check(feeds, pasts, H, 2, 128, 128, window, keep, sink=True, gate=True, seed=1)
    _check(feeds, pasts, H, 4, 64, 64, window, keep, seed=2)
    _check(feeds, pasts, H, 4, 96, 200, window, keep, sink=True, seed=3)
    _check(feeds, pasts, H, 4, 64, 72, window, keep, cap=30.0, seed=4)      # transformed scores: whole
    torch.cuda.synchronize()
    # every word of a ticket's line, as fl_join counts arrivals and published parts in four of them
    assert all(int(words.as_strided((words.numel(), 32), (32, 1)).abs().sum()) == 0 for _, words in ops._SK_WS.values())


@pytest.mark.parametrize("most", [None, 0, 2100])
def test_prompts_of_any_context_bound(most):
    """The bound on the context only says whether keys go in parts: prompts without one are taken, whole."""
    g = torch.Generator().manual_seed(8)
    q, kc, vc = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((33, 8 * 64), (132, 16, 2 * 64), (132, 16, 2 * 64)))
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32, device=DEV)      # noqa: E731
    args = (q, kc, vc, i32([0, 33]), i32([2100]), i32(torch.randperm(132, generator=g).view(1, 132)), i32(range(2067, 2100)), 0.125, 0.0, 0, 0, None, 8, 2, 64, 64)
    y, z = (seqmix.window_attention(*args, max_q=33, max_ctx=n).double() for n in (most, 2100))
    assert (y - z).norm() <= 4e-3 * z.norm()


@pytest.mark.parametrize("D,Dv", [(64, 64), (128, 128), (64, 128), (96, 96)])
@pytest.mark.parametrize("window", [300, 513, 600, 0])
def test_runs_of_few_tiles_and_many(D, Dv, window):
    # four to six tiles a run and more, around which the waves of a SIMD go half a tile apart; transformed scores in step
    _check([900], [60], 32, 8, D, Dv, window, 5, sink=True, gate=True, seed=1)
    _check([900], [60], 32, 8, D, Dv, window, 5, cap=30.0, gate=True, seed=2)
    _check([900], [60], 32, 8, D, Dv, window, 0, slopes=True, sink=True, seed=3)
