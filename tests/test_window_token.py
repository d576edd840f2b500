"""Token steps of the windowed paged attention on the matrix cores
(csrc/kernels/attn_window_token.hip), against float64: tile and wave edges, windows and kept
tokens, key splits, page and head sizes, heads per group.

Bound: scores, weights (three bf16 each) and sums are f32, so only the result's rounding to bf16
shows: |error| <= 2^-8 |result| + 2^-18 sum(p |v|) (and 2^-20 of a soft cap in the scores)."""
import math

import pytest
import torch

from loqa_hub_amd import ops
from loqa_hub_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(feeds, pasts, H, G, D, Dv, window=0, keep=0, cap=0.0, slopes=False, sink=False, gate=False, blk=16, splits=None, seed=0):
    g = torch.Generator().manual_seed(seed)
    B, T, lens = len(feeds), sum(feeds), [f + p for f, p in zip(feeds, pasts)]
    per = [-(-n // blk) for n in lens]
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
    o = seqmix.window_attention(q, kc.to(DEV), vc.to(DEV), cu, torch.tensor(lens, dtype=torch.int32, device=DEV), bt.to(DEV), pos,
                                D ** -0.5, cap, window, keep, gt, H, G, D, Dv, max_q=max(feeds), max_ctx=max(lens),
                                matrix_cores=False, key_splits=splits, sink=sk, slopes=sl)
    for b, (f, n) in enumerate(zip(feeds, lens)):
        rows = slice(int(cu[b]), int(cu[b]) + f)
        k = ks[b].repeat_interleave(H // G, 1).permute(1, 2, 0).contiguous()
        v = vs[b].repeat_interleave(H // G, 1).transpose(0, 1).contiguous()
        s = torch.bmm(q[rows].double().view(f, H, D).transpose(0, 1), k) * D ** -0.5
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
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -18 * size + 2.0 ** -20 * cap * size + 1e-6).all(), (b, f, n)


# one key up to several rounds of 16 waves, and the edges of a tile
ROWS = ([1] * 9, [0, 30, 31, 32, 63, 510, 511, 512, 1600])


@pytest.mark.parametrize("D,Dv", [(64, 64), (64, 128), (128, 64), (128, 128), (96, 72), (40, 120)])
@pytest.mark.parametrize("window,keep", [(0, 0), (1, 0), (32, 0), (100, 5), (100, 100), (513, 40)])
def test_windows(D, Dv, window, keep):
    _check(*ROWS, 8, 2, D, Dv, window, keep, sink=True, gate=True, seed=window + D)


@pytest.mark.parametrize("H,G", [(4, 4), (16, 1), (15, 3), (20, 1)])
def test_heads_per_group(H, G):
    _check(*ROWS, H, G, 64, 64, sink=True, seed=H)


@pytest.mark.parametrize("blk", [1, 24, 64, 256])
@pytest.mark.parametrize("splits", [1, 2, 5])
def test_pages_and_key_splits(blk, splits):
    _check(*ROWS, 8, 2, 128, 128, 700, 3, sink=True, gate=True, blk=blk, splits=splits, seed=blk)


@pytest.mark.parametrize("rows", [3, 40])
def test_many_rows(rows):
    # from 256 rows x key heads on: four waves a workgroup
    _check([rows, 5, rows], [77, 600, 0], 8, 4, 128, 128, 300, 2, slopes=True, seed=rows)
    _check([rows, 5, rows], [77, 600, 0], 8, 4, 64, 128, cap=15.0, gate=True, seed=rows)


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
def test_values_that_are_not_finite(value):
    # keys 0 .. 99, one of them with such values: the result where it is seen, nothing else of it
    kc, vc = torch.randn(7, 16, 64, device=DEV).bfloat16(), torch.randn(7, 16, 64, device=DEV).bfloat16()
    bt, cu = torch.arange(7, dtype=torch.int32, device=DEV)[None].contiguous(), torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    ctx, pos = torch.tensor([100], dtype=torch.int32, device=DEV), torch.tensor([99], dtype=torch.int32, device=DEV)
    q = torch.randn(1, 128, device=DEV).bfloat16()
    for key in (0, 31, 60, 99):
        v = vc.clone()
        v.view(-1, 64)[key, 5] = value
        for window in (0, 40):
            o = seqmix.window_attention(q, kc, v, cu, ctx, bt, pos, 0.125, 0.0, window, 0, None, 2, 1, 64, 64, max_q=1, max_ctx=100)
            hit = o.view(2, 64)[:, 5].float().cpu()
            if window and key < 60:
                assert hit.isfinite().all()
            else:
                assert torch.equal(hit, torch.full((2,), value)) or math.isnan(value) and hit.isnan().all(), (key, hit)
            o.view(2, 64)[:, 5] = 0
            assert o.isfinite().all()


def test_key_splits_of_the_other_form():
    # caches that do not start on 16 bytes take the other kernel, whose workgroups read 256 keys a
    # round: as many splits as before (with the splits of this form twice the time)
    T, G, n = 8, 4, 3000
    per = -(-n // 16)
    flat = torch.randn(T * per * 16 * G * 128 + 4, device=DEV).bfloat16()
    kc = flat[4:].view(T * per, 16, G * 128)
    bt = torch.randperm(T * per, device=DEV).int().view(T, per).contiguous()
    q, cu = torch.randn(T, 16 * 128, device=DEV).bfloat16(), torch.arange(T + 1, dtype=torch.int32, device=DEV)
    ctx, pos = torch.full((T,), n, dtype=torch.int32, device=DEV), torch.full((T,), n - 1, dtype=torch.int32, device=DEV)

    def us(splits):
        call = lambda: seqmix.window_attention(q, kc, kc, cu, ctx, bt, pos, 0.1, 0.0, 0, 0, None, 16, G, 128, 128, max_q=1, max_ctx=n,
                                               key_splits=splits)
        for _ in range(3):
            call()
        got = []
        for _ in range(8):            # the fastest of eight: clocks that have yet to rise do not count
            at = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            at[0].record()
            for _ in range(20):
                call()
            at[1].record()
            torch.cuda.synchronize()
            got.append(at[0].elapsed_time(at[1]))
        return min(got)
    assert us(None) < 1.4 * us(12)


@pytest.mark.parametrize("splits", [None, 2, 16, 64, 65])
def test_splits_join_in_the_launch(splits):
    # splits without keys, rows with fewer tiles than splits; more than 64 go to the other form
    _check([1] * 4, [0, 40, 700, 2100], 8, 2, 128, 128, sink=True, gate=True, splits=splits, seed=3)
    _check([1, 3], [2500, 90], 15, 3, 40, 120, 1000, 5, slopes=True, splits=splits, seed=4)
    torch.cuda.synchronize()
    assert all(int(words.as_strided((words.numel(), 32), (32, 1)).abs().sum()) == 0 for _, words in ops._SK_WS.values())


def test_splits_repeat_bit_for_bit():
    kc, vc = torch.randn(140, 16, 256, device=DEV).bfloat16(), torch.randn(140, 16, 256, device=DEV).bfloat16()
    bt, cu = torch.arange(140, dtype=torch.int32, device=DEV)[None].contiguous(), torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    ctx, pos = torch.tensor([2200], dtype=torch.int32, device=DEV), torch.tensor([2199], dtype=torch.int32, device=DEV)
    q = torch.randn(1, 1024, device=DEV).bfloat16()
    run = lambda: seqmix.window_attention(q, kc, vc, cu, ctx, bt, pos, 0.09, 0.0, 0, 0, None, 8, 2, 128, 128, max_q=1, max_ctx=2200)
    assert seqmix.window_token_splits(-(-2200 // 32), 2, 128) == 9
    first = run()
    assert all(torch.equal(run(), first) for _ in range(10))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert torch.equal(y, first) and torch.equal(run(), first)


@pytest.mark.parametrize("window,keep", [((1 << 31) - 1, 0), (1 << 31, 0), ((1 << 32) + 5, 3), (1 << 62, 1 << 62), (40, 1 << 31), (40, (1 << 31) - 1), ((1 << 31) - 1, (1 << 31) - 1)])
def test_windows_and_kept_keys_beyond_all_positions(window, keep):
    _check([1, 1, 2], [0, 700, 90], 8, 2, 128, 128, window, keep, sink=True)
    _check([1, 40], [300, 64], 8, 2, 72, 72, window, keep)
