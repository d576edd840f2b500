"""The pipelined attention kernel (csrc/kernels/flash_pipe.h, attention.hip) at the edges of its
tiles, key runs and pages, against float64.

Bound: the weights are rounded to bf16 (relative 2^-9) in the numerator and in their sum, the
result once more; scores and sums are f32. |error| <= 3 * 2^-9 * sum(p |v|) / sum(p) + f32 noise."""
import math

import pytest
import torch

from loqa_hub_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(qlens, klens, Hq, Hkv, D, causal, page=0, q_pad=0, shift=0, seed=0, spread=1.0):
    g = torch.Generator().manual_seed(seed)
    B, Tq, Tk = len(qlens), sum(qlens), sum(klens)
    q = (spread * torch.randn(Tq, Hq * D + q_pad, generator=g)).bfloat16().to(DEV)
    k = torch.randn(Tk, Hkv, D, generator=g).bfloat16().to(DEV)
    v = torch.randn(Tk, Hkv, D, generator=g).bfloat16().to(DEV)
    cu = lambda x: torch.tensor([0] + x).cumsum(0).int().to(DEV)
    kw = dict(n_heads=Hq, n_kv=Hkv, head_dim=D, causal=causal, max_q=max(qlens))
    cq, ck = cu(qlens), cu(klens)
    if page:
        per = [-(-x // page) for x in klens]
        ids = torch.randperm(sum(per) + 3, generator=g).int()
        bt = torch.zeros(B, max(per), dtype=torch.int32)
        kc = torch.full((sum(per) + 3, Hkv, page, D), float("nan"), dtype=torch.bfloat16, device=DEV)
        vc = kc.clone()
        at = 0
        for b, n in enumerate(klens):
            for x in range(per[b]):
                bt[b, x] = ids[at]
                m = min(page, n - x * page)
                rows = slice(int(ck[b]) + x * page, int(ck[b]) + x * page + m)
                kc[ids[at], :, :m], vc[ids[at], :, :m] = k[rows].transpose(0, 1), v[rows].transpose(0, 1)
                at += 1
        ctx = torch.tensor(klens, dtype=torch.int32, device=DEV)
        o = ops.attention(q, kc, vc, cq, ctx_lens=ctx, block_tables=bt.to(DEV), max_k=max(klens), **kw)
    else:
        o = torch.empty(Tq, Hq * D + shift, dtype=torch.bfloat16, device=DEV)[:, shift:]
        ops.attention(q, k.view(Tk, -1), v.view(Tk, -1), cq, cu_k=ck, out=o, **kw)
    for b, (n, m) in enumerate(zip(qlens, klens)):
        qs = q[int(cq[b]):int(cq[b]) + n, :Hq * D].double().view(n, Hq, D).transpose(0, 1)
        ks = k[int(ck[b]):int(ck[b]) + m].double().repeat_interleave(Hq // Hkv, 1).permute(1, 2, 0).contiguous()
        vs = v[int(ck[b]):int(ck[b]) + m].double().repeat_interleave(Hq // Hkv, 1).transpose(0, 1).contiguous()
        s = torch.bmm(qs, ks) / math.sqrt(D)
        if causal:
            away = torch.arange(m, device=DEV)[None] - (torch.arange(n, device=DEV)[:, None] + m - n)
            s.masked_fill_(away > 0, -math.inf)
        p = s.softmax(-1)
        want, size = torch.bmm(p, vs), torch.bmm(p, vs.abs())
        got = o[int(cq[b]):int(cq[b]) + n].double().view(n, Hq, D).transpose(0, 1)
        assert ((got - want).abs() <= 3 * 2.0 ** -9 * size + 1e-5).all(), (b, n, m)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_tiles_and_runs(D, causal):
    # row blocks of 32, one to five key tiles (every way they split into runs), and their edges
    lens = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 256, 257, 319]
    _check(lens, lens, 4, 2, D, causal)
    _check([1, 5, 40, 64, 3], [64, 197, 129, 321, 1500], 2, 1, D, causal, seed=1)
    _check([70], [70], 4, 2, D, causal, q_pad=8, seed=2)


@pytest.mark.parametrize("D,B,H,n", [(64, 1, 20, 1500), (64, 3, 20, 1500), (128, 1, 32, 520), (128, 5, 32, 520)])
def test_every_block_height(D, B, H, n):
    # the grids that take 128 rows with two runs, and 128 rows with one
    _check([n] * B, [n] * B, H, H // 4, D, D == 128, seed=3)


@pytest.mark.parametrize("page", [1, 8, 16, 24, 32, 64, 128, 1024])
@pytest.mark.parametrize("D", [64, 128])
def test_pages(D, page):
    # unused rows of a page hold NaN; more than 64 pages a sequence where they are small
    _check([1, 7, 65, 130], [700, 7, 1100, 193], 4, 2, D, True, page=page, seed=4)


def test_peaked_and_flat():
    for spread in (0.0, 1e-3, 30.0):
        _check([100], [300], 2, 2, 64, False, seed=5, spread=spread)
        _check([100], [300], 2, 2, 128, True, seed=6, spread=spread)


def test_rows_off_16_bytes_take_the_other_kernel():
    _check([50, 9], [50, 200], 2, 2, 64, True, q_pad=4, seed=7)
    _check([50, 9], [50, 200], 2, 2, 128, False, shift=4, seed=8)


def _us(call, n=20):
    for _ in range(3):
        call()
    us = []
    for _ in range(8):                # the fastest of eight: clocks that have yet to rise do not count
        at = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        torch.cuda._sleep(500000)     # the host is ahead
        at[0].record()
        for _ in range(n):
            call()
        at[1].record()
        torch.cuda.synchronize()
        us.append(at[0].elapsed_time(at[1]) * 1e3 / n)
    return min(us)


@pytest.mark.parametrize("D,H,G", [(64, 20, 20), (128, 32, 8)])
def test_other_places_cost_no_multiple(D, H, G):
    # blocks that are no power of two find a row per chunk (1.2 to 1.9 times the time of the
    # others, 4 to 5.5 times on a kernel without key runs)
    def call(page):
        per = -(-1000 // page)
        kc = torch.randn(per, G, page, D, device=DEV).bfloat16()
        q, bt = torch.randn(40, H * D, device=DEV).bfloat16(), torch.randperm(per, device=DEV).int()[None].contiguous()
        cu, ctx = torch.tensor([0, 40], dtype=torch.int32, device=DEV), torch.tensor([1000], dtype=torch.int32, device=DEV)
        return lambda: ops.attention(q, kc, kc, cu, n_heads=H, n_kv=G, head_dim=D, causal=True, max_q=40, ctx_lens=ctx,
                                     block_tables=bt, max_k=1000)
    assert _us(call(12)) < 3 * _us(call(16))


def test_long_causal_prompts():
    # heads of 64 from 1024 rows on: two key runs where more, but shorter, prompts take one
    _check([1100], [1100], 20, 4, 64, True, seed=9)
    _check([2000], [2100], 20, 4, 64, True, page=16, seed=10)

    def call(H, n=2048):
        q, cu = torch.randn(n, 3 * H * 64, device=DEV).bfloat16(), torch.tensor([0, n], dtype=torch.int32, device=DEV)
        return lambda: ops.attention(q[:, :H * 64], q[:, H * 64:2 * H * 64], q[:, 2 * H * 64:], cu, n_heads=H, n_kv=H, head_dim=64,
                                     causal=True, max_q=n, cu_k=cu)
    # fewer heads take no longer (0.96 of 32 heads' time; 1.22 on one run)
    assert _us(call(20)) < 1.1 * _us(call(32))


def test_one_tile_has_nothing_to_merge():
    def call(n, H=32):
        q, cu = torch.randn(n, 3 * H * 64, device=DEV).bfloat16(), torch.tensor([0, n], dtype=torch.int32, device=DEV)
        return lambda: ops.attention(q[:, :H * 64], q[:, H * 64:2 * H * 64], q[:, 2 * H * 64:], cu, n_heads=H, n_kv=H, head_dim=64,
                                     causal=True, max_q=n, cu_k=cu)
    # 0.88 of the time of two tiles; 1.00 with the merge of runs that have none
    assert _us(call(64)) < 0.95 * _us(call(100))


def test_many_short_prompts():
    # 128-column heads: more prompts than CUs do not take a second round (a ninth prompt: 1.0 of the
    # time; 1.8 with two key runs)
    _check([20, 1, 64, 33, 40, 40, 40, 40, 40], [20, 90, 64, 33, 40, 400, 40, 40, 41], 32, 8, 128, True, page=16, seed=11)

    def call(B, n=40, H=32, G=8, D=128):
        q, kc = torch.randn(B * n, H * D, device=DEV).bfloat16(), torch.randn(3 * B, G, 16, D, device=DEV).bfloat16()
        cu, ctx = torch.arange(0, B * n + 1, n, dtype=torch.int32, device=DEV), torch.full((B,), n, dtype=torch.int32, device=DEV)
        bt = torch.arange(3 * B, dtype=torch.int32, device=DEV).view(B, 3)
        return lambda: ops.attention(q, kc, kc, cu, n_heads=H, n_kv=G, head_dim=D, causal=True, max_q=n, ctx_lens=ctx, block_tables=bt,
                                     max_k=n)
    assert _us(call(9)) < 1.4 * _us(call(8))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("qlens,klens,Hq,page", [([33], [2100], 8, 16), ([1, 64, 40], [4100, 450, 700], 4, 64), ([100, 7], [1300, 1507], 8, 8),
                                                 ([130], [9000], 4, 1024), ([64], [1024], 8, 32), ([90, 90], [2000, 1100], 4, 0)])
def test_parts_of_the_keys(D, qlens, klens, Hq, page):
    """One to eight parts of a block's keys in workgroups of their own, uneven ones, short sequences beside long ones."""
    assert ops.attn_parts(max(qlens), Hq * len(qlens), max(klens) if page else sum(klens) // len(klens)) > 1
    _check(qlens, klens, Hq, 2, D, True, page=page, seed=7)
    _check(qlens, klens, Hq, 2, D, False, page=page, seed=8, spread=4.0)
    torch.cuda.synchronize()
    # every word of a ticket's line, as fl_join counts arrivals and published parts in four of them
    assert all(int(words.as_strided((words.numel(), 32), (32, 1)).abs().sum()) == 0 for _, words in ops._SK_WS.values())


def test_when_keys_are_in_parts():
    assert [ops.attn_parts(*x) for x in ((64, 32, 1024), (64, 32, 1023), (64, 64, 4000), (200, 32, 4000), (257, 32, 4000), (1, 1, 1024), (0, 8, 4000))] == \
        [8, 1, 4, 2, 1, 8, 1]


@pytest.mark.parametrize("n,H,D", [(40, 4, 64), (200, 20, 64), (1500, 20, 64), (40, 4, 128), (1100, 32, 128)])
def test_one_tile_on_every_block_height(n, H, D):
    # all rows see one tile of keys: the runs without one have left (64 rows on four and two runs, 128 rows on two)
    for m in (1, 33, 64):
        _check([n, 1, 33], [m, 64, 1], H, H // 4, D, False, seed=m)
        _check([m, 1], [m, 64], H, H // 4, D, True, page=16, seed=m)
    _check([n, 70], [64, 65], H, H // 4, D, False, seed=3)          # one tile beside two


@pytest.mark.parametrize("D", [64, 128])
def test_runs_of_few_tiles_and_many(D):
    # five and six tiles a run, around which the waves of a SIMD go half a tile apart: two runs of 128 rows, four (two) of 64
    for n in (640, 641):
        _check([700], [n], 20, 20, D, False, seed=n)
    _check([850], [1400], 32, 8, D, True, page=16, seed=1)
    _check([850], [1400], 32, 8, D, True, page=64, seed=2)
    _check([64, 40], [1280, 1281], 8, 8, D, False, seed=3)
    _check([64, 40], [640, 641], 8, 8, D, False, seed=4)
