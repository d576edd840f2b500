"""The prompt pass of the latent attention (csrc/kernels/attn_latent_prefill.hip) at the edges of row
blocks, key runs and windows, for every built head size, against float64.

Bound: weights rounded to bf16 in numerator and sum, the gate through a 1-ulp reciprocal, the
result rounded once: |error| <= 4 * 2^-9 * sum(p |v|) / den + f32 noise."""
import math

import pytest
import torch

from loqa_hub_amd import ops
from loqa_hub_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(feeds, pasts, H, DK, DV, Dv, window=0, sink=False, gate=False, scale=None, shift=0, gate_shift=0, kv_shift=0, seed=0):
    g = torch.Generator().manual_seed(seed)
    lens = [f + p for f, p in zip(feeds, pasts)]
    kept = [min(n, f + window - 1) if window else n for f, n in zip(feeds, lens)]
    T, L, scale = sum(feeds), sum(kept), DK ** -0.5 if scale is None else scale
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(DEV)
    at = lambda t: torch.cat([torch.zeros(kv_shift, dtype=t.dtype, device=DEV), t.reshape(-1)])[kv_shift:].view(t.shape)
    q, k, v = rnd(T, H, DK), at(rnd(L, H, DK)), at(rnd(L, H, DV))
    cu = lambda x: torch.tensor([0] + x).cumsum(0).int().to(DEV)
    cq, ck = cu(feeds), cu(kept)
    pos = torch.cat([torch.arange(p, p + f) for f, p in zip(feeds, pasts)]).int().to(DEV)
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    sk = torch.randn(H, generator=g).to(DEV) if sink else None
    gt = rnd(T, H * Dv + gate_shift)[:, gate_shift:] if gate else None
    o = torch.empty(T, H * Dv + shift, dtype=torch.bfloat16, device=DEV)[:, shift:]
    seqmix.latent_prefill(q, k, v, cq, ck, ctx, pos, sk, scale, max(feeds), Dv, window, gt, out=o)
    for b, (f, n, m) in enumerate(zip(feeds, lens, kept)):
        rows, keys = slice(int(cq[b]), int(cq[b]) + f), slice(int(ck[b]), int(ck[b]) + m)
        s = torch.bmm(q[rows].double().transpose(0, 1), k[keys].double().permute(1, 2, 0).contiguous()) * scale
        away = pos[rows, None] - torch.arange(n - m, n, device=DEV)[None]
        seen = (away >= 0) & (away < window) if window else away >= 0
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sk is not None:
            top = torch.maximum(top, sk.double()[:, None, None])
        p = (s - top).exp()
        p = p / (p.sum(-1, keepdim=True) + ((sk.double()[:, None, None] - top).exp() if sk is not None else 0.0))
        vs = v[keys, :, :Dv].double().transpose(0, 1).contiguous()
        want, size = torch.bmm(p, vs), torch.bmm(p, vs.abs())
        if gt is not None:
            w = torch.sigmoid(gt[rows].double()).view(f, H, Dv).transpose(0, 1)
            want, size = want * w, size * w
        got = o[rows].double().view(f, H, Dv).transpose(0, 1)
        assert ((got - want).abs() <= 4 * 2.0 ** -9 * size + 1e-5).all(), (b, f, n)


@pytest.mark.parametrize("DK", seqmix.PREFILL_DK)
@pytest.mark.parametrize("DV", seqmix.PREFILL_DV)
def test_sizes_and_edges(DK, DV):
    _check([1, 33, 64, 129, 200], [300, 0, 191, 31, 64], 2, DK, DV, DV, sink=True, gate=True, seed=DK)
    _check([70, 5], [250, 700], 2, DK, DV, DV - 12, window=65, seed=DV)
    _check([90], [0], 2, DK, DV, DV - 3, gate=True, scale=-0.05, seed=1)
    _check([40, 30], [100, 0], 2, DK, DV, DV, gate=True, shift=3, gate_shift=1, kv_shift=1, seed=2)


@pytest.mark.parametrize("B,T,H", [(1, 700, 8), (2, 700, 24), (4, 900, 24)])
def test_every_block_height(B, T, H):
    _check([T] * B, [7] * B, H, 192, 128, 128, 300, sink=True, seed=B)


@pytest.mark.parametrize("feeds,pasts,H,window", [([33], [2100], 8, 0), ([1, 64, 40], [4000, 450, 700], 4, 0), ([100, 7], [1200, 1500], 16, 0),
                                                  ([130], [3000], 8, 1030), ([64, 64], [1530, 600], 16, 0)])
def test_parts_of_the_keys(feeds, pasts, H, window):
    """One to eight parts of a block's keys in workgroups of their own, uneven ones, blocks of other lengths in one launch."""
    kept = sum(min(f + p, f + window - 1) if window else f + p for f, p in zip(feeds, pasts))
    assert ops.attn_parts(max(feeds), H * len(feeds), kept // len(feeds)) > 1
    for DK, DV in ((192, 128), (256, 64), (64, 64)):
        _check(feeds, pasts, H, DK, DV, DV - 12, window=window, sink=True, gate=True, seed=DK)
    _check(feeds, pasts, H, 128, 128, 128, window=window, scale=-0.05, seed=5)
    torch.cuda.synchronize()
    # every word of a ticket's line, as fl_join counts arrivals and published parts in four of them
    assert all(int(words.as_strided((words.numel(), 32), (32, 1)).abs().sum()) == 0 for _, words in ops._SK_WS.values())


def test_parts_repeat_bit_for_bit():
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(n, 16, d, generator=g).bfloat16().to(DEV) for n, d in ((64, 192), (2064, 192), (2064, 128)))
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)
    run = lambda: seqmix.latent_prefill(q, k, v, i32(0, 64), i32(0, 2064), i32(2064), torch.arange(2000, 2064, device=DEV).int(), None, 0.07, 64, 128)
    first = run()
    assert all(torch.equal(run(), first) for _ in range(10))
    graph = torch.cuda.CUDAGraph()
    args = (q, k, v, i32(0, 64), i32(0, 2064), i32(2064), torch.arange(2000, 2064, device=DEV).int(), None, 0.07, 64, 128)
    with torch.cuda.graph(graph):
        y = seqmix.latent_prefill(*args)
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert torch.equal(y, first) and torch.equal(run(), first)


@pytest.mark.parametrize("window", [(1 << 31) - 1, 1 << 31, (1 << 32) + 5])
def test_windows_beyond_all_positions(window):
    _check([33, 5], [100, 0], 2, 128, 128, 128, window=window, sink=True)
    g = torch.Generator().manual_seed(1)
    T, H, R, dims = 3, 4, 128, 64
    qa, qr, cache = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((H, T, R), (T, H, dims), (9, 16, R + dims)))
    ints = lambda *x: torch.tensor(x, dtype=torch.int32, device=DEV)      # noqa: E731
    cs = torch.randn(256, dims // 2, 2, generator=g).to(DEV)
    run = lambda w: seqmix.latent_attention(qa, qr, cache, ints(0, 1, 3), ints(130, 2), torch.arange(9, dtype=torch.int32, device=DEV)[None].repeat(2, 1),      # noqa: E731
                                            ints(129, 0, 1), cs, None, 0.1, R, dims, 130, window=w)
    assert torch.equal(run(window), run(0))
