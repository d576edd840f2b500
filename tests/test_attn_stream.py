"""Decode attention streamed through LDS (csrc/kernels/attn_stream.hip): tiles of 32 keys and their
remainders, pages of every size, groups of heads up to 16 rows, splits taken together."""
import math

import pytest
import torch

from loqa_hub_amd import ops


def _reference(q, ks, vs, qlens, H, G, D, causal):
    """64 bits; ks, vs per sequence [keys, Hkv, D]."""
    out, at = [], 0
    for k, v, n in zip(ks, vs, qlens):
        x = q[at:at + n].double().view(n, H, D)
        s = torch.einsum("thd,lhd->htl", x, k.double().repeat_interleave(G, 1)) * D ** -0.5
        if causal:
            seen = torch.arange(k.shape[0], device=q.device)[None] <= torch.arange(k.shape[0] - n, k.shape[0], device=q.device)[:, None]
            s = s.masked_fill(~seen[None], -math.inf)
        out.append(torch.einsum("htl,lhd->thd", torch.softmax(s, -1), v.double().repeat_interleave(G, 1)).flatten(1))
        at += n
    return torch.cat(out)


def _close(a, b):
    # weights rounded to bf16 (2^-9 of each) and a bf16 result: 2^-8 of the values that the weights average
    assert (a.double() - b).abs().max() <= 2.0 ** -7 * b.abs().max(), ((a.double() - b).abs().max(), b.abs().max())
    assert (a.double() - b).norm() <= 4e-3 * b.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("D,G,blk", [(64, 1, 16), (64, 4, 32), (64, 16, 64), (128, 1, 128), (128, 4, 16), (128, 3, 16), (128, 8, 64)])
@pytest.mark.parametrize("keys", [1, 31, 33, 129, 300, 1030])
def test_paged(D, G, blk, keys):
    Hkv, g = 2, torch.Generator().manual_seed(keys + D)
    H = Hkv * G
    most = 16 // G
    lens, qlens = [keys, max(1, keys - 17), min(keys, 5)], [1, min(most, max(1, keys - 17)), 1]
    need = [-(-n // blk) for n in lens]
    order = torch.randperm(sum(need) + 2, generator=g)
    kc, vc = (torch.randn(sum(need) + 2, Hkv, blk, D, generator=g).bfloat16().cuda() for _ in range(2))
    bt, at = torch.zeros(3, max(need), dtype=torch.int32), 0
    for b, n in enumerate(need):
        bt[b, :n] = order[at:at + n]
        at += n
    def rows(c):
        return [c[bt[b, :need[b]].long().cuda()].transpose(1, 2).reshape(-1, Hkv, D)[:lens[b]] for b in range(3)]
    q = torch.randn(sum(qlens), H * D, generator=g).bfloat16().cuda()
    cu = torch.tensor([0, qlens[0], qlens[0] + qlens[1], sum(qlens)], dtype=torch.int32).cuda()
    ref = _reference(q, rows(kc), rows(vc), qlens, H, G, D, True)
    kw = dict(n_heads=H, n_kv=Hkv, head_dim=D, causal=True, max_q=max(qlens), ctx_lens=torch.tensor(lens, dtype=torch.int32).cuda(),
              block_tables=bt.cuda(), grouped=True)
    for split in (32, 128, 256):
        ns = -(-max(lens) // split)
        ws = ops.AttnWorkspace("cuda", 64, H, D, ns + 1)
        for more in (0, 1):                       # as many splits as there are keys for, and one more
            y = ops.attention(q, kc, vc, cu, split_keys=split, num_splits=ns + more, workspace=ws, **kw)
            _close(y, ref)
            assert torch.equal(y, ops.attention(q, kc, vc, cu, split_keys=split, num_splits=ns + more, workspace=ws, **kw))
        assert int(ws.counters.abs().sum()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,T", [(1, 1500), (3, 50), (40, 333)])
def test_rows_in_place(D, B, T):
    """Key and value columns of one matrix, utterances in another order than their rows, lengths of their own; the general
    kernel (8 waves; queries off 16 bytes) beside it."""
    H, g = 4, torch.Generator().manual_seed(B)
    kv = torch.randn(B * T, 2 * H * D, generator=g).bfloat16().cuda()
    who = torch.randperm(B, generator=g)
    lens = [T - 3 * i % T for i in range(B)]
    q = torch.randn(B, H * D + 4, generator=g).bfloat16().cuda()
    rows = [kv[b * T:b * T + n].view(n, 2, H, D) for b, n in zip(who.tolist(), lens)]
    cu = torch.arange(B + 1, dtype=torch.int32).cuda()
    starts, ctx = (who * T).int().cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    ws = ops.AttnWorkspace("cuda", 64, H, D, 8)

    def run(x):
        return ops.attention(x, kv, kv[:, H * D:], cu, n_heads=H, n_kv=H, head_dim=D, causal=False, max_q=1, cu_k=starts, ctx_lens=ctx,
                             grouped=True, split_keys=256, num_splits=-(-T // 256), workspace=ws)
    x = q[:, :H * D].contiguous()
    ref = _reference(x, [r[:, 0] for r in rows], [r[:, 1] for r in rows], [1] * B, H, 1, D, False)
    _close(run(x), ref)
    _close(run(q[:, :H * D]), ref)                # rows 8 bytes off: the general kernel
    assert int(ws.counters.abs().sum()) == 0


@pytest.mark.gpu
def test_replays_of_a_captured_call():
    """The grid is made for the longest context, later contexts are shorter and longer."""
    D, H, Hkv, blk = 128, 8, 2, 16
    g = torch.Generator().manual_seed(2)
    kc, vc = (torch.randn(40, Hkv, blk, D, generator=g).bfloat16().cuda() for _ in range(2))
    bt = torch.randperm(40, generator=g)[None].int().cuda()
    q, ctx = torch.randn(1, H * D, generator=g).bfloat16().cuda(), torch.tensor([640], dtype=torch.int32).cuda()
    cu, ws = torch.tensor([0, 1], dtype=torch.int32).cuda(), ops.AttnWorkspace("cuda", 16, H, D, 5)

    def run():
        return ops.attention(q, kc, vc, cu, n_heads=H, n_kv=Hkv, head_dim=D, causal=True, max_q=1, ctx_lens=ctx, block_tables=bt,
                             grouped=True, split_keys=128, num_splits=5, workspace=ws)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = run()
    for n in (640, 1, 129, 600, 32):
        ctx.fill_(n)
        graph.replay()
        torch.cuda.synchronize()
        rows = [c[bt[0].long()].transpose(1, 2).reshape(-1, Hkv, D)[:n] for c in (kc, vc)]
        _close(y, _reference(q, [rows[0]], [rows[1]], [1], H, H // Hkv, D, True))
        assert torch.equal(y, run())


def _same_kind(a, b):
    """Infinities and NaN where ``b`` has them, the other values close."""
    a, fine = a.double(), b.isfinite()
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isfinite(), fine)
    assert torch.equal(a[~fine & ~b.isnan()], b[~fine & ~b.isnan()])
    _close(a[fine], b[fine])


@pytest.mark.gpu
@pytest.mark.parametrize("D,G", [(64, 1), (64, 4), (128, 8)])
@pytest.mark.parametrize("keys", [1, 40, 700])
def test_values_that_are_not_finite(D, G, keys):
    """An infinite value counts with every weight that is not zero, the row's largest (exactly one) among them: the
    result is infinite, or NaN where both infinities meet, as in the form that the GEMM prologues run."""
    Hkv, blk, g = 2, 16, torch.Generator().manual_seed(keys)
    H, need = Hkv * G, -(-keys // 16)
    kc, vc = (torch.randn(need, Hkv, blk, D, generator=g).bfloat16() for _ in range(2))
    for i, x in enumerate((math.inf, -math.inf, math.nan)):
        vc[:, 0, :, 8 * i] = x                        # all values of a column
        vc[min(1, need - 1), 1, min(keys - 1, 15) % blk, 8 * i + 3] = x       # one of them
    vc[0, 0, 0, 40] = math.inf
    vc[need - 1, 0, (keys - 1) % blk, 40] = -math.inf
    bt = torch.randperm(need, generator=g)[None].int()
    kc, vc, bt = kc.cuda(), vc.cuda(), bt.cuda()
    q = (3 * torch.randn(1, H * D, generator=g)).bfloat16().cuda()
    ks, vs = ([c[bt[0].long()].transpose(1, 2).reshape(-1, Hkv, D)[:keys]] for c in (kc, vc))
    # the sum term by term: a product over all keys at once may take 0 x inf for its padding
    p = torch.softmax(torch.einsum("hd,lhd->hl", q.double().view(H, D), ks[0].double().repeat_interleave(G, 1)) * D ** -0.5, -1)
    ref = (p.t()[:, :, None] * vs[0].double().repeat_interleave(G, 1)).sum(0).flatten()[None]
    ws, ns = ops.AttnWorkspace("cuda", 16, H, D, 6), -(-keys // 128)
    for streamed in (False, True):
        _same_kind(ops.attention(q, kc, vc, torch.tensor([0, 1], dtype=torch.int32).cuda(), n_heads=H, n_kv=Hkv, head_dim=D, causal=True, max_q=1,
                                 ctx_lens=torch.tensor([keys], dtype=torch.int32).cuda(), block_tables=bt, grouped=True,
                                 split_keys=128, num_splits=ns, workspace=ws, streamed=streamed), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_empty_sequences_and_feeds_of_no_tokens(D):
    """A row without a key is zero; a feed of no tokens writes nothing and leaves the tickets of its splits zero."""
    H, Hkv, blk, g = 8, 2, 16, torch.Generator().manual_seed(D)
    kc, vc = (torch.randn(30, Hkv, blk, D, generator=g).bfloat16().cuda() for _ in range(2))
    bt = torch.randperm(30, generator=g)[:30].view(1, 30).repeat(4, 1).int().cuda()
    lens, qlens = [0, 450, 300, 33], [1, 0, 2, 1]
    cu = torch.tensor([0, 1, 1, 3, 4], dtype=torch.int32).cuda()
    q = torch.randn(4, H * D, generator=g).bfloat16().cuda()
    ws = ops.AttnWorkspace("cuda", 16, H, D, 4)
    rows = [[c[bt[0].long()].transpose(1, 2).reshape(-1, Hkv, D)[:n] for n in lens[2:]] for c in (kc, vc)]
    ref = _reference(q[1:], *rows, qlens[2:], H, H // Hkv, D, True)
    for streamed in (False, True):
        out = torch.full((4, H * D), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.attention(q, kc, vc, cu, n_heads=H, n_kv=Hkv, head_dim=D, causal=True, max_q=2, ctx_lens=torch.tensor(lens, dtype=torch.int32).cuda(),
                      block_tables=bt, grouped=True, split_keys=128, num_splits=4, workspace=ws, out=out, streamed=streamed)
        assert (out[0] == 0).all()
        _close(out[1:], ref)
        assert int(ws.counters.abs().sum()) == 0


def _us(calls):
    """Least time of a call in a graph of ten, for each of ``calls`` in turn."""
    graphs = []
    for call in calls:
        call()
        torch.cuda.synchronize()
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            for _ in range(10):
                call()
    best = [math.inf] * len(calls)
    for _ in range(10):
        for i, graph in enumerate(graphs):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            best[i] = min(best[i], a.elapsed_time(b) * 100)
    return best


def _token(D, Hkv, G, B, keys, split, splits):
    g, H, need = torch.Generator().manual_seed(keys), Hkv * G, -(-keys // 16)
    kc, vc = (torch.randn(B * need, Hkv, 16, D, generator=g).bfloat16().cuda() for _ in range(2))
    i32 = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()      # noqa: E731
    q, cu, ctx = torch.randn(B, H * D, generator=g).bfloat16().cuda(), i32(range(B + 1)), i32([keys - b % 7 for b in range(B)])
    bt, ws = i32(torch.randperm(B * need, generator=g).view(B, need)), ops.AttnWorkspace("cuda", B, H, D, splits)
    return lambda streamed=True: ops.attention(q, kc, vc, cu, n_heads=H, n_kv=Hkv, head_dim=D, causal=True, max_q=1, ctx_lens=ctx, block_tables=bt,
                                               grouped=True, split_keys=split, num_splits=splits, workspace=ws, streamed=streamed)


@pytest.mark.gpu
def test_merge_of_many_splits_is_one_trip():
    """16 splits of 128 keys: 0.86 of the other form's time; 1.22 where the partials came one after the other."""
    call = _token(64, 4, 8, 4, 2000, 128, 16)
    us, former = _us([call, lambda: call(False)])
    assert us < 1.05 * former, (us, former)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_pages_cost_what_rows_cost(D):
    """1500 keys a workgroup: 1.04 of the time off contiguous rows; 1.24 with divisions by the page's rows for each load."""
    paged, ws = _token(D, 20, 1, 1, 1500, 1536, 1), ops.AttnWorkspace("cuda", 1, 20, D, 1)
    q, kv = torch.randn(1, 20 * D, device="cuda").bfloat16(), torch.randn(1500, 40 * D, device="cuda").bfloat16()
    cu, st, ctx = (torch.tensor(x, dtype=torch.int32).cuda() for x in ([0, 1], [0], [1500]))
    rows = lambda: ops.attention(q, kv[:, :20 * D], kv[:, 20 * D:], cu, n_heads=20, n_kv=20, head_dim=D, causal=True, max_q=1, cu_k=st,      # noqa: E731
                                 ctx_lens=ctx, grouped=True, split_keys=1536, num_splits=1, workspace=ws)
    us, other = _us([paged, rows])
    assert us < 1.12 * other, (us, other)


@pytest.mark.gpu
@pytest.mark.parametrize("D,Hkv,B,keys,split,former", [(128, 8, 33, 200, 224, True), (128, 8, 32, 200, 224, False), (128, 8, 33, 100, 128, False),
                                                       (128, 8, 33, 200, 128, False), (64, 8, 65, 200, 224, True), (64, 8, 64, 200, 224, False),
                                                       (64, 8, 97, 500, 512, True), (64, 8, 97, 520, 544, False), (64, 8, 96, 520, 544, True),
                                                       (128, 8, 20, 600, 256, True), (128, 8, 10, 600, 256, False), (128, 8, 20, 380, 128, False),
                                                       (64, 8, 40, 1000, 512, True), (64, 8, 32, 1000, 512, False)])
def test_many_sequences_take_the_former_kernel(D, Hkv, B, keys, split, former):
    """Either side of each line of the rule, the forms told apart by their sums' last bits; both right."""
    call = _token(D, Hkv, 2, B, keys, split, -(-keys // split))
    y, z = call(), call(False)
    assert torch.equal(y, z) == former
    _close(y, z.double())
