"""K chunks of the pipelined tiles (csrc/kernels/gemm_pipe_tile.h): every workgroup of a tile sums up
its share of it, the last to arrive those that others gave up."""
import pytest
import torch

from loqa_hub_amd import ops


def _close(a, b, k):
    # as in test_gemm_pipe.py: half a bf16 ulp of the value, and the f32 sum's own rounding
    tol = 2.0 ** -8 * b.abs() + (k * 2.0 ** -22 + 2.0 ** -9) * b.std()
    assert torch.all((a.double() - b).abs() <= tol), ((a.double() - b).abs() - tol).max().item()


def _words_are_zero():
    torch.cuda.synchronize()
    assert all(int(cnt.abs().sum()) == 0 for _, cnt in ops._SK_WS.values())


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [k for k in sorted({**ops.SK_LAYOUTS, **ops.SK_ROWS160}) if k >= ops.SK_PIPE])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 8, 9, 14])
def test_shares_of_a_tile(layout, splits):
    """More chunks than units of 16 x 16 in a share divide evenly, more than SK_SHARE, ragged rows, every epilogue."""
    bn, bm = ops._sk_tile(layout)[:2]
    K, N, M = 64 * 14, 2 * bn, bm + 21
    g = torch.Generator().manual_seed(layout)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) / 16).bfloat16().cuda()
    b = torch.randn(N, generator=g).cuda()
    ref = x.double() @ w.double().t()
    first = ops.gemm_sk(x, w, bias=b, layout=layout, splits=splits)
    _close(first, ref + b.double(), K)
    assert torch.equal(ops.gemm_sk(x, w, bias=b, layout=layout, splits=splits), first)
    z = ref + b.double()
    _close(ops.gemm_sk(x, w, bias=b, act="gelu", layout=layout, splits=splits), 0.5 * z * torch.erfc(-z * 0.5 ** 0.5), K)
    res = torch.randn(M, N, generator=g).bfloat16().cuda()
    want = res.double() + z
    _close(ops.gemm_sk(x, w, epi="resid", bias=b, residual=res, layout=layout, splits=splits), want, K)
    h = ref[:, :bn]
    _close(ops.gemm_sk(x, w, epi="swiglu", layout=layout, splits=splits), h * torch.sigmoid(h) * ref[:, bn:], K)
    _words_are_zero()


@pytest.mark.gpu
def test_a_chunk_that_starts_a_round_later():
    """300 workgroups of one a compute unit: chunks of one tile in different rounds, longer apart than a workgroup
    waits, so that shares are given up."""
    g = torch.Generator().manual_seed(1)
    K = 64 * 180
    x = torch.randn(2500, K, generator=g).bfloat16().cuda()
    w = (torch.randn(2560, K, generator=g) / 64).bfloat16().cuda()
    first = ops.gemm_sk(x, w, layout=12, splits=3)
    _close(first, x.double() @ w.double().t(), K)
    for _ in range(3):
        assert torch.equal(ops.gemm_sk(x, w, layout=12, splits=3), first)
    _words_are_zero()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [k for k in sorted({**ops.SK_LAYOUTS, **ops.SK_ROWS160}) if k >= ops.SK_PIPE])
@pytest.mark.parametrize("splits", [2, 4, 5, 8])
def test_shares_given_up(layout, splits, monkeypatch):
    """No looks at a tile's word: every workgroup but the last to arrive goes through publishing what it kept and giving
    its share up, in every epilogue, with and without kept shares. Whoever sums a share up, it is the same bits."""
    bn, bm = ops._sk_tile(layout)[:2]
    K, N, M = 64 * 14, 4 * bn, 2 * bm + 21
    g = torch.Generator().manual_seed(layout)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) / 16).bfloat16().cuda()
    b, res = torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).bfloat16().cuda()
    run = lambda: [ops.gemm_sk(x, w, bias=b, layout=layout, splits=splits), ops.gemm_sk(x, w, bias=b, act="gelu", layout=layout, splits=splits),      # noqa: E731
                   ops.gemm_sk(x, w, epi="resid", bias=b, residual=res.clone(), layout=layout, splits=splits),
                   ops.gemm_sk(x, w, epi="swiglu", layout=layout, splits=splits)]
    want, lib, calls = run(), ops.kernels(), []

    class Hurried:
        def __getattr__(self, name):
            return getattr(lib, name)

        def loqa_gemm_sk(self, call, stream):
            call._obj.hurry = 1 << 20
            calls.append(call._obj.S)
            return lib.loqa_gemm_sk(call, stream)

    monkeypatch.setattr(ops, "kernels", Hurried)
    for _ in range(3):
        assert all(torch.equal(y, z) for y, z in zip(run(), want))
    assert calls == 12 * [splits]
    _words_are_zero()


@pytest.mark.gpu
def test_launches_of_a_capture_share_a_workspace():
    """Two graphs, each with a launch that outgrows the first one's partials: their own memory, and every
    replay, on two streams at once, equal to the eager result."""
    g = torch.Generator().manual_seed(2)
    K = 64 * 24
    x = torch.randn(300, K, generator=g).bfloat16().cuda()
    ws = [(torch.randn(n, K, generator=g) / 16).bfloat16().cuda() for n in (256, 1024, 256)]
    run = lambda: [ops.gemm_sk(x, w, layout=15, splits=3) for w in ws]      # noqa: E731
    want = run()
    graphs, outs = [], []
    for _ in range(2):
        n = len(ops._SK_WS_GRAPHS)
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            outs.append(run())
        assert len(ops._SK_WS_GRAPHS) == n + 2                              # the first launch's, and the larger one's
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(5):
        for out in outs:
            for y in out:
                y.fill_(7)
        torch.cuda.synchronize()
        for s, gr in zip(streams, graphs):
            with torch.cuda.stream(s):
                gr.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(y, z) for out in outs for y, z in zip(out, want))
        assert all(torch.equal(y, z) for y, z in zip(run(), want))
    assert all(int(cnt.abs().sum()) == 0 for _, cnt in ops._SK_WS_GRAPHS)


@pytest.mark.gpu
def test_a_captures_workspace_grows_to_the_largest_of_both():
    """Launches that want many partials and launches that want many tickets, in turn: the first two of a capture make
    its workspace, the others find it."""
    g = torch.Generator().manual_seed(3)
    x = torch.randn(64, 64 * 40, generator=g).bfloat16().cuda()
    ws = [(torch.randn(n, x.shape[1], generator=g) / 16).bfloat16().cuda() for n in (512, 2048)]
    # 2 tiles of 256 x 256 in five chunks; 32 tiles of 64 x 64 in two
    run = lambda: [ops.gemm_sk(x, w, layout=lay, splits=s) for w, lay, s in 3 * ((ws[0], 12, 5), (ws[1], ops.SK_SMALL, 2))]      # noqa: E731
    want, n = run(), len(ops._SK_WS_GRAPHS)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    assert len(ops._SK_WS_GRAPHS) == n + 2
    for _ in range(3):
        for y in got:
            y.zero_()
        graph.replay()
        assert all(torch.equal(y, z) for y, z in zip(got, want))
        assert all(torch.equal(y, z) for y, z in zip(run(), want))


@pytest.mark.gpu
def test_captures_give_their_workspaces_back():
    """Graphs captured and dropped again and again: what is held for them does not grow, the memory is that of before, and a
    graph that lives replays right beside eager launches and later captures."""
    g = torch.Generator().manual_seed(4)
    x = torch.randn(300, 64 * 24, generator=g).bfloat16().cuda()
    w = (torch.randn(256, x.shape[1], generator=g) / 16).bfloat16().cuda()
    run = lambda: ops.gemm_sk(x, w, layout=15, splits=3)      # noqa: E731

    def capture():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = run()
        return graph, y
    want, (kept, out) = run(), capture()
    before = torch.cuda.memory_allocated()
    for _ in range(ops._SK_WS_KEPT + 3):
        graph, y = capture()
        y.zero_()
        graph.replay()
        assert torch.equal(y, want)
        del graph, y
        assert 0 < len(ops._SK_WS_GRAPHS) <= ops._SK_WS_KEPT
    assert torch.equal(run(), want)
    assert not ops._SK_WS_GRAPHS and not ops._SK_WS_CAPTURE and torch.cuda.memory_allocated() <= before
    for _ in range(3):
        junk = [torch.full((1 << 20,), 7.0, device="cuda") for _ in range(4)]
        out.zero_()
        kept.replay()
        assert torch.equal(out, want) and torch.equal(run(), want) and all((j == 7).all() for j in junk)
    _words_are_zero()


@pytest.mark.gpu
def test_launches_of_a_capture_whose_workspace_is_let_go():
    """The workspace of a running capture goes (another thread's eager launch may do that): the launches behind
    clear their own."""
    g = torch.Generator().manual_seed(5)
    x = torch.randn(300, 64 * 24, generator=g).bfloat16().cuda()
    ws = [(torch.randn(n, x.shape[1], generator=g) / 16).bfloat16().cuda() for n in (256, 1024, 512)]
    run = lambda w: ops.gemm_sk(x, w, layout=15, splits=3)      # noqa: E731
    want = [run(w) for w in ws]
    graph, got = torch.cuda.CUDAGraph(), []
    with torch.cuda.graph(graph):
        for w in ws:
            got.append(run(w))
            ops._sk_let_go()
    for _ in range(3):
        for y in got:
            y.zero_()
        graph.replay()
        assert all(torch.equal(y, z) for y, z in zip(got, want))
        assert all(torch.equal(run(w), z) for w, z in zip(ws, want))
