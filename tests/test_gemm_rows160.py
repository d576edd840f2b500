"""The pipelined tiles of 160 rows: where they are chosen, and that they are the product."""
import pytest
import torch

from loqa_hub_amd import ops

LAYOUTS = sorted(ops.SK_ROWS160)


def _close(a, b, k):
    # as in test_gemm_pipe.py: half a bf16 ulp of the value, and the f32 sum's own rounding
    tol = 2.0 ** -8 * b.abs() + (k * 2.0 ** -22 + 2.0 ** -9) * b.std()
    assert torch.all((a.double() - b).abs() <= tol), ((a.double() - b).abs() - tol).max().item()


def test_choice():
    """The plan stands where its time is less, where the pipelined tiles do not go, and where a caller asks for it; whole
    chunks on one round of the compute units."""
    taken = 0
    for M in (1, 100, 160, 161, 300, 320, 321, 640, 1500, 3000):
        for N, K in ((28672, 4096), (6144, 4096), (4096, 14336), (11264, 2048), (1280, 1280), (1088, 512), (192, 64)):
            for gelu in (False, True):
                plan, (lay, s) = ops._sk_plan(M, N, K, True, None, gelu), ops._sk_choice(M, N, K, True, gelu)
                assert ops._sk_choice(M, N, K, False, gelu) == ops._sk_plan(M, N, K, False, None, gelu)
                if (lay, s) == plan:
                    continue
                taken += 1
                bn, bm = ops.SK_ROWS160[lay][:2]
                assert N % bn == 0 and K // 64 // s >= 1 and (s == 1 or -(-M // bm) * (N // bn) * s <= ops.SK_CUS)
                assert ops._sk_us(lay, M, N, K, s, gelu) < ops._sk_us(*plan[:1], M, N, K, plan[1], gelu)
    assert taken and ops._sk_choice(320, 28672, 4096, True) == (21, 1)


@pytest.mark.parametrize("M,N,K,want", [(257, 4096, 14336, (17, 4)), (320, 4096, 14336, (17, 4)), (320, 4096, 4096, (17, 4)),
                                        (1600, 3072, 8192, (17, 1)), (2432, 2048, 8192, (17, 1)), (1599, 2048, 5632, (20, 1)),
                                        (160, 4096, 14336, (22, 8)), (161, 4096, 14336, (17, 8)), (640, 4096, 14336, (21, 4)), (1280, 2048, 8192, (21, 4))])
def test_chunks_that_a_pass_pays_for(M, N, K, want):
    """At most one chunk more than the plan's and none where it has none; 128 x 160 for one tile of rows."""
    assert ops._sk_choice(M, N, K, True) == want


@pytest.mark.gpu
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("stages,splits", [(1, 1), (2, 1), (7, 1), (7, 2), (14, 5), (14, 9)])
def test_tiles(layout, stages, splits):
    """Fewer K steps than the rings hold and more, rows around the tile's edge, K chunks with shares and without, every epilogue."""
    bn, bm = ops.SK_ROWS160[layout][:2]
    K, N = 64 * stages, 2 * bn
    g = torch.Generator().manual_seed(layout + stages)
    for M in (1, bm - 1, bm, bm + 1, 2 * bm + 17):
        x = torch.randn(M, K + 24, generator=g).bfloat16().cuda()[:, 8:8 + K]
        w, b = (torch.randn(N, K, generator=g) / 8).bfloat16().cuda(), torch.randn(N, generator=g).cuda()
        z = x.double() @ w.double().t()
        wide = torch.full((M, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
        _close(ops.gemm_sk(x, w, bias=b, layout=layout, splits=splits, out=wide[:, 32:32 + N]), z + b.double(), K)
        assert (wide[:, :32] == 7).all() and (wide[:, 32 + N:] == 7).all()
        v = z + b.double()
        _close(ops.gemm_sk(x, w, bias=b, act="gelu", layout=layout, splits=splits), 0.5 * v * torch.erfc(-v * 0.5 ** 0.5), K)
        res = torch.randn(M, N, generator=g).bfloat16().cuda()
        want = res.double() + z
        _close(ops.gemm_sk(x, w, epi="resid", residual=res, layout=layout, splits=splits), want, K)
        h = z[:, :bn]
        _close(ops.gemm_sk(x, w, epi="swiglu", layout=layout, splits=splits), h * torch.sigmoid(h) * z[:, bn:], K)
    torch.cuda.synchronize()
    assert all(int(cnt.abs().sum()) == 0 for _, cnt in ops._SK_WS.values())
