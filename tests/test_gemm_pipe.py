"""The pipelined tiles behind ops.gemm_sk (csrc/kernels/gemm_pipe.hip): which operands they
take, the edges of tiles and rings, and GELU at the ends of its range."""
import pytest
import torch

from loqa_hub_amd import ops


def _close(a, b, k):
    # a bf16 result of an f32 sum of k products: half an ulp (2^-9) of the value, and the sum's
    # own rounding, at most k 2^-24 of the magnitudes added (bounded by 4 sigma of the sum)
    tol = 2.0 ** -8 * b.abs() + (k * 2.0 ** -22 + 2.0 ** -9) * b.std()
    assert torch.all((a.double() - b).abs() <= tol), ((a.double() - b).abs() - tol).max().item()


def test_plan_takes_the_general_layouts_where_the_tiles_do_not_fit():
    for M, N, K in ((1, 64, 64), (300, 192, 256), (5000, 4160, 512)):
        assert N % 128 and ops.gemm_sk_plan(M, N, K)[0] == 7
    for M in (1, 64, 65, 320, 2048, 9000):
        for N, K in ((1280, 5120), (6144, 4096), (128, 64), (28672, 4096)):
            assert ops.gemm_sk_plan(M, N, K, pipe=False)[0] in (1, 7)
            lay, s = ops.gemm_sk_plan(M, N, K)
            assert lay >= ops.SK_PIPE and N % ops.SK_LAYOUTS[lay][0] == 0
            assert s == 1 or K // 64 // s >= 8


def test_plan_of_a_shape_is_made_once():
    M, N, K = 333, 6144, 4096
    plan = ops.gemm_sk_plan(M, N, K)
    made = ops._sk_plan.cache_info().misses
    assert [ops.gemm_sk_plan(M, N, K, epi) for epi in ("bf16", "resid", "swiglu")] == [plan] * 3
    assert ops._sk_plan.cache_info().misses == made
    assert ops.gemm_sk_plan(M, N, K, pipe=False) != plan and ops._sk_plan.__wrapped__(M, N, K, True) == plan


def test_plan_among_some_layouts():
    for layouts in ((0, 1, 2, 3, 4, 5), [12], (6,), (20, 7)):
        lay, _ = ops.gemm_sk_plan(300, 6144, 4096, "bf16", layouts)
        assert lay in {ops.SK_RENAMED.get(x, x) for x in layouts}
    assert ops.gemm_sk_plan(300, 6144, 4096, layouts=(0, 4), pipe=False)[0] in (1, 7)
    assert set(ops.SK_RENAMED) | set(ops.SK_LAYOUTS) == set(range(21))


def test_largest_tiles_are_not_split():
    # 1280 x 4096 x 14336: 160 us in three chunks of 256 x 256 tiles, 135 in two of 256 x 192
    for M in (1, 80, 640, 1000, 1280, 2048, 3000, 9000):
        for N, K in ((512, 2048), (1280, 5120), (4096, 4096), (4096, 14336), (7168, 8192), (8192, 28672)):
            lay, s = ops.gemm_sk_plan(M, N, K)
            assert lay != ops.SK_WHOLE or s == 1, (M, N, K)
    assert ops.gemm_sk_plan(1280, 4096, 14336) == (13, 2) and ops.gemm_sk_plan(2048, 4096, 14336) == (16, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", sorted(ops.SK_RENAMED))
@pytest.mark.parametrize("off", [0, 4])
def test_layout_numbers_that_are_gone(layout, off):
    """They still name a tile; output rows that are not 16-byte aligned take the general one."""
    g = torch.Generator().manual_seed(layout)
    x, w = torch.randn(150, 1024, generator=g).bfloat16().cuda(), (torch.randn(512, 1024, generator=g) / 32).bfloat16().cuda()
    for splits in (None, 1, 2):
        y = torch.zeros(150, 512 + off, dtype=torch.bfloat16, device="cuda")[:, :512]
        ops.gemm_sk(x, w, layout=layout, splits=splits, out=y)
        _close(y, x.double() @ w.double().t(), 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [k for k in sorted(ops.SK_LAYOUTS) if k >= ops.SK_PIPE])
@pytest.mark.parametrize("stages", [1, 2, 3, 7])
def test_short_k_and_ragged_rows(layout, stages):
    """Fewer K steps than the rings hold, rows around the tile's edge, rows wider than K, and
    an output that is a column block of a wider matrix."""
    bn, bm = ops.SK_LAYOUTS[layout][:2]
    K = 64 * stages
    g = torch.Generator().manual_seed(layout)
    for M in (1, bm - 1, bm, bm + 1):
        x = torch.randn(M, K + 24, generator=g).bfloat16().cuda()[:, 8:8 + K]
        w = torch.randn(2 * bn, K, generator=g).bfloat16().cuda()
        ref = x.double() @ w.double().t()
        wide = torch.full((M, 2 * bn + 64), 7.0, dtype=torch.bfloat16, device="cuda")
        y = ops.gemm_sk(x, w, layout=layout, splits=1, out=wide[:, 32:32 + 2 * bn])
        _close(y, ref, K)
        assert (wide[:, :32] == 7).all() and (wide[:, 32 + 2 * bn:] == 7).all()
        res = torch.randn(M, 2 * bn, generator=g).bfloat16().cuda()
        want = res.double() + ref
        _close(ops.gemm_sk(x, w, epi="resid", residual=res, layout=layout, splits=stages), want, K)
        h = ref[:, :bn]
        _close(ops.gemm_sk(x, w, epi="swiglu", layout=layout, splits=1), h * torch.sigmoid(h) * ref[:, bn:], K)


@pytest.mark.gpu
@pytest.mark.parametrize("epi", ["bf16", "resid", "swiglu"])
def test_rows_that_are_not_16_byte_aligned(epi):
    """Output rows 8 bytes apart from alignment take the general form: same result."""
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(150, 256, generator=g).bfloat16().cuda(), torch.randn(256, 256, generator=g).bfloat16().cuda()
    n = 128 if epi == "swiglu" else 256
    want = ops.gemm_sk(x, w, epi=epi, residual=torch.zeros(150, 256, dtype=torch.bfloat16, device="cuda") if epi == "resid" else None)
    wide = torch.zeros(150, n + 4, dtype=torch.bfloat16, device="cuda")
    y = ops.gemm_sk(x, w, epi=epi, residual=wide[:, :n] if epi == "resid" else None, out=None if epi == "resid" else wide[:, :n])
    _close(y, want.double(), 256)


@pytest.mark.gpu
@pytest.mark.parametrize("lo,hi,more", [(-13.1, -9, 0.006), (-9, -7, 0.001), (-7, -5, 0.0002), (-5, -0.001, 0.00002), (0.001, 9, 0.000002)])
def test_gelu_relative_error(lo, hi, more):
    """Relative to the value, down to the smallest ones that bf16 holds: its half ulp (2^-9 of the next power
    of two, 2^-8 of the value at most) and ``more``, the largest relative error of the f32 value with a margin of a
    fifth or more (measured 0.0048, 0.00065, 0.00016, 0.00001 and 0.0000003)."""
    b = torch.linspace(lo, hi, 4096).cuda()
    x, w = torch.zeros(1, 64, dtype=torch.bfloat16, device="cuda"), torch.zeros(4096, 64, dtype=torch.bfloat16, device="cuda")
    y, v = ops.gemm_sk(x, w, bias=b, act="gelu")[0].double(), b.double()
    want = 0.5 * v * torch.special.erfc(-v / 2 ** 0.5)
    assert torch.all((y - want).abs() <= (2.0 ** -8 + more * 1.01) * want.abs())


@pytest.mark.gpu
def test_gelu_over_its_whole_range():
    """gelu(b) for biases from the far negative tail to the largest finite value, and the
    infinities and NaN as 0.5 v (1 + erf(v / sqrt 2)) gives them."""
    b = torch.cat([torch.linspace(-8, 8, 1021), torch.tensor([3e38, 1e20, -1e20])]).cuda()
    x, w = torch.zeros(3, 64, dtype=torch.bfloat16, device="cuda"), torch.zeros(1024, 64, dtype=torch.bfloat16, device="cuda")
    y = ops.gemm_sk(x, w, bias=b, act="gelu")[1].double()
    v = b.double()
    want = 0.5 * v * torch.special.erfc(-v / 2 ** 0.5)
    # bf16's half ulp; f32 rounding, and values below bf16's normal ones (relative errors: above)
    assert torch.all((y - want).abs() <= 2.0 ** -8 * want.abs() + 1e-7 * v.abs().clamp(max=16))
    edge = torch.full((128,), float("inf"), device="cuda")
    edge[1], edge[2] = -float("inf"), float("nan")
    got = ops.gemm_sk(x, w[:128], bias=edge, act="gelu")[0]
    assert got[0] == float("inf") and got[1].isnan() and got[2].isnan()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(192 * 16 + 1, 2048, 128), (192 * 32 - 191, 2048, 64), (6000, 1280, 1280)])
def test_two_gelu_workgroups_on_a_compute_unit(M, N, K):
    """More 128 x 192 tiles than compute units: ragged rows, one and two K steps (fewer than stages), several rounds."""
    assert ops.SK_LAYOUTS[ops.SK_PAIRED][:2] == (128, 192) and -(-M // 192) * (N // 128) > ops.SK_CUS
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).cuda()
    y = ops.gemm_sk(x, w, bias=b, act="gelu", layout=ops.SK_PAIRED, splits=1)
    z = x.double() @ w.double().t() + b.double()
    want = 0.5 * z * torch.erfc(-z * 0.5 ** 0.5)
    # half a bf16 ulp of the value, and the f32 sum's own rounding
    assert torch.all((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (K * 2.0 ** -22 + 2.0 ** -9) * want.std())
    # every tile size sums a value's K steps in the same order
    assert torch.equal(y, ops.gemm_sk(x, w, bias=b, act="gelu", layout=20, splits=1))


def test_the_plan_with_gelu():
    for M, N, K in ((9000, 2048, 512), (12000, 3072, 768), (24000, 5120, 1280)):
        assert ops.gemm_sk_plan(M, N, K, "gelu") == (ops.SK_PAIRED, 1)
    for M, N, K in ((100, 2048, 512), (1500, 2048, 512), (6000, 5120, 1280)):
        assert ops.gemm_sk_plan(M, N, K, "gelu") == ops.gemm_sk_plan(M, N, K) and ops.gemm_sk_plan(M, N, K)[0] != ops.SK_PAIRED
    assert ops.gemm_sk_plan(9000, 1088, 512, "gelu")[0] in (1, 7)


def test_the_plan_takes_small_tiles_for_small_grids():
    for M, N, K in ((1500, 512, 512), (1500, 512, 2048), (300, 1280, 1280), (1500, 384, 1536)):
        assert ops.gemm_sk_plan(M, N, K) == (ops.SK_SMALL, 1)
    for M, N, K in ((1500, 768, 3072), (1500, 1280, 1280), (9000, 512, 512), (320, 4096, 14336)):
        assert ops.gemm_sk_plan(M, N, K)[0] != ops.SK_SMALL
    assert not ops.gemm_sk_plan(1500, 576, 2048)[0] >= ops.SK_PIPE          # whole 128 features, as every pipelined tile


def test_chunks_are_one_round():
    """Chunks beyond the compute units took 1.14 to 1.4 times the whole tiles' time, and many rows' whole tiles less than
    their chunks (1600 x 4096 x 14336: 238 us in five chunks, 167 whole)."""
    for M in (17, 160, 320, 640, 1100, 1600, 2200, 3300, 9000):
        for N, K in ((1280, 5120), (2048, 8192), (3072, 8192), (4096, 11008), (4096, 14336), (5120, 3072), (16384, 3072)):
            lay, s = ops.gemm_sk_plan(M, N, K)
            bn, bm = ops.SK_LAYOUTS[lay][:2]
            assert s == 1 or -(-M // bm) * (N // bn) * s <= ops.SK_CUS, (M, N, K, lay, s)
    for shape, plan in (((1600, 4096, 14336), (16, 1)), ((3300, 5120, 3072), (17, 1)), ((2200, 4096, 11008), (13, 1)), ((1100, 16384, 3072), (17, 1)),
                        ((1100, 4096, 11008), (13, 2)), ((2500, 2048, 8192), (17, 1)), ((320, 4096, 4096), (17, 4)), ((320, 4096, 14336), (17, 4))):
        assert ops.gemm_sk_plan(*shape) == plan, shape


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [None, 1, 2])
def test_small_tiles_by_number_take_what_their_number_took(splits):
    """11 named the 128 x 64 tiles before it named these: rows off 16 bytes still take the general form."""
    g = torch.Generator().manual_seed(11)
    x, w = torch.randn(150, 1024, generator=g).bfloat16().cuda(), (torch.randn(512, 1024, generator=g) / 32).bfloat16().cuda()
    for out in (None, torch.zeros(150, 516, dtype=torch.bfloat16, device="cuda")[:, :512]):
        _close(ops.gemm_sk(x, w, layout=ops.SK_SMALL, splits=splits, out=out), x.double() @ w.double().t(), 1024)
