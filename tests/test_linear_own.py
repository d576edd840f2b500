"""Plain products (``ops.linear``): which of them the pipelined tiles take, and that those are the product."""
import pytest
import torch

from loqa_hub_amd import ops

gpu = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,own", [(32, 1024, 512, True), (1, 1024, 512, True), (32, 6144, 4096, False), (33, 6144, 4096, True),
                                       (0, 1024, 512, False), (512, 1024, 480, False), (64, 16384, 4160, True), (65, 16384, 4160, False),
                                       (512, 1088, 512, False), (512, 0, 512, False), (512, 128, 0, False), (1200, 16384, 4160, False),
                                       (1201, 16384, 4160, True), (1200, 16384, 4096, True)])
def test_shapes(M, N, K, own):
    assert ops._linear_shape(M, N, K) is own


@pytest.mark.parametrize("M,N,K,own", [(64, 8192, 4096, False), (64, 4096, 8192, True), (96, 2048, 4096, False), (400, 2048, 4096, True),  # 64 x 64 in chunks, and whole
                                       (320, 5120, 3072, False), (192, 5632, 2048, True), (193, 5632, 2048, False), (257, 4096, 2048, True),
                                       (257, 3072, 8192, False), (160, 3072, 8192, True), (1024, 2048, 5632, False),                       # 128 x 64
                                       (3500, 4096, 4096, False), (2048, 22016, 4096, True),                                               # 256 x 256
                                       (2048, 131072, 16384, False), (2048, 131072, 16320, True)])                                         # 2^31 entries
def test_what_the_vendor_keeps(M, N, K, own):
    assert ops._linear_shape(M, N, K) is own


@pytest.mark.parametrize("strides,whole,at,own", [((64, 1), True, 32, True), ((72, 1), True, 0, True), ((64, 2), True, 0, False),
                                                  ((56, 1), True, 0, False), ((0, 1), True, 0, False), ((68, 1), True, 0, False),
                                                  ((64, 1), False, 0, False), ((64, 1), True, 8, False), ((1 << 21, 1), True, 0, False)])
def test_places(strides, whole, at, own):
    assert ops._linear_places(strides, 64, whole, at) is own


def test_host_products_stay(monkeypatch):
    monkeypatch.setattr(ops, "gemm_sk", lambda *a, **k: pytest.fail("not on the host"))
    x, w = torch.randn(64, 128).bfloat16(), torch.randn(128, 128).bfloat16()
    assert torch.equal(ops.linear(x, w), torch.nn.functional.linear(x, w))
    g = torch.fx.symbolic_trace(lambda a, b: ops.linear(a, b))
    assert torch.equal(g(x, w), torch.nn.functional.linear(x, w))


def _operands(M, N, K, ld=None):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, ld or K, generator=g, device="cuda").bfloat16()[:, :K]
    return x, torch.randn(N, K, generator=g, device="cuda").bfloat16()


def _close(y, x, w):
    # an output is rounded once (2^-8 of it) after f32 sums: their error is below K 2^-24 of the sum of magnitudes, and the vendor's
    # order of adding has the same bound
    exact, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((y.double() - exact).abs() <= 2.0 ** -8 * exact.abs() * 1.01 + x.shape[1] * 2.0 ** -24 * mag).all()


@gpu
@pytest.mark.parametrize("M,N,K,ld", [(1, 256, 512, None), (33, 128, 64, None), (191, 1536, 1536, None), (257, 384, 576, 584), (1201, 256, 128, 160),
                                      (320, 1024, 5632, None)])
def test_own_products(M, N, K, ld):
    x, w = _operands(M, N, K, ld)
    assert ops._linear_own(x, w)
    _close(ops.linear(x, w), x, w)


@gpu
def test_what_stays_with_torch():
    x, w = _operands(96, 256, 128)
    off = torch.empty(96 * 128 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(96, 128).copy_(x)
    wide = torch.empty(96, 256, dtype=torch.bfloat16, device="cuda")[:, ::2].copy_(x)
    for a, b in ((off, w), (wide, w), (x[None], w), (x, w.t().contiguous().t()), (x.float(), w.float()), (x[:1].expand(96, 128), w)):
        assert not ops._linear_own(a, b)
        assert torch.equal(ops.linear(a, b), torch.nn.functional.linear(a, b))
    assert not ops._linear_own(x.to_sparse(), w) and not ops._linear_own(x, w.to_sparse())
    assert not ops._linear_own(torch._neg_view(x), w) and torch.equal(ops.linear(torch._neg_view(x), w), torch.nn.functional.linear(-x, w))
    leaf = w.clone().requires_grad_()
    ops.linear(x, leaf).float().sum().backward()
    assert leaf.grad is not None
    with torch.no_grad():
        assert ops._linear_own(x, leaf) and ops._linear_own(x, torch.nn.Parameter(w))
    assert torch.func.vmap(lambda a: ops.linear(a, w))(x[None].repeat(2, 1, 1)).shape == (2, 96, 256)
    _, tangent = torch.func.jvp(lambda a: ops.linear(a, w), (x,), (x,))
    _close(tangent, x, w)
    with torch.autocast("cuda", torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
