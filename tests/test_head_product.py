"""A product per head for few rows (``seqmix.head_product``)."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


@pytest.mark.parametrize("T", [0, 1, 5])
def test_host(T):
    x, w = torch.randn(T, 3, 128).bfloat16(), torch.randn(3, 128, 64).bfloat16()
    assert torch.equal(seqmix.head_product(x, w), torch.bmm(x.transpose(0, 1), w).transpose(0, 1))


def _close(y, x, w):
    # an output is rounded once (2^-8 of it at most) after f32 sums, whose error is below K 2^-24 of the sum of magnitudes
    exact, mag = (torch.bmm(f(x.double()).transpose(0, 1), f(w.double())).transpose(0, 1) for f in (lambda a: a, torch.abs))
    assert ((y.double() - exact).abs() <= 2.0 ** -8 * 1.01 * exact.abs() + x.shape[2] * 2.0 ** -24 * mag).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 15, 31, 32, 33, 64, 65])
@pytest.mark.parametrize("K,N", [(128, 512), (256, 64), (384, 128), (512, 128), (64, 64), (640, 64), (128, 96)])
def test_rows(T, K, N):
    """Rows around a block's edges, every number of steps, sizes that stay with the vendor's, and rows that are a part of wider ones."""
    g = torch.Generator(device="cuda").manual_seed(T + K + N)
    wide = torch.randn(T, 3, K + 64, generator=g, device="cuda").bfloat16()
    w = torch.randn(3, K, N, generator=g, device="cuda").bfloat16()
    for x in (wide[:, :, :K], wide.transpose(0, 1).contiguous().transpose(0, 1)[:, :, 4:K + 4]):
        y = seqmix.head_product(x, w)
        assert y.shape == (T, 3, N)
        _close(y, x, w)
    wide[0, 0, 0] = float("inf")
    y = seqmix.head_product(wide[:, :, :K], w)
    assert not torch.isfinite(y[0, 0]).any() and torch.isfinite(y[1:]).all() and torch.isfinite(y[:, 1:]).all()
