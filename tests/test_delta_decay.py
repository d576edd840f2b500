"""Decays of the delta rule's input stage, exp(a softplus(z)), over the range of their
pre-activations, per head and per channel, against 64 bits; infinities and NaN as the formula has them."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


@pytest.mark.gpu
@pytest.mark.parametrize("D", [128, 24])
@pytest.mark.parametrize("lo,hi", [(-104, -20), (-20, -2), (-2, 2), (2, 30), (30, 120)])
def test_decays(D, lo, hi):
    T, H, G = 200, 2, 1
    g = torch.Generator().manual_seed(D + lo + 200)
    z = torch.rand(T, H * D, generator=g) * (hi - lo) + lo
    z[0, :3] = torch.tensor([float("inf"), -float("inf"), float("nan")])
    z, a = z.cuda(), -(torch.rand(H, generator=g) * 4 + 0.01).cuda()
    C, i32 = (2 * G + H) * D, {"dtype": torch.int32, "device": "cuda"}
    where = (torch.zeros(1, **i32), torch.tensor([0, T], **i32), torch.arange(T, **i32))
    u, cw, tail = torch.zeros(T, C + H).bfloat16().cuda(), torch.zeros(4, C).cuda(), torch.zeros(1, 3, C).cuda()
    act, _ = seqmix.delta_prep(u, None, G, D, H, D, cw, tail, a, torch.zeros(H * D).cuda(), *where, chan=(z, C))
    gz = torch.cat([torch.zeros(T, H).cuda(), z[:, ::D]], 1)
    _, tok = seqmix.delta_prep(u, gz.contiguous(), G, D, H, D, cw, tail, a, torch.zeros(H).cuda(), *where)
    for y, v, an in ((act[:, C:], z, a.repeat_interleave(D)), (tok[:, :, 0], z[:, ::D], a)):
        x = an.double() * torch.nn.functional.softplus(v.double(), threshold=1e9)
        want = torch.exp(x)
        # the exponent in f32: a rounding of softplus (1.5 ulp) and of the product, and expf's own ulp
        tol = want * (2.0 ** -23 + x.abs() * 4 * 2.0 ** -24) + 2e-38
        ok = v.isfinite()
        assert torch.all(((y.double() - want).abs() <= tol) | ~ok)
    assert act[0, C].item() == 0.0 and act[0, C + 1].item() == 1.0 and act[0, C + 2].isnan()
