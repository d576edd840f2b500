"""Norms with a wave per row (norm.hip): widths around a piece's and a lane's edge, rows around a
workgroup's, both sides of the rule that chooses between a wave and a workgroup."""
import pytest
import torch

from loqa_hub_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("d", [8, 504, 512, 520, 1280, 3072, 3080, 4096, 4104])
@pytest.mark.parametrize("rows", [1, 5, 1023, 1300, 1799, 2050])
def test_norms(rows, d):
    g = torch.Generator().manual_seed(rows * 7 + d)
    x, r = ((torch.randn(rows, d, generator=g) + 0.5).bfloat16().cuda() for _ in range(2))
    w, b = (torch.randn(d, generator=g).bfloat16().cuda() for _ in range(2))
    idx = torch.randint(0, rows, (min(rows, 70),), generator=g).cuda()

    def want(v, ln):
        v = v.double()
        v = v - v.mean(-1, keepdim=True) if ln else v
        y = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-5) * w.double()
        return y + b.double() if ln else y

    def check(y, v, ln):
        # bf16's half ulp, and f32 sums of d values: a few 2^-24 of the terms w and b scale
        t = want(v, ln)
        assert torch.all((y.double() - t).abs() <= 2.0 ** -8 * t.abs() + 1e-5 * (1 + b.double().abs() + t.abs().amax()))
    for ln in (True, False):
        f = (lambda v, **k: ops.layernorm(v, w, b, 1e-5, **k)) if ln else (lambda v, **k: ops.rmsnorm(v, w, 1e-5, **k))
        check(f(x), x, ln)
        check(f(x, row_idx=idx), x[idx], ln)
        s = r.clone()
        y = f(x, residual=s)
        assert torch.equal(s, (x.float() + r.float()).bfloat16())
        check(y, s, ln)


@pytest.mark.gpu
@pytest.mark.parametrize("ln", [False, True])
@pytest.mark.parametrize("d", [2048, 3072, 4096])
def test_small_entries_behind_a_large_one(ln, d):
    """Squares of 1 behind one of 2^24 in a lane's chain round away one by one; a piece's own sum does not. eps
    leaves a ten-thousandth of the mean square, so that what the sum lost shows in bf16."""
    x = torch.ones(2048, d)
    x[:, 7:512:8] = 4096
    if ln:
        x.view(2048, -1, 2, 8)[:, :, 1] *= -1      # a mean of 0
    v = x.double()
    v = v - v.mean(-1, keepdim=True) if ln else v
    ms = v.square().mean(-1, keepdim=True)
    eps = -float(ms[0]) * (1 - 1e-4)
    w, b = torch.ones(d).bfloat16().cuda(), torch.zeros(d).bfloat16().cuda()
    xd = x.bfloat16().cuda()
    y = (ops.layernorm(xd, w, b, eps) if ln else ops.rmsnorm(xd, w, eps)).double().cpu()
    want = v / (ms + torch.tensor(eps, dtype=torch.float32).double()).sqrt()
    # bf16's half ulp, and of the mean square 6 half ulps of f32 (7 squares of 1 rounded to even in a lane,
    # the lanes' sums, the quotient; one chain: 23, 39 and 55), ten thousand times, halved by the root
    assert torch.all((y - want).abs() <= (2.0 ** -8 + 6 * 2.0 ** -24 * 0.5e4) * want.abs())
