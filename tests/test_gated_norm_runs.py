"""Grouped gated norms with several lanes a group (lightning.hip): every group width that takes them
and one on each side, counts of groups around the rule and a workgroup's, gates in a column slice."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


@pytest.mark.gpu
@pytest.mark.parametrize("per", [56, 64, 128, 256, 512, 520])
@pytest.mark.parametrize("T,groups", [(1023, 2), (683, 3), (2049, 1), (2900, 1)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_groups(per, T, groups, dt):
    g, n = torch.Generator().manual_seed(per + T), per * groups
    o, w = torch.randn(T, n, generator=g).cuda(), torch.randn(n, generator=g).cuda()
    wide = torch.randn(T, n + 24, generator=g).to(dt).cuda()
    for gate in (wide[:, 8:8 + n], wide[:, 3:3 + n]):
        z = gate.double()
        for kw, act, first in (({}, torch.sigmoid, False), ({"gate_act": "silu"}, torch.nn.functional.silu, False),
                               ({"silu_first": True}, torch.nn.functional.silu, True)):
            v = (o.double() * act(z) if first else o.double()).view(T, groups, per)
            want = (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-6)).view(T, n) * w.double()
            want = want if first else want * act(z)
            y = seqmix.gated_rmsnorm(o, w, gate, 1e-6, dt, groups=groups, **kw).double()
            # half an ulp of bf16 results, a few 2^-24 of f32 ones
            assert torch.all((y - want).abs() <= (2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20) * want.abs() + 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("per", [64, 128, 256, 512])
def test_small_entries_behind_a_large_one(per):
    """Squares of 1 behind one of 2^24 round away one by one in a chain. eps leaves a ten-thousandth of the mean
    square, so that what the sum lost shows."""
    T = 4096
    x = torch.ones(T, per)
    x[:, ::8] = 4096
    ms = x.double().square().mean(-1, keepdim=True)
    eps = -float(ms[0]) * (1 - 1e-4)
    o, w, z = x.cuda(), torch.ones(per).cuda(), torch.zeros(T, per).cuda()
    y = seqmix.gated_rmsnorm(o, w, z, eps, torch.float32).double().cpu()
    want = 0.5 * x.double() / (ms + torch.tensor(eps, dtype=torch.float32).double()).sqrt()
    # of the mean square 4 half ulps of f32 (a square of 1 a lane, the lanes' sums; a chain of eight: 7),
    # ten thousand times, halved by the root
    assert torch.all((y - want).abs() <= 4 * 2.0 ** -24 * 0.5e4 * want.abs())
