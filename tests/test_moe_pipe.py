"""Grouped expert products on the pipelined tiles (csrc/kernels/moe_pipe.hip): experts without
tokens, segments around a tile's rows, feature counts that are no multiple of a tile, identity
experts, and the sizes the tiles do not take, against 64-bit products."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["swiglu", "clamped", "relu2"])
@pytest.mark.parametrize("T,d,F,E,top", [(1, 64, 8, 4, 1), (3, 192, 136, 5, 3), (65, 128, 264, 3, 2), (300, 256, 120, 16, 4),
                                         (1100, 128, 200, 4, 2), (2600, 64, 72, 2, 1), (70, 96, 64, 4, 2), (70, 64, 68, 4, 2)])
def test_experts_against_reference(act, T, d, F, E, top):
    g = torch.Generator().manual_seed(T + F)
    h = torch.randn(T, d, generator=g).bfloat16()
    # one expert gets no token, one nearly all; indices of E and more pass the input through
    idx = torch.stack([torch.randperm(E + 2, generator=g)[:top] for _ in range(T)]).int()
    idx[idx == 1] = 0
    idx[: T * 3 // 4, 0] = 2
    wt = torch.rand(T, top, generator=g)
    gated = act != "relu2"
    up = (torch.randn(E, 2 * F if gated else F, d, generator=g) * d ** -0.5).bfloat16()
    down = (torch.randn(E, d, F, generator=g) * F ** -0.5).bfloat16()
    limit = 1.0 if act == "clamped" else None
    want = torch.zeros(T, d, dtype=torch.float64)
    for e in range(E):
        for k in range(top):
            rows = (idx[:, k] == e).nonzero()[:, 0]
            a = h[rows].double() @ up[e].double().t()
            if act == "relu2":
                a = a.clamp(min=0).square()
            elif act == "swiglu":
                a = a[:, :F] * torch.sigmoid(a[:, :F]) * a[:, F:]
            else:
                gt = a[:, :F].clamp(max=limit)
                a = gt * torch.sigmoid(1.702 * gt) * (a[:, F:].clamp(-limit, limit) + 1)
            want[rows] += wt[rows, k, None] * (a @ down[e].double().t())
    want += ((idx >= E) * wt).sum(1, keepdim=True) * h.double()
    got = seqmix.moe_experts(h.cuda(), idx.cuda(), wt.cuda(), up.cuda(), down.cuda(), gated, limit).cpu()
    # the activation and an expert's output are rounded to bfloat16, by 2^-9 of each value at
    # most; f32 sums add far less
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("P,E", [(1, 1), (63, 64), (1025, 7), (9000, 130), (20000, 1023)])
def test_plan_is_a_permutation_by_expert(P, E):
    from loqa_hub_amd.ops._lib import check, kernels, ptr, stream_ptr
    idx = torch.randint(0, E + 3, (P,), dtype=torch.int32, generator=torch.Generator().manual_seed(P)).cuda()
    plan = torch.full((E + 2 + 2 * P,), -1, dtype=torch.int32, device="cuda")
    check(kernels().loqa_moe_plan(ptr(idx), P, E, ptr(plan), stream_ptr(idx)), "moe_plan")
    off, perm, pos = plan[:E + 2].cpu(), plan[E + 2:E + 2 + P].cpu().long(), plan[E + 2 + P:].cpu()
    e = idx.cpu().clamp(max=E).long()
    assert off.tolist() == [0] + torch.bincount(e, minlength=E + 1).cumsum(0).tolist()
    assert torch.equal(perm.sort().values, torch.arange(P)) and torch.equal(pos[perm], torch.arange(P, dtype=torch.int32))
    assert torch.equal(e[perm], e.sort().values)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 200])
@pytest.mark.parametrize("gated", [True, False])
def test_identity_experts_only(T, gated):
    h, wt = torch.randn(T, 64).bfloat16(), torch.rand(T, 2)
    up, down = torch.empty(0, 128 if gated else 64, 64).bfloat16(), torch.empty(0, 64, 64).bfloat16()
    got = seqmix.moe_experts(h.cuda(), torch.randint(0, 3, (T, 2), dtype=torch.int32).cuda(), wt.cuda(), up.cuda(), down.cuda(), gated)
    # two f32 products of 24 x 8 bits and their sum
    assert torch.allclose(got.cpu(), h.float() * wt.sum(1, keepdim=True), rtol=2.0 ** -21, atol=0)


@pytest.mark.gpu
def test_activation_keeps_32_bits():
    # gate sums of two columns, up products of one, an identity behind them: the output is the
    # activation itself, rounded to bfloat16
    T, F = 4096, 64
    a = -20 - 60 * torch.rand(T, F, generator=torch.Generator().manual_seed(0), dtype=torch.float64)
    hi = a.bfloat16()
    lo = (a - hi.double()).bfloat16()
    h = torch.cat([hi, lo, torch.ones(T, 1).bfloat16(), torch.zeros(T, F - 1).bfloat16()], 1)
    up, down = torch.zeros(1, 2 * F, 3 * F), torch.zeros(1, 3 * F, F)
    up[0, :F, :F] = up[0, :F, F:2 * F] = down[0, :F] = torch.eye(F)
    up[0, F:, 2 * F] = 1
    got = seqmix.moe_experts(h.cuda(), torch.zeros(T, 1, dtype=torch.int32).cuda(), torch.ones(T, 1).cuda(), up.bfloat16().cuda(),
                             down.bfloat16().cuda(), True).cpu()[:, :F]
    s = hi.double() + lo.double()
    want = (s * torch.sigmoid(s)).bfloat16().float()
    # an error of 2 ulp (exponential, sum and quotient: 2^-22) moves 2^-22 / 2^-8 of the values over
    # a rounding boundary at the most; sigmoid_fast's some 2e-4 of them
    assert (got != want).float().mean() <= 2.0 ** -14
