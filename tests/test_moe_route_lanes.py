"""Router decisions with a token's scores in 16 to 64 lanes (moe.hip): output counts around each lane
count, groups with and without a limit, last workgroups with one token, against the reference."""
import pytest
import torch

from loqa_hub_amd.ops import reference as ref
from loqa_hub_amd.ops import seqmix


@pytest.mark.gpu
@pytest.mark.parametrize("E,G,keep,top", [(1, 1, 1, 1), (5, 5, 2, 2), (16, 4, 2, 4), (16, 1, 1, 16), (17, 1, 1, 3), (32, 2, 1, 4),
                                          (33, 11, 4, 2), (64, 8, 3, 8), (64, 1, 1, 64), (65, 5, 2, 4)])
@pytest.mark.parametrize("T", [1, 15, 17, 65])
def test_route(E, G, keep, top, T):
    g = torch.Generator().manual_seed(E * 100 + T)
    z, b, c = torch.randn(T, E, generator=g) * 2, torch.randn(E, generator=g), torch.rand(E, generator=g)
    for corr in (None, c):
        for kw in ({}, {"sigmoid": True, "renorm": True, "weight_scale": 2.5}, {"group_rank": 2, "weight_scale": 0.5},
                   {"top_softmax": True, "bias": b}):
            if kw.get("top_softmax") and (G > 1 or corr is not None):
                continue
            kd = {k: v.cuda() if torch.is_tensor(v) else v for k, v in kw.items()}
            i, w = seqmix.moe_route(z.cuda(), None if corr is None else corr.cuda(), G, keep, top, **kd)
            ri, rw = ref.moe_route(z, corr, G, keep, top, **kw)
            # f32 on both sides: expf, the sums' and the quotient's roundings, 2^-20 of a weight (at
            # most 64 addends); choices could differ only between scores as close as that
            assert torch.equal(i.cpu(), ri)
            assert torch.all((w.cpu().double() - rw.double()).abs() <= rw.double().abs() * 2.0 ** -20)
