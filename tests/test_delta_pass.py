"""The chunked delta rule's pass over feeds of every small number of chunks: the waves that form
the outputs take turns, their inputs are four turns ahead and what the chain leaves goes through
a ring of three, so each length ends in another place of all of them."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


@pytest.mark.gpu
@pytest.mark.parametrize("D,Dv", [(64, 3), (128, 17), (256, 32)])
@pytest.mark.parametrize("off", [0, 1, 15])
def test_feeds_of_few_chunks(D, Dv, off):
    H, B = 2, 13
    lens = [16 * n + 16 - off for n in range(B)]
    T, g = sum(lens), torch.Generator().manual_seed(D + off)
    q, k = (torch.nn.functional.normalize(torch.randn(T, H, D, generator=g), dim=-1) for _ in range(2))
    v, dec = torch.randn(T, H, Dv, generator=g), torch.rand(T, H, D, generator=g) ** 0.1
    act = torch.cat([x.reshape(T, -1) for x in (q, k, v, dec)], 1).cuda()
    tok = torch.stack([torch.ones(T, H), torch.rand(T, H, generator=g)], -1).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    pos = torch.cat([torch.arange(n) + (b % 3) * 5 for b, n in enumerate(lens)]).int().cuda()
    slots = torch.randperm(B, generator=g).int().cuda()
    state = torch.randn(B, H, Dv, D, generator=g)
    got = []
    for chunked in (True, False):
        s = state.cuda()
        got.append((seqmix.delta_scan(act, H, D, Dv, 0, H * D, 2 * H * D, 1, s, slots, cu, pos, tok,
                                      g_off=2 * H * D + H * Dv, chunked=chunked), s))
    for x, y in zip(*got):       # the same f32 sums in another order, over at most 208 tokens
        assert (x - y).abs().max() < 3e-5 * max(1.0, float(y.abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("chan", [True, False])
@pytest.mark.parametrize("D,Dv,hpg,shift", [(64, 64, 2, 0), (20, 1, 1, 0), (66, 37, 2, 0), (128, 200, 1, 0), (128, 128, 2, 3), (130, 70, 1, 0),
                                            (256, 300, 2, 0), (192, 64, 1, 1)])
def test_block_columns_and_alignments(D, Dv, hpg, shift, chan):
    # key and value columns over whole and part waves, rows in 16-byte pieces and off them
    H, lens = 4, [65, 16, 47]
    T, G, g = sum(lens), 4 // hpg, torch.Generator().manual_seed(D + Dv)
    q, k = (torch.nn.functional.normalize(torch.randn(T, G, D, generator=g), dim=-1) for _ in range(2))
    parts = [torch.zeros(T, shift), q, k, torch.randn(T, H, Dv, generator=g)] + [torch.rand(T, H, D, generator=g) ** 0.1] * chan
    act = torch.cat([x.reshape(T, -1) for x in parts], 1).cuda()
    tok = torch.stack([torch.rand(T, H, generator=g) ** 0.1, torch.rand(T, H, generator=g)], -1).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    pos = torch.cat([torch.arange(n) + b for b, n in enumerate(lens)]).int().cuda()
    slots, state = torch.arange(3).int().cuda(), torch.randn(3, H, Dv, D, generator=g)
    got = []
    for chunked in (True, False):
        s = state.cuda()
        got.append((seqmix.delta_scan(act, H, D, Dv, shift, shift + G * D, shift + 2 * G * D, hpg, s, slots, cu, pos, tok,
                                      g_off=shift + 2 * G * D + H * Dv if chan else None, chunked=chunked), s))
    for x, y in zip(*got):       # the same f32 sums in another order, over at most 65 tokens
        assert (x - y).abs().max() < 3e-5 * max(1.0, float(y.abs().max()))
