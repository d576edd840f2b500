"""Keys and values straight from latent pages (csrc/kernels/latent_kv.hip) and queries turned in the
prompt attention's launch: ragged and empty sequences, row counts around the tiles' edges, contexts
longer than what is gathered, each tile size."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix


def _pages(lens, ctx, blk, W, g):
    need = [-(-c // blk) for c in ctx]
    order = torch.randperm(sum(need) + 2, generator=g).int()
    bt, at = torch.zeros(len(lens), max(need) + 1, dtype=torch.int32), 0
    for b, n in enumerate(need):
        bt[b, :n] = order[at:at + n]
        at += n
    return torch.randn(len(order), blk, W, generator=g).bfloat16().cuda(), bt.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", sorted(seqmix.KV_LAYOUTS))
@pytest.mark.parametrize("H,DK,DV,D,R,Dr", [(8, 192, 128, 128, 512, 64), (4, 64, 64, 32, 64, 16), (2, 256, 128, 160, 128, 48),
                                            (8, 128, 64, 128, 192, 0)])
@pytest.mark.parametrize("lens", [(1,), (191,), (0, 65, 0, 1, 130), (64, 128, 0), (7,) * 33])
def test_keys_values(layout, H, DK, DV, D, R, Dr, lens, monkeypatch):
    bn = seqmix.KV_LAYOUTS[layout][0]
    if H * DK % bn or H * DV % bn:
        pytest.skip("no whole tiles")
    monkeypatch.setattr(seqmix, "KV_LAYOUTS", {layout: seqmix.KV_LAYOUTS[layout]})
    g = torch.Generator().manual_seed(sum(lens) + R + layout)
    ctx = [n + 5 * (i % 3) for i, n in enumerate(lens)]
    pages, bt = _pages(lens, ctx, 16, R + Dr, g)
    w = torch.randn(H * (DK + DV), R, generator=g) * R ** -0.5
    w.view(-1)[:H * DK * R].view(H, DK, R)[:, D:] = 0
    w = w.bfloat16().cuda()
    cu = torch.tensor([0] + list(lens)).cumsum(0).int().cuda()
    lens_d, total = torch.tensor(ctx).int().cuda(), sum(lens)
    k, v = seqmix.latent_keys_values(pages, bt, cu, lens_d, total, max(ctx), w, H, DK, DV, D)
    cl, kr = seqmix.latent_gather(pages, bt, cu, lens_d, total, max(ctx), R)
    for got, part in ((k, w[:H * DK]), (v, w[H * DK:])):
        want = (cl.double() @ part.double().t()).view(total, H, -1)
        if got is k:
            assert torch.equal(k[:, :, D:D + Dr], kr[:, None].expand(-1, H, -1))
            assert not k[:, :, D + Dr:].any()
            got, want = k[:, :, :D], want[:, :, :D]
        # bf16's half ulp and the f32 sum of R products
        assert torch.all((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5)


@pytest.mark.parametrize("case", ["fits", "rank", "rotary part", "tiles", "head width", "all heads' rows", "cache size", "no rows"])
def test_which_form(case, monkeypatch):
    """Everything that the launch refuses is gathered and multiplied, nothing else is."""
    H, DK, DV, D, R, Dr, blocks, total, dev = 4, 192, 128, 128, 512, 64, 8, 5, "cpu"
    if case == "rank":
        R = 520
    elif case == "rotary part":
        Dr, D = 80, 112
    elif case == "tiles":
        H, DK, DV, D = 1, 192, 32, 128
    elif case == "head width":
        H, DK, D, Dr = 16, 136, 64, 64
    elif case == "all heads' rows":
        H, DK, DV, D, R, Dr, dev = 8192, 64, 64, 32, 64, 16, "meta"
    elif case == "cache size":
        blocks, dev = 1 << 18, "meta"
    elif case == "no rows":
        total = 0
    cache = torch.zeros(blocks, 16, R + Dr, dtype=torch.bfloat16, device=dev)
    w = torch.zeros(H * (DK + DV), R, dtype=torch.bfloat16, device=dev)

    class Gathered(Exception):
        pass

    def gather(*a):
        raise Gathered
    monkeypatch.setattr(seqmix, "latent_gather", gather)
    i32 = torch.zeros(2, dtype=torch.int32)
    # (past the rule the launch wants GPU tensors)
    with pytest.raises(AssertionError if case == "fits" else Gathered):
        seqmix.latent_keys_values(cache, i32[None, :1], i32, i32[:1], total, 5, w, H, DK, DV, D)


@pytest.mark.gpu
@pytest.mark.parametrize("off,dims", [(128, 64), (128, 32), (64, 40), (130, 12)])
def test_queries_turned_in_the_launch(off, dims):
    g = torch.Generator().manual_seed(dims)
    lens, H, DK, DV = (70, 1, 33), 4, 192, 128
    T = sum(lens)
    q, k = (torch.randn(T, H, DK, generator=g).bfloat16().cuda() for _ in range(2))
    v = torch.randn(T, H, DV, generator=g).bfloat16().cuda()
    cu = torch.tensor([0] + list(lens)).cumsum(0).int().cuda()
    pos = torch.cat([torch.arange(n) for n in lens]).int().cuda()
    ctx = torch.tensor(lens).int().cuda()
    cs = seqmix.rope_table_pairs(dims, 64, 10000.0, None, "cuda")     # shorter than the longest position: clamped
    keep = q.clone()
    y = seqmix.latent_prefill(q, k, v, cu, cu, ctx, pos, None, DK ** -0.5, max(lens), DV, rot=(off, dims, cs))
    assert torch.equal(q, keep)
    seqmix.rope_pairs_(q, off, dims, pos, cs)
    want = seqmix.latent_prefill(q, k, v, cu, cu, ctx, pos, None, DK ** -0.5, max(lens), DV)
    # the same f32 products, contracted in another order: a turned entry may round to its bf16 neighbour
    assert (y.double() - want.double()).norm() <= 2.0 ** -9 * want.double().norm()
