"""Rotation and cache append in 16-byte pieces (elementwise.hip): head widths and counts at the edges of
a workgroup's passes, rows of a wider tensor, rows 8 bytes off (which keep the general kernels),
padding rows and no rotation, against 64 bits."""
import pytest
import torch

from loqa_hub_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D", [(1, 1, 16), (32, 8, 128), (33, 8, 128), (20, 20, 64), (6, 1, 256), (64, 16, 128),
                                   (65, 16, 128), (9, 3, 32), (5, 1, 512), (24, 8, 96), (24, 16, 96), (7, 7, 40)])
@pytest.mark.parametrize("off", [0, 8, 4])
@pytest.mark.parametrize("rot", [True, False])
def test_rope_runs(H, G, D, off, rot):
    T, blk, N = 37, 16, (H + 2 * G) * D
    g = torch.Generator().manual_seed(H * D + off)
    wide = torch.randn(T, N + 24, generator=g).bfloat16()
    pos, slots = torch.randint(0, 400, (T,), generator=g, dtype=torch.int32), torch.randperm(8 * blk, generator=g)[:T].int()
    slots[5] = -1
    ang = torch.rand(400, D // 2, generator=g) * 6
    cs = torch.stack([ang.cos(), ang.sin()], -1)
    kc, vc = torch.randn(8, G, blk, D, generator=g).bfloat16(), torch.randn(8, G, blk, D, generator=g).bfloat16()
    dev, dk, dv = wide.cuda(), kc.cuda(), vc.cuda()
    ops.rope_kv_append(dev[:, off:off + N], pos.cuda() if rot else None, cs.cuda() if rot else None, dk, dv, slots.cuda(), H, G, D)
    x = wide[:, off:off + N].double().view(T, H + 2 * G, D).clone()
    if rot:
        a, b = x[:, :H + G, :D // 2].clone(), x[:, :H + G, D // 2:].clone()
        c, s = cs[pos.long()].double()[:, None].unbind(-1)
        x[:, :H + G] = torch.cat([a * c - b * s, b * c + a * s], -1)
    want = wide.double().clone()
    want[:, off:off + H * D] = x[:, :H].reshape(T, H * D)
    wk, wv = kc.double().clone(), vc.double().clone()
    for t in range(T):
        if slots[t] >= 0:
            p, o = divmod(int(slots[t]), blk)
            wk[p, :, o], wv[p, :, o] = x[t, H:H + G], x[t, H + G:]
    # half an ulp of bf16 is 2^-8 of the value at most; the f32 products' roundings beside it
    for got, ref in ((dev, want), (dk, wk)):
        assert torch.all((got.cpu().double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-6)
    assert torch.equal(dv.cpu().double(), wv)
    if not rot:
        assert torch.equal(dev.cpu(), wide) and torch.equal(dk.cpu().double(), wk)
