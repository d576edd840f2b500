"""The encoder's conv stem on the pipelined tiles (csrc/kernels/conv_pipe.hip): windows that end
inside tiles, both strides, odd and even lengths, rows wider than the channels."""
import pytest
import torch

from loqa_hub_amd import ops


@pytest.mark.parametrize("device,layout", [("cpu", None)] + [pytest.param("cuda", n, marks=pytest.mark.gpu) for n in (None, *ops.CONV_LAYOUTS)])
@pytest.mark.parametrize("B,tin,cin,N,stride", [(1, 300, 128, 128, 1), (3, 97, 64, 256, 2), (5, 33, 128, 384, 1), (2, 1, 64, 128, 1),
                                                (70, 2, 64, 128, 2), (2, 3000, 128, 256, 1), (4, 1500, 512, 512, 2), (7, 190, 64, 512, 1),
                                                (130, 2, 64, 256, 2)])
def test_conv(device, layout, B, tin, cin, N, stride, monkeypatch):
    if layout is not None:
        if N % ops.SK_LAYOUTS[layout][0]:
            pytest.skip("no whole tiles")
        monkeypatch.setattr(ops, "CONV_LAYOUTS", (layout,))
    g = torch.Generator().manual_seed(tin + N)
    tout = (tin - 1) // stride + 1
    x = torch.randn(B * tin, cin + 16, generator=g).bfloat16()[:, 8:8 + cin]
    w = (torch.randn(N, cin, 3, generator=g) * (3 * cin) ** -0.5).bfloat16()
    bias, pos = torch.randn(N, generator=g) * 0.1, torch.randn(tout, N, generator=g).bfloat16()
    wt = ops.conv_k3_weight(w.reshape(N, -1), cin).to(device)
    v = torch.nn.functional.conv1d(x.double().view(B, tin, cin).transpose(1, 2), w.double(), bias.double(), stride, 1)
    a = v.transpose(1, 2).reshape(B * tout, N)
    v = torch.nn.functional.gelu(a)
    wide = torch.zeros(B * tin, cin + 16, dtype=torch.bfloat16)
    wide[:, 8:8 + cin] = x
    for xd in (wide.to(device)[:, 8:8 + cin], x.contiguous().to(device)):
        for p in (None, pos):
            want = v if p is None else v + p.double().repeat(B, 1)
            y = ops.conv_k3_gelu(xd, wt, bias.to(device), B, stride, pos=None if p is None else p.to(device)).double().cpu()
            # bf16 has 8 significant bits: half an ulp is at most 2^-8 of the value. That of the result
            # and, in the plain form, of GELU's
            # argument (times GELU's largest slope, 1.13) and of its value before the positions; f32
            # sums of 3 cin products
            tol = 2.0 ** -8 * (want.abs() + v.abs() + 1.13 * a.abs()) * 1.01 + 1e-5
            assert torch.all((y - want).abs() <= tol), (y - want).abs().max()


@pytest.mark.parametrize("case", ["fits", "features", "channels", "rows 8 bytes off", "weights 8 bytes off", "positions 8 bytes off",
                                  "row stride", "rows far apart", "short windows far apart"])
def test_which_kernel(case, monkeypatch):
    """Everything that the pipelined launch refuses goes to gemm_tile, nothing else does."""
    monkeypatch.setattr(ops, "_gpu", lambda x: True)
    monkeypatch.setattr(ops, "gemm_tile", lambda *a, **k: "gemm_tile")
    monkeypatch.setattr(ops, "stream_ptr", lambda x: 0)
    asked = []
    monkeypatch.setattr(ops, "check", lambda *a: None)
    monkeypatch.setattr(ops, "kernels", lambda: type("K", (), {"loqa_conv_pipe": lambda self, p, s: asked.append(p)})())
    N, cin, tin, ld, dev = 128, 64, 40, 64, "cpu"
    if case == "features":
        N = 192
    if case == "channels":
        cin = ld = 96
    if case == "row stride":
        ld = 68
    if case == "rows far apart":
        ld, dev = 1 << 21, "meta"
    if case == "short windows far apart":
        ld, tin, dev = (1 << 21) - 8, 1, "meta"

    def make(rows, cols, off=0):
        return torch.zeros(rows * cols + 16, dtype=torch.bfloat16, device=dev)[off:off + rows * cols].view(rows, cols)
    x = make(2 * tin, ld, 4 if case.startswith("rows 8") else 0)[:, :cin]
    w, pos = make(N, 3 * cin, 4 if case.startswith("weights") else 0), make(tin, N, 4 if case.startswith("positions") else 0)
    y = ops.conv_k3_gelu(x, w, torch.zeros(N), 2, 2 if tin == 1 or ld > 1 << 20 else 1, pos=pos)
    assert (y == "gemm_tile") if case != "fits" else (len(asked) == 1 and y.shape == (80, N))


def test_layouts_are_ranked_by_the_plans_times():
    """As a projection of whole tiles with GELU: its cost per value, and the longer steps of the 64 x 64 tiles from K = 2112 on."""
    assert ops._conv_layout(9000, 1024, 384, ops.CONV_LAYOUTS) == 20          # 27.5 us, 27.9 in 256 x 128
    assert ops._conv_layout(1500, 384, 1152, ops.CONV_LAYOUTS) == ops.SK_SMALL
    for M, N, K in ((1500, 512, 2304), (700, 768, 2304), (9000, 1280, 384), (24000, 1280, 3840)):
        best = min((lay for lay in ops.CONV_LAYOUTS if N % ops.SK_LAYOUTS[lay][0] == 0), key=lambda lay: ops._sk_us(lay, M, N, K, 1, True))
        assert ops._conv_layout(M, N, K, ops.CONV_LAYOUTS) == best
        assert ops._sk_plan(M, N, K, True, ops.CONV_LAYOUTS, True)[0] == best or ops._sk_plan(M, N, K, True, ops.CONV_LAYOUTS, True)[1] > 1
