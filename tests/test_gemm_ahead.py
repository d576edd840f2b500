"""Weights touched ahead by a projection's launch (ops._ahead, gemm_pipe.hip): when, and that the
product does not notice."""
import pytest
import torch

from loqa_hub_amd import ops
from loqa_hub_amd.ops import _lib


def _params(N, K, layout=15, S=1):
    p = _lib.GemmSkParams()
    p.N, p.K, p.S, p.layout = N, K, S, layout
    return p


def test_what_is_touched():
    big, small = torch.empty(5120, 1280, dtype=torch.bfloat16), torch.empty(512, 2048, dtype=torch.bfloat16)

    def touched(p, ahead, tiles):
        ops._ahead(p, ahead, tiles)
        return p.ahead_wgs, [int(n) for n in p.ahead_bytes]
    assert touched(_params(5120, 1280), (big,), 240) == (16, [big.numel() * 2, 0])
    assert touched(_params(5120, 1280), (big, small), 240) == (16, [big.numel() * 2, small.numel() * 2])
    assert touched(_params(5120, 1280), (big,), 249) == (0, [0, 0])         # no compute units left
    assert touched(_params(5120, 1280), (big,), 244) == (0, [0, 0])         # too few: they would outlast the tiles
    assert touched(_params(5120, 1280), (big,), 720) == (0, [0, 0])         # several rounds of tiles
    assert touched(_params(512, 512), (small,), 96) == (0, [0, 0])          # small weights come by themselves
    assert touched(_params(28672, 4096, 13), (torch.empty(1, dtype=torch.bfloat16).expand(4096, 14336),), 224) == (0, [0, 0])
    assert touched(_params(5120, 1280), (big.t(),), 240) == (0, [0, 0])     # not one run of memory
    # a launch that its own weights keep the memory busy for
    assert touched(_params(28672, 4096, 13), (torch.empty(4096, 4096, dtype=torch.bfloat16),), 224) == (0, [0, 0])


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_only_tensors_of_the_same_device(device):
    """What is touched goes to the launch as an address: tensors elsewhere are refused before it."""
    x, w = torch.zeros(300, 1024, dtype=torch.bfloat16, device=device), torch.zeros(256, 1024, dtype=torch.bfloat16, device=device)
    here = torch.zeros(2_200_000, dtype=torch.bfloat16, device=device)
    others = [here.to("meta"), here.data_ptr(), None] + ([here.cpu()] if device == "cuda" else [])
    for call in (ops.proj, ops.gemm_sk):
        call(x, w, ahead=(here,))
        for bad in others:
            with pytest.raises(ValueError):
                call(x, w, ahead=(here, bad))


@pytest.mark.gpu
@pytest.mark.parametrize("layout", [k for k in sorted({**ops.SK_LAYOUTS, **ops.SK_ROWS160}) if k >= ops.SK_PIPE])
def test_product_is_the_same(layout, monkeypatch):
    g = torch.Generator().manual_seed(layout)
    x = torch.randn(300, 1024, generator=g).bfloat16().cuda()
    w = (torch.randn(768, 1024, generator=g) / 32).bfloat16().cuda()
    bias, old = torch.randn(768, generator=g).cuda(), torch.randn(300, 768, generator=g).bfloat16().cuda()
    later = torch.randn(2_200_001, generator=g).bfloat16().cuda()[:2_200_000 + layout % 2]   # off whole kilobytes
    seen, rule = [], ops._ahead

    def counted(p, *a):
        rule(p, *a)
        seen.append((p.ahead_wgs, sum(n > 0 for n in p.ahead_bytes)))
    monkeypatch.setattr(ops, "_ahead", counted)
    for splits in (1, 2) if layout != ops.SK_WHOLE else (1,):
        for kw in ({}, {"bias": bias}, {"act": "gelu"}, {"act": "gelu", "bias": bias}, {"epi": "swiglu"}, {"epi": "resid"},
                   {"epi": "resid", "bias": bias}):
            def call(**more):
                if kw.get("epi") == "resid":         # added to in place
                    more["residual"] = old.clone()
                return ops.gemm_sk(x, w, layout=layout, splits=splits, **kw, **more)
            want = call()
            keep = later.clone()
            for ahead in ((later,), (later, w), (w[:8], later[:2_100_000])):
                seen.clear()
                assert torch.equal(call(ahead=ahead), want)
                assert len(seen) == 1 and seen[0][0] >= ops.AHEAD_WGS[0] and seen[0][1] == len(ahead)
            assert torch.equal(later, keep)
