"""The prompt form of qk_prep_append (csrc/kernels/attn_window.hip: eight entries a lane) against
the general form, which passes of fewer than 256 tokens take: every option that both accept.

The two add a head's squares in another order (f32), so a result may round the other way: one
bf16 step, 2^-7 of the value."""
import pytest
import torch

from loqa_hub_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,G", [(1, 1), (3, 1), (16, 4), (7, 7)])
@pytest.mark.parametrize("mode", ["head", "weights", "none", "keys as values", "temperature", "mix", "odd view"])
def test_against_the_general_form(D, H, G, mode):
    g = torch.Generator().manual_seed(D + H)
    T, blk = 300, 16
    dims = {"none": 0, "head": D, "weights": 2}.get(mode, 32)
    own = mode != "keys as values"
    Dv = 40 if mode == "mix" and G % 2 == 0 else D
    W = (H + G) * D + (G * Dv if own else 0)
    pad = 4 if mode == "odd view" else 0           # rows off 16 bytes: the general form at any length
    u = torch.randn(T, W + pad, generator=g).bfloat16().to(DEV)[:, :W]
    table = seqmix.rope_table_pairs(dims, 512, 10000.0, None, DEV) if dims else None
    slots = torch.randperm(T + 20, generator=g)[:T].int()
    slots[5] = -1
    pos = torch.arange(T, dtype=torch.int32) + 40
    wq = torch.rand(D, generator=g).to(DEV) if mode == "weights" else None
    wk = torch.rand(D, generator=g).to(DEV) if mode == "weights" else None
    mix = (torch.randn(T, G * Dv, generator=g).bfloat16().to(DEV), 0.25) if mode == "mix" else None
    temp = (0.1, 64) if mode == "temperature" else None

    def run(rows):
        kc = torch.zeros(-(-(T + 20) // blk), blk, G * D, dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros(-(-(T + 20) // blk), blk, G * Dv, dtype=torch.bfloat16, device=DEV)
        q = [seqmix.qk_prep_append(u[s:s + rows], H, G, D, Dv, (H + G) * D if own else -1, table, dims, 1e-6, temp, pos[s:s + rows].to(DEV),
                                   kc, vc, slots[s:s + rows].to(DEV), torch.bfloat16, q_norm=wq, k_norm=wk,
                                   v_mix=(mix[0][s:s + rows], mix[1]) if mix else None, norm=mode != "none") for s in range(0, T, rows)]
        return torch.cat(q), kc, vc
    for a, b in zip(run(T), run(100)):
        assert ((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs()).all()
