"""Grouped expert products through the ring of k-steps (csrc/gemm_tile.hip): experts with no rows, one row, and rows about the edges of
64- and 128-row tiles, columns that end within a tile, fewer k-steps than the ring is deep, against plain products in 32 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

RAGGED = [0, 1, 63, 64, 65, 127, 128, 129, 200, 17]


@pytest.mark.parametrize("kind", ["gelu", "weighted gelu", "interleaved", "silu", "weighted"])
# rows of each expert, F, K, rows of a tile
@pytest.mark.parametrize("counts,F,K,tile", [(RAGGED, 64, 64, 64), (RAGGED, 192, 128, 64), (RAGGED, 320, 1024, 64), ([9, 30], 128, 192, 64),
                                             ([64] * 60 + [1, 127, 128, 0], 832, 64, 128), ([100] * 40 + RAGGED, 576, 320, 128),
                                             ([70] * 32, 64, 256, 64), ([300, 400, 129, 500, 1, 200, 64, 350], 256, 256, 64), ([20] * 60, 896, 64, 64)])
@pytest.mark.parametrize("ring", [3, 1, 2])  # both products through it, or one beside the kernel without it (64 rows)
def test_ring_of_steps(kind, counts, F, K, tile, ring, monkeypatch):
    from llmss_amd.ops import glu_interleave, hip
    if ring != 3 and tile == 128:
        pytest.skip("128 rows: both")
    E, P = len(counts), sum(counts)
    assert P > hip.MOE_DEC_ROWS * E
    plans = []
    monkeypatch.setattr(hip, "_moe_plan", lambda *a: plans.append(a) or (tile, ring))
    g = torch.Generator().manual_seed(P + F)
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P, generator=g)].int().view(P, 1).cuda()
    wide = torch.randn(P, K + 8, generator=g).bfloat16().cuda()
    h, w = wide[:, :K], torch.rand(P, 1, generator=g).cuda() + 0.5
    gate, up, down = (torch.randn(E, a, b, generator=g).mul(b ** -0.5).bfloat16().cuda() for a, b in ((F, K), (F, K), (K, F)))
    if "gelu" in kind:
        y = hip.moe_experts(h, idx, w, None, up, down, 0.0, 0.0, act="gelu", weight_input="weighted" in kind)
    elif kind == "interleaved":
        y = hip.moe_experts(h, idx, w, None, glu_interleave(gate, up, 1).contiguous(), down, 0.0, 0.0, act="silu", interleaved=True)
    else:
        y = hip.moe_experts(h, idx, w, gate, up, down, 0.0, 0.0, act="silu", weight_input=kind == "weighted")
    assert len(plans) == 1 and not (kind == "weighted gelu" and plans[0][-1])  # (256 x 256 tiles without a gate do not weight their inputs)
    want = torch.zeros(P, K, device="cuda")
    for e in range(E):
        r = (idx[:, 0] == e).nonzero()[:, 0]
        s = w[r] if "weighted" in kind else 1.0
        u = h[r].float() @ up[e].float().t() * s
        a = torch.nn.functional.gelu(u) if "gelu" in kind else torch.nn.functional.silu(h[r].float() @ gate[e].float().t() * s) * u
        want[r] = a.bfloat16().float() @ down[e].float().t() * (1.0 if "weighted" in kind else w[r])
    # sums in 32 bits on both sides; an activation that lies near the middle of two bf16 numbers may round to the other (2^-8 of it, few do)
    assert ((y - want).norm() / want.norm()).item() < 2.0 ** -10
    assert (y - want).abs().max() <= 2.0 ** -7 * want.abs().max()
