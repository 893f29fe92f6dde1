"""Expert products with a weight that does not start at a multiple of 16 bytes: every kernel choice takes them, with the results of
the aligned copy."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def shifted(t):  # the same numbers, two bytes further on
    s = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    s[1:] = t.flatten()
    return s[1:].view(t.shape)


# pairs per expert: few (16-row tiles), 128 and up (256-row tiles without a gate matrix), 256 and up (with one)
@pytest.mark.parametrize("T", [3, 130, 260, 400])
@pytest.mark.parametrize("kind", ["gelu", "interleaved", "silu"])
@pytest.mark.parametrize("which", ["up", "down", "gate"])
def test_weights_at_odd_places(T, kind, which):
    from llmss_amd.ops import glu_interleave, hip
    E, W, F = 2, 256, 256
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, W, generator=g).bfloat16().cuda()
    gate, up, down = ((torch.randn(*s, generator=g) * 0.06).bfloat16().cuda() for s in ((E, F, W), (E, F, W), (E, W, F)))
    if kind == "interleaved":
        gate, up = None, glu_interleave(gate, up, 1).contiguous()
    elif kind == "gelu":
        gate = None
    if which == "gate" and gate is None:
        return
    idx = torch.stack([torch.randperm(E, generator=g) for _ in range(T)]).int().cuda()
    w = torch.rand(T, E, generator=g).cuda()
    ws = {"gate": gate, "up": up, "down": down}

    def run(ws):
        return hip.moe_experts(h, idx, w, ws["gate"], ws["up"], ws["down"], 0.0, 0.0, act="gelu" if kind == "gelu" else "silu",
                               interleaved=kind == "interleaved")
    want = run(ws)
    got = run({**ws, which: shifted(ws[which])})
    # the same products with fp32 sums in another order, and one bf16 rounding of the activation rows (2^-9 each)
    assert ((got - want).norm() / want.norm()).item() < 2.0 ** -8
