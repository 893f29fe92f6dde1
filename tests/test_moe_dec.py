"""Grouped expert products of a few rows per expert (csrc/moe_dec.hip) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# K of one step up to more than a wave's eight, F that is no multiple of 128; one row, an expert with more rows than a tile, one with none
@pytest.mark.parametrize("E,top,W,F,T", [(4, 2, 32, 32, 1), (8, 2, 96, 160, 15), (5, 3, 1056, 96, 13), (40, 1, 2048, 768, 21)])
@pytest.mark.parametrize("kind", ["silu", "weighted", "clamp", "interleaved", "gelu"])
def test_moe_dec(E, top, W, F, T, kind, monkeypatch):
    from llmss_amd.ops import hip, glu_interleave
    g = torch.Generator().manual_seed(E + W + F)
    h = torch.randn(T, W + 8, generator=g).bfloat16().cuda()[:, :W]
    gate, up = ((torch.randn(E, F, W, generator=g) * W ** -0.5).bfloat16().cuda() for _ in range(2))
    down = (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16().cuda()
    idx = torch.stack([torch.randperm(E - 1, generator=g)[:top] for _ in range(T)]).int()
    idx[:, 0] = torch.where((idx[:, 1:] == 0).any(1), idx[:, 0], 0)  # most rows choose expert 0, nobody the last one
    idx = idx.cuda()
    w = torch.rand(T, top, generator=g).cuda()
    lib, calls = hip.lib(), []

    class Seen:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)
    monkeypatch.setattr(hip, "lib", Seen)
    weighted = kind == "weighted"
    act = {"clamp": "glu_clamp", "gelu": "gelu"}.get(kind, "silu")
    if kind == "interleaved":
        y = hip.moe_experts(h, idx, w, None, glu_interleave(gate, up, 1).contiguous(), down, 0.0, 0.0, act=act, interleaved=True)
    else:
        y = hip.moe_experts(h, idx, w, None if kind == "gelu" else gate, up, down, 1.5, 1.702, act=act, weight_input=weighted)
    assert calls.count("moe_dec") == 2
    want = torch.zeros(T, W, dtype=torch.float64, device="cuda")
    lim = torch.zeros_like(want)
    hd = h.double()
    for t in range(T):
        for j in range(top):
            e, s = int(idx[t, j]), w[t, j].double()
            a, b = gate[e].double() @ hd[t], up[e].double() @ hd[t]
            # fp32 sums in any order
            ea, eb = ((W + 8) * 2.0 ** -24 * (m[e].double().abs() @ hd[t].abs()) for m in (gate, up))
            if weighted:
                a, b, ea, eb = a * s, b * s, ea * s, eb * s
            if act == "silu":
                v, u = a * torch.sigmoid(a), b
            elif act == "gelu":
                v, u, ea, eb = torch.nn.functional.gelu(b), torch.ones_like(b), eb + 2.0 ** -23 * 3, torch.zeros_like(eb)
            else:
                a = a.clamp(max=1.5)
                v, u = a * torch.sigmoid(1.702 * a), b.clamp(-1.5, 1.5) + 1
            # slopes of the activations stay below 1.13; the rounding of the row to bf16 and 16 of fp32
            ev = 1.13 * ea * u.abs() + (v.abs() + 0.1) * eb + (2.0 ** -8 + 16 * 2.0 ** -24) * (v * u).abs()
            d = down[e].double()
            z, ez = d @ (v * u), d.abs() @ ev + (F + 8) * 2.0 ** -24 * (d.abs() @ (v * u).abs())
            want[t] += z if weighted else s * z
            lim[t] += ez if weighted else s * ez
    assert ((y.double() - want).abs() <= lim * (1 + 2.0 ** -16) + 1e-6).all()
