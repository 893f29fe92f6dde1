"""Grouped expert products of a few rows per expert (csrc/moe_dec.hip) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# K of one step up to more than a wave's eight, F that is no multiple of 128; one row, an expert with more rows than a tile, one with none; in
# whole lines, steps that do not divide evenly among a wave's four; without and with a tile list (so does a layer of many experts by itself)
@pytest.mark.parametrize("E,top,W,F,T", [(4, 2, 32, 32, 1), (8, 2, 96, 160, 15), (5, 3, 1056, 96, 13), (40, 1, 2048, 768, 21), (16, 2, 1088, 704, 33),
                                         (12, 2, 2304, 320, 9), (160, 8, 64, 64, 150), (1024, 8, 64, 64, 2), (200, 3, 96, 64, 64), (256, 1, 64, 32, 255)])
@pytest.mark.parametrize("kind", ["silu", "weighted", "clamp", "interleaved", "gelu"])
@pytest.mark.parametrize("grouped", [False, True])
def test_moe_dec(E, top, W, F, T, kind, grouped, monkeypatch):
    from llmss_amd.ops import hip, glu_interleave
    monkeypatch.setattr(hip, "_moe_own_rows", lambda *a: not grouped)
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
    assert calls.count("moe_dec") == 2 and calls.count("moe_group") == (1 if grouped or T * top > 1024 else 0)
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


# One look at the choices instead of a grouping launch, the shared expert in the same launches: experts of no, one, 16, 17, 32, 33 and all
# rows (tiles past an expert's first), the largest number of pairs, a shared expert of another width, further columns behind it; both launches in
# whole lines, several looks of a wave with a partial last one, up to 16 rows and more
@pytest.mark.parametrize("E,top,W,F,Fs,D,T", [(4, 1, 64, 32, 64, 24, 1), (9, 3, 96, 96, 32, 0, 16), (8, 1, 160, 64, 96, 40, 33),
                                              (16, 2, 256, 96, 160, 256, 64), (128, 16, 64, 32, 32, 7, 64),
                                              (16, 2, 2048, 768, 1024, 40, 8), (16, 2, 1088, 1344, 1088, 24, 33), (8, 1, 2304, 1344, 320, 8, 40)])
@pytest.mark.parametrize("kind", ["silu", "weighted", "clamp", "interleaved"])
def test_moe_dec_own_rows(E, top, W, F, Fs, D, T, kind, monkeypatch):
    from llmss_amd.ops import glu_interleave, hip
    from llmss_amd.ops import reference as ref
    g = torch.Generator().manual_seed(E + T)
    inter, weighted = kind == "interleaved", kind == "weighted"
    D = 0 if inter else D
    rnd = lambda *s: (torch.randn(*s, generator=g) * s[-1] ** -0.5).bfloat16().cuda()  # noqa: E731
    h = torch.randn(T, W + 8, generator=g).bfloat16().cuda()[:, :W]
    gate, up, down, sg, su, sd, more = rnd(E, F, W), rnd(E, F, W), rnd(E, W, F), rnd(Fs, W), rnd(Fs, W), rnd(W, Fs), rnd(max(D, 1), W)[:D]
    idx = torch.stack([torch.randperm(E - 1, generator=g)[:top] for _ in range(T)]).int()
    idx[:, 0] = torch.where((idx[:, 1:] == 0).any(1), idx[:, 0], 0)  # most rows choose expert 0, nobody the last one
    if top == 1:
        idx[T // 2:, 0] = 1  # (17 rows and 16 of 33)
    w, sw = torch.rand(T, top, generator=g).cuda(), torch.rand(T, generator=g).cuda()
    act = "glu_clamp" if kind == "clamp" else "silu"
    lib, calls = hip.lib(), []

    class Seen:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)
    monkeypatch.setattr(hip, "lib", Seen)
    sgu = glu_interleave(sg, su) if inter else torch.cat([sg, su, more])
    y, gu = hip.moe_experts(h, idx.cuda(), w, None if inter else gate, glu_interleave(gate, up, 1).contiguous() if inter else up, down, 1.5,
                            1.702, act=act, weight_input=weighted, shared_w=sw, interleaved=inter,
                            shared_mlp=(sgu.contiguous(), sd, Fs, inter, 0.7))
    assert calls.count("moe_dec") == 2 and calls.count("moe_group") == 0 and calls.count("gemm") == 0
    x = h.double()

    def glu(a, b, limit):
        if act == "silu":
            return a * torch.sigmoid(a) * b
        a = a.clamp(max=limit)
        return a * torch.sigmoid(1.702 * a) * (b.clamp(-limit, limit) + 1)
    want = sw.double()[:, None] * (glu(x @ sg.double().T, x @ su.double().T, 0.7) @ sd.double().T)
    for t in range(T):
        for j in range(top):
            e, s = int(idx[t, j]), w[t, j].double()
            a, b = gate[e].double() @ x[t], up[e].double() @ x[t]
            v = down[e].double() @ (glu(s * a, s * b, 1.5) if weighted else glu(a, b, 1.5))
            want[t] += v if weighted else s * v
    # roundings to bf16: gate, up and activations, then the shared expert's rows - half a unit in the last place each, sums in fp32
    assert ((y.double() - want).norm() / want.norm()).item() < 2.0 ** -7.5
    if D:
        z = x @ more.double().T
        assert ((gu[:, 2 * Fs:].double() - z).abs() <= 2.0 ** -8 * z.abs() + (W + 8) * 2.0 ** -24 * (x.abs() @ more.double().abs().T)).all()
    else:
        assert gu is None
    assert ref.moe_experts(h.cpu(), idx, w.cpu(), *(t.cpu() for t in (gate, up, down)), 1.5, 1.702, act=act, weight_input=weighted,
                           shared_w=sw.cpu(), shared_mlp=(torch.cat([sg, su, more]).cpu(), sd.cpu(), Fs, False, 0.7))[0].sub(
        y.cpu()).norm() / want.norm().cpu() < 2.0 ** -7
