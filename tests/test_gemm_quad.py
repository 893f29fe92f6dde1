"""The 256 x 256 prompt GEMM of four waves (csrc/gemm_quad.hip) against a float64 product."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def bound(x, w, y64, slope=1.0):
    # fp32 accumulation in any order: (K + 2) 2^-24 of the products' absolute sum; one rounding to bf16: 2^-8 of the result.
    # Two further units of fp32 for bias, activation and gating.
    s = x.double().abs() @ w.double().abs().t()
    return slope * (x.shape[1] + 4) * 2.0 ** -24 * s + 2.0 ** -8 * y64.abs() + 1e-6


# K: one step, fewer steps than the ring holds, an odd number, many; M and N: one row, edges of tiles and their neighbours
@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (255, 264, 128), (256, 256, 192), (257, 8, 320), (300, 504, 448), (513, 1000, 1088),
                                   (700, 768, 4096)])
@pytest.mark.parametrize("act,bias", [("none", False), ("none", True), ("gelu", True), ("relu", False)])
def test_plain(M, N, K, act, bias):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g).bfloat16().cuda()[:, :K]
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if bias else None
    y = hip.linear(x, w, b, act, False, nt_hint=4 << 8, split_hint=1)
    ref = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    if act == "gelu":
        ref = torch.nn.functional.gelu(ref)
    if act == "relu":
        ref = ref.relu()
    # (gelu's slope stays below 1.13; erff is good to 4 units of its own last place, times |x| / 2 <= 3 where it matters)
    lim = bound(x, w, ref, 1.13) + (6 * 2.0 ** -23 * 3 if act == "gelu" else 0.0)
    assert ((y.double() - ref).abs() <= lim).all()


@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (255, 288, 128), (513, 544, 1088)])
@pytest.mark.parametrize("bias", [False, True])
def test_glu(M, N, K, bias):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if bias else None
    y = hip.linear(x, w, b, "none", True, nt_hint=4 << 8, split_hint=1)
    z = (x.double() @ w.double().t() + (b.double() if bias else 0.0)).view(M, N // 32, 2, 16)
    ga, up = z[:, :, 0].reshape(M, N // 2), z[:, :, 1].reshape(M, N // 2)
    ref = torch.nn.functional.silu(ga) * up
    e = ((K + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -24 * z.reshape(M, N).abs()).view(M, N // 32, 2, 16)
    eg, eu = e[:, :, 0].reshape(M, N // 2), e[:, :, 1].reshape(M, N // 2)
    # silu's slope stays below 1.1; __expf and the quotient: 8 units of fp32 and |gate| units of the exponent
    lim = 1.1 * eg * up.abs() + (ga.abs() + 1) * eu + (8 + 2 * ga.abs()) * 2.0 ** -23 * ref.abs() + 2.0 ** -8 * ref.abs() + 1e-6
    assert ((y.double() - ref).abs() <= lim).all()


# P / E >= the bound of the 256-row tiles; widths with remainders of the tile's 256 columns, one expert nobody chooses, steps of 64 and 192
@pytest.mark.parametrize("E,top,W,F,T", [(3, 2, 256, 320, 900), (2, 1, 320, 272, 1100), (4, 2, 320, 256, 1000)])
@pytest.mark.parametrize("act,weighted", [("silu", True), ("silu", False), ("glu_clamp", False)])
def test_experts_two_matrices(E, top, W, F, T, act, weighted, monkeypatch):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(E + W + F)
    h = torch.randn(T, W + 8, generator=g).bfloat16().cuda()[:, :W]
    gate, up = ((torch.randn(E, F, W, generator=g) * W ** -0.5).bfloat16().cuda() for _ in range(2))
    down = (torch.randn(E, W, F, generator=g) * F ** -0.5).bfloat16().cuda()
    idx = torch.stack([torch.randperm(E - 1 if top < E - 1 else E, generator=g)[:top] for _ in range(T)]).int().cuda()
    w = torch.rand(T, top, generator=g).cuda()
    lib, calls = hip.lib(), []

    class Seen:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)
    monkeypatch.setattr(hip, "lib", Seen)
    y = hip.moe_experts(h, idx, w, gate, up, down, 1.5, 1.702, act=act, weight_input=weighted)
    assert "moe_pp_glu" in calls
    want = torch.zeros(T, W, dtype=torch.float64, device="cuda")
    lim = torch.zeros_like(want)
    hd = h.double()
    for e in range(E):
        for j in range(top):
            r = (idx[:, j] == e).nonzero()[:, 0]
            if not len(r):
                continue
            s = w[r, j].double()[:, None]
            a, b = (hd[r] @ m[e].double().t() for m in (gate, up))
            ea, eb = ((W + 4) * 2.0 ** -24 * (hd[r].abs() @ m[e].double().abs().t()) for m in (gate, up))
            if weighted:
                a, b, ea, eb = a * s, b * s, ea * s, eb * s
            if act == "silu":
                v, u = a * torch.sigmoid(a), b
            else:
                a = a.clamp(max=1.5)
                v, u = a * torch.sigmoid(1.702 * a), b.clamp(-1.5, 1.5) + 1
            # slopes of the activations stay below 1.1; the rounding of the row to bf16 and 16 of fp32
            ev = 1.1 * ea * u.abs() + (v.abs() + 0.1) * eb + (2.0 ** -8 + 16 * 2.0 ** -24) * (v * u).abs()
            d = down[e].double()
            z, ez = (v * u) @ d.t(), ev @ d.abs().t() + (F + 4) * 2.0 ** -24 * ((v * u).abs() @ d.abs().t())
            want[r] += z if weighted else s * z
            lim[r] += ez if weighted else s * ez
    assert ((y.double() - want).abs() <= lim * (1 + 2.0 ** -20) + 1e-6).all()
