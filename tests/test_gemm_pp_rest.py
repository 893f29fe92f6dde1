"""The 256 x 256 ping-pong GEMM (csrc/gemm.hip) at what it is left with: K off 64, widths off 8, rows spread over more than 31 bits of
bytes, plain and as grouped expert products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def spread(x, ld):
    y = torch.empty((x.shape[0] - 1) * ld + x.shape[1], dtype=x.dtype, device=x.device).as_strided(x.shape, (ld, 1))
    return y.copy_(x)


@pytest.mark.parametrize("M,N,K,ldx", [(300, 264, 144, 0), (257, 256, 560, 0), (300, 268, 128, 0), (513, 12, 64, 0), (260, 264, 192, 1 << 22)])
def test_plain(M, N, K, ldx):
    from llmss_amd.ops import hip
    x = torch.randn(M, K, device="cuda").bfloat16()
    if ldx:
        x = spread(x, ldx)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    out = torch.full((M, (N // 8 + 2) * 8), 7.0, device="cuda").bfloat16()
    ref = x.double() @ w.double().t()
    hip.linear(x, w, out=out[:, :N], nt_hint=4 << 8, split_hint=1)
    # fp32 sums of K products, one rounding to bf16
    lim = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * ref.abs()
    assert ((out[:, :N].double() - ref).abs() <= lim).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("W,F,N,ldh", [(264, 264, 256, 0), (256, 256, 260, 0), (256, 256, 256, 1 << 22)])
@pytest.mark.parametrize("kind", ["gelu", "interleaved"])
def test_experts(W, F, N, ldh, kind, monkeypatch):
    from llmss_amd.ops import glu_interleave, hip
    if kind == "interleaved" and F % 16:
        F = 272
    E, top, T = 2, 1, 300
    g = torch.Generator().manual_seed(W + N)
    h = torch.randn(T, W, generator=g).bfloat16().cuda()
    gate, up = ((torch.randn(E, F, W, generator=g) * W ** -0.5).bfloat16().cuda() for _ in range(2))
    down = (torch.randn(E, N, F, generator=g) * F ** -0.5).bfloat16().cuda()
    idx, w = torch.randint(0, E, (T, top), generator=g).int().cuda(), torch.rand(T, top, generator=g).cuda()
    lib, calls = hip.lib(), []

    class Seen:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)
    monkeypatch.setattr(hip, "lib", Seen)
    rows = spread(h, ldh) if ldh else h
    if kind == "gelu":
        y = hip.moe_experts(rows, idx, w, None, up, down, 0.0, 0.0, act="gelu")
    else:
        y = hip.moe_experts(rows, idx, w, None, glu_interleave(gate, up, 1).contiguous(), down, 0.0, 0.0, act="silu", interleaved=True)
    assert calls.count("moe_pp") == 2
    for e in range(E):
        r = (idx[:, 0] == e).nonzero()[:, 0]
        x, s = h[r].double(), w[r].double()
        a, b = (x @ m[e].double().t() for m in (gate, up))
        v = torch.nn.functional.gelu(b) if kind == "gelu" else torch.nn.functional.silu(a) * b
        want = s * (v @ down[e].double().t())
        # the activations rounded to bf16 once (2^-9 of each, of random sign over F of them), sums in fp32
        assert ((y[r].double() - want).norm() / want.norm()).item() < 4e-3
