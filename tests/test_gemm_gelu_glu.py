"""Gated products with the tanh form of GELU (act "gelu_tanh", glu): every plan's epilogue against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows of the streaming, decode, one and several row tiles; columns and K with remainders of every tile
@pytest.mark.parametrize("M,N,K", [(1, 96, 64), (16, 544, 272), (33, 160, 1088), (64, 544, 272), (100, 288, 576), (513, 544, 1088)])
@pytest.mark.parametrize("bias", [False, True])
def test_gelu_gates_of_every_plan(M, N, K, bias):
    from llmss_amd.ops import hip
    from llmss_amd.ops.autotune import candidates
    g = torch.Generator().manual_seed(M + N + K)
    x = (2 * torch.randn(M, K, generator=g)).bfloat16().cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if bias else None
    z = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    parts = lambda t: [t.view(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1)]
    ga, up = parts(z)
    gate = torch.nn.functional.gelu(ga, approximate="tanh")
    ref = gate * up
    eg, eu = parts((K + 4) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2.0 ** -24 * z.abs())
    # The gate's slope stays below 1.13. exp's argument 1.6 (g + 0.045 g^3) is good to 4 units of its size, which it passes on to gates
    # below 0 (there the gate itself falls faster); 8 units for __expf and the quotient.
    arg = 1.6 * (ga.abs() + 0.045 * ga.abs() ** 3)
    lim = 1.13 * eg * up.abs() + (gate.abs() + 0.2) * eu + (8 + 4 * arg) * 2.0 ** -23 * ref.abs() + 2.0 ** -8 * ref.abs() + 1e-6
    plans = [(0, 0)] + candidates(M, N, K, True, False) + [(4 << 8, 1)] * (K % 64 == 0)
    done = 0
    for nt, split in plans:
        try:
            y = hip.linear(x, w, b, "gelu_tanh", True, nt_hint=nt, split_hint=split)
        except RuntimeError as e:  # (tiles whose waves hold no whole gate and up are refused on the host, as for SiLU)
            assert "SwiGLU" in str(e)
            continue
        done += 1
        assert ((y.double() - ref).abs() <= lim).all(), (nt, split)
    assert done > 8
