"""The row kernels of csrc/streams.hip that move four to eight numbers an access, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# widths: one access, edges of 1024, 2048 and 4096, beyond; more streams than the kernel takes; outputs in both types
@pytest.mark.parametrize("S,T,W", [(1, 3, 4), (2, 5, 1020), (2, 1, 1024), (3, 7, 1028), (4, 2, 2048), (2, 3, 2052), (1, 2, 4096),
                                   (2, 2, 4100), (5, 2, 256), (2, 3, 1022), (2, 5, 256), (4, 3, 260), (1, 2, 508), (3, 2, 768)])
@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
def test_stream_add_norm(S, T, W, rms, dtype, out):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(S * W + T)
    x0 = torch.randn(S, T, W, generator=g).cuda()
    y = torch.randn(T, W + 4, generator=g).to(dtype).cuda()[:, :W]
    w = (1 + 0.1 * torch.randn(W, generator=g)).to(dtype).cuda()
    mix = (torch.eye(S) + 0.3 * torch.randn(S, S, generator=g)).cuda()
    outw, inw = torch.randn(S, generator=g).cuda(), torch.randn(S, generator=g).cuda()
    x = x0.clone()
    h = hip.stream_add_norm(x, y, mix, outw, 0.7, inw, w, 1e-5, rms, out)
    nx = torch.einsum("st,snw->tnw", mix.double(), x0.double()) + 0.7 * outw.double()[:, None, None] * y.double()
    # S + 2 fp32 roundings of terms no larger than their absolute sum
    big = torch.einsum("st,snw->tnw", mix.double().abs(), x0.double().abs()) + 0.7 * outw.double().abs()[:, None, None] * y.double().abs()
    eu = (S + 3) * 2.0 ** -24
    assert ((x.double() - nx).abs() <= eu * big).all()
    u = torch.einsum("s,snw->nw", inw.double(), x.double())
    ub = torch.einsum("s,snw->nw", inw.double().abs(), x.double().abs())
    d = u if rms else u - u.mean(-1, keepdim=True)
    inv = 1 / torch.sqrt(d.pow(2).mean(-1, keepdim=True) + 1e-5)
    want = d * inv * w.double()
    # u's own error, the mean's (sums of W / 256 + 12 steps), and 16 relative roundings of the norm
    e = (eu * (ub + ub.mean(-1, keepdim=True)) + 32 * 2.0 ** -24 * ub.mean(-1, keepdim=True)) * inv * w.double().abs() \
        + 32 * 2.0 ** -24 * want.abs()
    if out == torch.bfloat16:
        e = e + 2.0 ** -8 * want.abs()
    assert ((h.double() - want).abs() <= e).all()


@pytest.mark.parametrize("T,F", [(1, 8), (3, 2040), (2, 2048), (5, 2056), (2, 5632), (3, 100), (2, 7),
                                 (4096, 256), (4097, 264), (514, 2040), (512, 2048), (511, 2056), (187, 5632), (8192, 200)])
@pytest.mark.parametrize("act", ["gelu_tanh", "silu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_glu_act(T, F, act, dtype):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(F)
    gu = torch.randn(T, 2 * F, generator=g) * 4
    gu[0, 0], gu[0, F - 1] = -40.0, 40.0
    gu = gu.to(dtype).cuda()
    got = hip.glu_act(gu, F, act).double()
    a, u = gu[:, :F].double(), gu[:, F:].double()
    z = 2 * 0.7978845608028654 * (a + 0.044715 * a ** 3) if act == "gelu_tanh" else a
    want = a * torch.sigmoid(z) * u
    # 8 roundings, the exponent's argument to 4 of its own units; bf16 results one rounding; below the smallest normal anything;
    # two units of the product where the tanh form is taken, for 1 + tanh near -1
    lim = (8 + 4 * z.abs()) * 2.0 ** -24 * want.abs() + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0) + 2 * 2.0 ** -24 * (a * u).abs() * (act == "gelu_tanh") + 1e-36
    assert ((got - want).abs() <= lim).all()


# groups on both sides of 512 and 4096 and at the edges of 1024 and 2048; the gate before the norm and after
@pytest.mark.parametrize("T,groups,n", [(3, 2, 516), (2, 1, 1024), (1, 3, 1028), (2, 1, 2048), (3, 1, 2052), (2, 2, 4096), (2, 1, 4100),
                                        (2, 1, 770)])
@pytest.mark.parametrize("act,first", [("silu", True), ("silu", False), ("sigmoid", False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_gated_group_norm(T, groups, n, act, first, dtype):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(n + T)
    o = torch.randn(T, groups * n, generator=g).cuda() * 3
    gate = torch.randn(T, groups * n + 4, generator=g).to(dtype).cuda()[:, 4:]
    w = (1 + 0.1 * torch.randn(groups * n, generator=g)).to(dtype).cuda()
    got = hip.gated_group_norm(o, gate, w, 1e-5, act, 0.9, out_dtype=dtype, groups=groups, gate_first=first).double()
    z = gate.double()
    a = torch.sigmoid(z) * (z if act == "silu" else 1)
    u = (o.double() * a if first else o.double()).view(T, groups, n)
    want = (0.9 * u / torch.sqrt(u.pow(2).mean(-1, keepdim=True) + 1e-5)).view(T, -1) * w.double() * (1 if first else a)
    # the gate's exponential and quotient (8 + |z| units), the norm (sum of squares in any order: n / 2 units at most of ss, in practice
    # steps of 16 and a tree of 8), 8 products; bf16 results one rounding
    lim = (32 + 2 * z.abs()) * 2.0 ** -24 * want.abs() + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0) + 1e-30
    assert ((got - want).abs() <= lim).all()
