"""The gates of 256 x 256 products (csrc/gemm_quad.h gate_by) off the range of ordinary numbers: infinities, NaN, zeros, and where the exponential
over- and underflows, dense and in experts' first products."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")
GATES = [0.0, -0.0, 1e-30, -1e-30, 0.5, -0.5, 1.0, -1.0, 20.0, -20.0, 80.0, -80.0, 87.0, -87.0, 87.5, -87.5, 88.0, -88.0, 88.5, -88.5, 89.0, -89.0,
         104.0, -104.0, 1e4, -1e4, 1e15, -1e15, 3e38, -3e38, INF, -INF, NAN]


def check(got, g, u, gate):
    """``got`` (bf16) against ``gate(g) * u`` as 32-bit arithmetic has it: the same infinities and NaN, else the 64-bit value rounded to bf16
    (the sign of a zero may be either). Where 1 + exp() is beyond 2^126 (negative gates of 87.3 and more) a gate, under 1e-36 then, may be zero: 0 u for it."""
    want, exact = gate(g) * u, gate(g.double()) * u.double()
    tiny = gate(g.double()).abs() < 1.2e-36
    slack = 1.2e-36 * u.double().abs()
    same = torch.where(want.isnan(), got.isnan(), torch.where(want.isinf(), got == want, (got.double() - exact).abs() <= slack + 2.0 ** -8 * exact.abs() + 1e-38))
    # (a gate of zero times an infinite factor is no number, and of under 1e-36 times a large one within the slack)
    same |= tiny & (u.isinf() & got.isnan() | ((got.double() - exact).abs() <= slack))
    # (products around the largest number of bf16 and of fp32 round to infinity or not)
    same |= (exact.abs() > 3.3e38) & (got.abs() > 3.3e38) & (got.sign() == exact.sign())
    assert same.all(), [(float(a), float(b), float(c), float(d)) for a, b, c, d in zip(g[~same], u[~same], got[~same], want[~same])][:9]


@pytest.mark.parametrize("act", ["none", "gelu_tanh"])
@pytest.mark.parametrize("M", [1, 300])
def test_dense(act, M):
    """Products of zero and a bias that carries the values; groups of 16 gates and their ups."""
    from llmss_amd.ops import hip

    pairs = list(itertools.product(GATES, [1.0, -2.0, 0.0, 1e-20, 1e30, INF, NAN]))
    pairs += [(0.0, 0.0)] * (-len(pairs) % 16)
    g, u = (torch.tensor(v).bfloat16() for v in zip(*pairs))
    b = torch.stack([g.view(-1, 16), u.view(-1, 16)], 1).reshape(-1).cuda()
    x, w = torch.zeros(M, 64, dtype=torch.bfloat16, device="cuda"), torch.zeros(b.numel(), 64, dtype=torch.bfloat16, device="cuda")
    y = hip.linear(x, w, b, act, True, nt_hint=4 << 8, split_hint=1).float().cpu()
    z = (lambda t: 1.5957691216057308 * (t + 0.044715 * t * t * t)) if act == "gelu_tanh" else (lambda t: t)
    for row in (y[0], y[-1]):
        check(row, g.float(), u.float(), lambda t: t / (1 + torch.exp(-z(t))))


@pytest.mark.parametrize("form", ["silu", "clamped"])
def test_experts(form):
    """Gates and ups of 1 and of a number each, scaled by the pairs' weights."""
    from llmss_amd.ops import hip

    L, F, K = hip.lib(), 256, 64
    s = torch.tensor(GATES)
    P, E = s.numel(), 1
    gv, uv = torch.ones(F), torch.tensor([1.0, -2.0, 0.25, 3.0]).repeat(F // 4)
    gv[128:] = -1.0
    h, gate, up = torch.zeros(P, K), torch.zeros(E, F, K), torch.zeros(E, F, K)
    h[:, 3], gate[0, :, 3], up[0, :, 3] = 1.0, gv, uv
    h, gate, up = (t.bfloat16().cuda() for t in (h, gate, up))
    idx, maxt = torch.zeros(P, 1, dtype=torch.int32, device="cuda"), -(-P // 256) + 1
    meta = torch.zeros(3 + E + 2 * maxt, dtype=torch.int32, device="cuda")
    order, place = (torch.empty(P, dtype=torch.int32, device="cuda") for _ in range(2))
    act, st = torch.empty(P, F, dtype=torch.bfloat16, device="cuda"), torch.cuda.current_stream().cuda_stream
    pw = s.cuda()
    assert L.moe_pp_glu_ok(K, maxt, 1, F, K)
    L.moe_group_tall(idx.data_ptr(), P, E, maxt, meta.data_ptr(), order.data_ptr(), place.data_ptr(), 256, 1, st)
    limit, alpha = 7.0, 1.702
    L.moe_pp_glu(h.data_ptr(), K, gate.data_ptr(), up.data_ptr(), meta.data_ptr(), order.data_ptr(), act.data_ptr(), E, maxt, 1, F, K, limit, alpha,
                 pw.data_ptr(), int(form == "silu"), st)
    got = act.float().cpu()[place.cpu().long()]
    g, u = s[:, None] * gv, s[:, None] * uv  # (NaN: the minimum with the limit is the limit, the maximum with its negative that)
    if form == "clamped":
        lim = torch.tensor(limit)
        g, u = torch.fmin(g, lim), torch.fmin(torch.fmax(u, -lim), lim) + 1
        check(got.reshape(-1), g.reshape(-1), u.reshape(-1), lambda t: t / (1 + torch.exp(-alpha * t)))
    else:
        check(got.reshape(-1), g.reshape(-1), u.reshape(-1), lambda t: t / (1 + torch.exp(-t)))
