"""Infinities and NaN in portions that the recurrences take chunk by chunk: what a token-by-token walk in float64 leaves finite stays
finite, with its value - the tokens before such a number, other columns, other heads, other sequences -, and what it does not, does not."""
import pytest
import torch

from llmss_amd import ops

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")
LENS = [130, 20]


def same(got, want, tol):
    got = got.double().cpu()
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    a, b = (x.where(torch.isfinite(want), torch.zeros((), dtype=torch.float64)) for x in (got, want))
    assert ((a - b).norm() / b.norm()).item() < tol


def prefix(lens):
    return torch.tensor([0] + lens).cumsum(0).to(torch.int32)


@pytest.mark.parametrize("dim,vdim", [(64, 40), (128, 64)])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("t", [3, 47, 79, 129, 133])  # inside blocks of 16, a chunk's and a portion's edges, the second sequence
@pytest.mark.parametrize("place,value", [("v", NAN), ("v", INF), ("v", -INF), ("k", NAN), ("k", INF), ("q", NAN), ("q", INF), ("dt", NAN),
                                         ("dt", INF), ("dt", -INF), ("S", INF)])
def test_linear(mode, dim, vdim, t, place, value):
    heads = 2
    gen = torch.Generator().manual_seed(t)
    T, B = sum(LENS), len(LENS)
    q, k, v = (torch.randn(T, heads, n, generator=gen).bfloat16() for n in (dim, dim, vdim))
    dt, S0 = torch.randn(T, heads, generator=gen).bfloat16(), torch.randn(B, heads, dim, vdim, generator=gen)
    {"v": v, "k": k, "q": q, "dt": dt.view(T, heads, 1), "S": S0[0]}[place][t if place != "S" else 0, 1, -1] = value
    if place == "S":
        S0[0, 0, 2, 5] = value
    decay, A_log, bias, D = torch.tensor([0.5, 0.97]), *(torch.randn(heads, generator=gen) for _ in range(3))
    Q, K, V = q.double(), k.double(), v.double()
    if mode == 0:
        Q, K, V = (x / (1 + torch.exp(-x)) for x in (Q, K, V))
        g, e = decay.double().expand(T, heads), torch.ones(T, heads, dtype=torch.float64)
    else:
        e = torch.nn.functional.softplus(dt.double() + bias.double())
        g = torch.exp(-torch.exp(A_log.double()) * e)
    o, states, r = torch.zeros_like(V), [], 0
    for b, n in enumerate(LENS):
        S = S0[b].double()
        for _ in range(n):
            S = g[r][:, None, None] * S + (e[r][:, None] * K[r])[:, :, None] * V[r][:, None, :]
            o[r] = (S * Q[r][:, :, None]).sum(1)
            r += 1
        states.append(S)
    if mode == 2:
        o = o + D.double()[:, None] * V
    c = lambda x: x.cuda()  # noqa: E731
    S, cu = c(S0), prefix(LENS)
    form = (S, c(cu), c(cu.diff() + 7), torch.arange(B, dtype=torch.int32, device="cuda"), heads)
    rows = [c(x).flatten(1) for x in (q, k, v)]
    if mode == 0:
        y = ops.decay_recurrence(*rows, c(decay), *form, dim, vdim, True, max_qlen=max(LENS))
    else:
        y = ops.ssd_recurrence(rows[2], rows[1], rows[0], c(dt), c(A_log), c(bias), c(D), *form, heads, dim, vdim, max_qlen=max(LENS))
    same(y.view(T, heads, vdim), o, 1e-5)  # the bound of the finite cases: fp32 sums over at most 256 terms and 64 tokens
    for b in range(B):
        same(S[b], states[b], 1e-5)


@pytest.mark.parametrize("dim,vdim", [(32, 36), (128, 64)])
@pytest.mark.parametrize("t", [3, 16, 47, 79, 129, 133])
@pytest.mark.parametrize("place,value", [("v", NAN), ("v", INF), ("k", NAN), ("k", INF), ("q", NAN), ("q", -INF), ("a", NAN), ("a", INF),
                                         ("a", -INF), ("b", NAN), ("b", INF), ("b", -INF), ("S", INF)])
def test_delta_rows32(dim, vdim, t, place, value):
    heads = 2
    gen = torch.Generator().manual_seed(t)
    T, B = sum(LENS), len(LENS)
    q, k, v = (torch.randn(T, heads, n, generator=gen) for n in (dim, dim, vdim))
    a, b_, S0 = torch.randn(T, heads, generator=gen), torch.randn(T, heads, generator=gen), torch.randn(B, heads, dim, vdim, generator=gen)
    if place == "S":
        S0[0, 0, 2, 5] = value
    else:
        {"v": v, "k": k, "q": q, "a": a.view(T, heads, 1), "b": b_.view(T, heads, 1)}[place][t, 1, -1] = value
    gate, w = torch.randn(T, heads * vdim, generator=gen), 1 + 0.1 * torch.randn(vdim, generator=gen)
    A_log, bias = torch.randn(heads, generator=gen) - 1, torch.randn(heads, generator=gen)
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    Q, K, V = unit(q.double()) * dim ** -0.5, unit(k.double()), v.double()
    g = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(a.double() + bias.double()))
    beta = torch.sigmoid(b_.double())
    o, states, r = torch.zeros_like(V), [], 0
    for b, n in enumerate(LENS):
        S = S0[b].double()
        for _ in range(n):
            S = S * g[r, :, None, None]
            u = beta[r, :, None] * (V[r] - (S * K[r, :, :, None]).sum(1))
            S = S + K[r, :, :, None] * u[:, None]
            o[r] = (S * Q[r, :, :, None]).sum(1)
            r += 1
        states.append(S)
    z = gate.double().view(T, heads, vdim)
    want = 0.7 * o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6) * w.double() * z * torch.sigmoid(z)
    c = lambda x: x.cuda()  # noqa: E731
    S, cu, out = c(S0), prefix(LENS), torch.empty(T, heads * vdim, device="cuda")
    rows = [c(x).flatten(1) for x in (q, k, v)]
    ab = c(torch.cat([a, b_], 1))
    ops.delta_mix(*rows, ab[:, :heads], ab[:, heads:], c(A_log), c(bias), S, c(cu), c(cu.diff() + 7), torch.arange(B, dtype=torch.int32, device="cuda"),
                  heads, heads, dim, vdim, c(gate), c(w), 1e-6, 0.7, out, max_qlen=max(LENS), num_decode=0)
    # the bound of the finite cases: fp32 sums over up to 128 terms, then substitution over 64 tokens
    same(out.view(T, heads, vdim), want, 2e-5)
    for b in range(B):
        same(S[b], states[b], 2e-5)
