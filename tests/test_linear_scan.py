"""The linear matrix recurrences in their step and chunk forms against a float64 walk, at the edges of chunks, tiles and
batches; rows are columns of a wider projection, as in the model."""
import pytest
import torch

from llmss_amd import ops

# fp32 products and sums over at most 256 terms and 64-token chunks, exponentials good to a few ulp: 2^-24 times a few dozen
REL = 1e-5


def walk(q, k, v, g, e, S0, lens, starts):
    """q, k [T, H, dim], v [T, H, vdim], g, e [T, H] in float64 -> (o [T, H, vdim], final states)."""
    o, states, t = torch.zeros_like(v), [], 0
    for b, n in enumerate(lens):
        S = S0[b].clone() if starts[b] else torch.zeros_like(S0[b])
        for _ in range(n):
            S = g[t][:, None, None] * S + (e[t][:, None] * k[t])[:, :, None] * v[t][:, None, :]
            o[t] = (S * q[t][:, :, None]).sum(1)
            t += 1
        states.append(S)
    return o, states


def rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm().clamp(min=1e-30))


def run(mode, lens, starts, nd, heads, groups, dim, vdim, decay=None, dt_shift=0.0, dtype=torch.bfloat16):
    gen = torch.Generator().manual_seed(1000 * dim + 10 * vdim + len(lens))
    T, B = sum(lens), len(lens)
    nq, nv = groups * dim, heads * vdim
    width = (2 * nq + nv + heads + 15) // 8 * 8
    proj = torch.randn(T, width, generator=gen).to(dtype)
    q, k, v, dt = proj[:, :nq], proj[:, nq:2 * nq], proj[:, 2 * nq:2 * nq + nv], proj[:, 2 * nq + nv:2 * nq + nv + heads]
    S0 = torch.randn(B + 1, heads, dim, vdim, generator=gen)
    slots = torch.randperm(B, generator=gen).to(torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    ctx = torch.tensor([n + s for n, s in zip(lens, starts)], dtype=torch.int32)
    A_log, bias, D = (torch.randn(heads, generator=gen) for _ in range(3))
    bias = bias + dt_shift
    f = lambda t, n: t.double().view(T, -1, n).repeat_interleave(heads // (t.shape[1] // n), 1)  # noqa: E731
    Q, K, V = f(q, dim), f(k, dim), f(v, vdim)
    if mode == 0:
        Q, K, V = (x * torch.sigmoid(x) for x in (Q, K, V))
        g, e = decay.double().expand(T, heads), torch.ones(T, heads, dtype=torch.float64)
    else:
        e = torch.nn.functional.softplus(dt.double() + bias.double())
        g = torch.exp(-torch.exp(A_log.double()) * e)
    o, states = walk(Q, K, V, g, e, S0[slots.long()].double(), lens, starts)
    if mode == 2:
        o = o + D.double()[:, None] * V
    c = lambda t: t.cuda()  # noqa: E731
    P, S = c(proj), c(S0)
    q, k, v, dt = P[:, :nq], P[:, nq:2 * nq], P[:, 2 * nq:2 * nq + nv], P[:, 2 * nq + nv:2 * nq + nv + heads]
    form = dict(max_qlen=max(lens[nd:], default=1), num_decode=0 if max(lens) == 1 else nd)
    if mode == 0:
        y = ops.decay_recurrence(q, k, v, c(decay), S, c(cu), c(ctx), c(slots), heads, dim, vdim, True, **form)
    else:
        y = ops.ssd_recurrence(v, k, q, dt, c(A_log), c(bias), c(D), S, c(cu), c(ctx), c(slots), heads, groups, dim, vdim,
                               **form)
    assert rel(y.view(T, heads, vdim), o) < REL
    for b in range(B):
        assert rel(S[slots[b]], states[b]) < REL, b
    assert torch.equal(S[B].cpu(), S0[B])  # a slot nobody holds


LENS = [([1, 1, 7, 64, 65], [5, 0, 0, 0, 9], 2), ([63, 128, 8], [0, 70, 1], 0), ([200], [0], 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim", [(8, 5), (40, 24), (64, 64), (128, 128), (200, 72), (256, 130)])
@pytest.mark.parametrize("lens,starts,nd", LENS)
def test_decay(dim, vdim, lens, starts, nd):
    run(0, lens, starts, nd, 3, 3, dim, vdim, torch.tensor([0.5, 0.96875, 0.999]))


@pytest.mark.gpu
def test_decay_signs():
    """Factors of zero, below zero and above one."""
    run(0, [1, 70, 65], [3, 0, 4], 1, 4, 4, 64, 64, torch.tensor([0.0, -0.9, 1.01, 1.0]))


@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim,groups", [(8, 5, 1), (128, 64, 1), (16, 64, 2), (128, 64, 4), (256, 36, 2)])
@pytest.mark.parametrize("lens,starts,nd", LENS)
def test_ssd(dim, vdim, groups, lens, starts, nd):
    run(2, lens, starts, nd, 4, groups, dim, vdim)


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [-12.0, 6.0, 60.0])
def test_ssd_steps_from_nothing_to_forgetting(shift):
    run(2, [1, 130], [2, 3], 1, 4, 1, 64, 64, dt_shift=shift)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("dim,vdim", [(128, 64), (129, 128), (12, 4), (32, 6)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_single_rows(mode, dim, vdim, dtype):
    run(mode, [1] * 5, [0, 4, 1, 9, 0], 5, 4, 4, dim, vdim, torch.tensor([0.5, 0.9, 0.99, 1.0]), dtype=dtype)


@pytest.mark.gpu
def test_padded_rows_leave_states_alone():
    heads, dim, vdim = 2, 64, 64
    S0 = torch.randn(3, heads, dim, vdim, device="cuda")
    for n in (1, 40):
        x = torch.randn(2 * n, heads * dim, device="cuda").bfloat16()
        cu = torch.tensor([0, n, 2 * n], dtype=torch.int32, device="cuda")
        ctx = torch.tensor([n + 3, 0], dtype=torch.int32, device="cuda")
        slots = torch.tensor([1, -1], dtype=torch.int32, device="cuda")
        S = S0.clone()
        y = ops.decay_recurrence(x, x, x, torch.full((heads,), 0.9, device="cuda"), S, cu, ctx, slots, heads, dim, vdim, True,
                                 max_qlen=n)
        assert not y[n:].any() and torch.equal(S[0], S0[0]) and torch.equal(S[2], S0[2]) and not torch.equal(S[1], S0[1])


def test_step_form_takes_what_fits():
    """Key dimensions up to the walk's largest, so that its launch never asks for more LDS than a workgroup gets by default."""
    from llmss_amd.ops import hip
    L = hip.lib()
    for vdim in (4, 8, 64, 1024):
        for dim in (1, 8, 31, 32, 512, 513, 4096, 7700, 8192):
            if L.linear_step_ok(dim, vdim):
                assert dim <= 512 and 4 * (2 * dim + 4 + 256 // (vdim // 4) * vdim) <= 64 << 10
    assert L.linear_step_ok(512, 4) and L.linear_step_ok(128, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,nd", [([1, 0, 1], 0), ([0], 0), ([1, 1, 0, 70, 0], 2)])
@pytest.mark.parametrize("mode", [0, 2])
def test_empty_portions(mode, lens, nd):
    """A sequence without rows changes nothing, its own state among it."""
    heads, dim, vdim, B, T = 2, 64, 64, len(lens), sum(lens)
    S0 = torch.randn(B, heads, dim, vdim, device="cuda")
    x = torch.randn(T, heads * dim, device="cuda").bfloat16()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    w = [torch.full((heads,), 0.5, device="cuda") for _ in range(3)]

    def step(lens, slots, S, **form):
        cu, ctx = i32([0] + lens).cumsum(0).to(torch.int32), i32([n + 3 for n in lens])
        if mode == 0:
            return ops.decay_recurrence(x, x, x, w[0], S, cu, ctx, i32(slots), heads, dim, vdim, True, **form)
        return ops.ssd_recurrence(x, x, x, x[:, :heads], *w, S, cu, ctx, i32(slots), heads, heads, dim, vdim, **form)
    S = S0.clone()
    y = step(lens, list(range(B)), S, max_qlen=max(1, max(lens)), num_decode=nd)
    kept = [b for b in range(B) if lens[b]]
    S1 = S0.clone()
    want = step([lens[b] for b in kept], kept, S1) if kept else x[:, :0].float()
    assert y.shape[0] == T and (not T or rel(y, want.double().cpu()) < REL)
    for b in range(B):
        assert torch.equal(S[b], S0[b]) if not lens[b] else rel(S[b], S1[b].double().cpu()) < REL
