"""The gated delta rule over fp32 rows, single rows and portions, against a float64 walk at the edges of chunks and tiles."""
import pytest
import torch

from llmss_amd import ops


def run(lens, starts, nd, heads, kv, dim, vdim, dtype, shift=0.0, same_key=False):
    gen = torch.Generator().manual_seed(7 * dim + vdim + len(lens))
    T, B, nq, nv = sum(lens), len(lens), kv * dim, heads * vdim
    qkv = torch.randn(T, 2 * nq + nv + 4, generator=gen)
    if same_key:
        qkv[:, nq:2 * nq] = qkv[:1, nq:2 * nq]
    ab = torch.randn(T, 2 * heads, generator=gen).to(dtype)
    gate, w = torch.randn(T, nv, generator=gen).to(dtype), (1 + 0.1 * torch.randn(vdim, generator=gen)).to(dtype)
    A_log, bias = torch.randn(heads, generator=gen) - 1, torch.randn(heads, generator=gen) + shift
    S0 = torch.randn(B + 1, heads, dim, vdim, generator=gen)
    slots = torch.randperm(B, generator=gen).to(torch.int32)
    cu, ctx = torch.tensor([0] + lens).cumsum(0).to(torch.int32), torch.tensor([n + s for n, s in zip(lens, starts)]).int()
    rep = heads // kv
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = unit(qkv[:, :nq].double().view(T, kv, dim)).repeat_interleave(rep, 1) * dim ** -0.5
    k = unit(qkv[:, nq:2 * nq].double().view(T, kv, dim)).repeat_interleave(rep, 1)
    v = qkv[:, 2 * nq:2 * nq + nv].double().view(T, heads, vdim)
    g = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(ab[:, :heads].double() + bias.double()))
    beta = torch.sigmoid(ab[:, heads:].double())
    o, states, t = torch.zeros(T, heads, vdim, dtype=torch.float64), [], 0
    for b, n in enumerate(lens):
        S = S0[slots[b]].double() if starts[b] else torch.zeros(heads, dim, vdim, dtype=torch.float64)
        for _ in range(n):
            S = S * g[t, :, None, None]
            u = beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
            S = S + k[t, :, :, None] * u[:, None]
            o[t] = (S * q[t, :, :, None]).sum(1)
            t += 1
        states.append(S)
    z = gate.double().view(T, heads, vdim)
    want = 0.7 * o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-6) * w.double() * z * torch.sigmoid(z)
    c = lambda x: x.cuda()  # noqa: E731
    Q, AB, S, out = c(qkv), c(ab), c(S0), torch.empty(T, nv, dtype=dtype, device="cuda")
    ops.delta_mix(Q[:, :nq], Q[:, nq:2 * nq], Q[:, 2 * nq:2 * nq + nv], AB[:, :heads], AB[:, heads:], c(A_log), c(bias), S, c(cu),
                  c(ctx), c(slots), heads, kv, dim, vdim, c(gate), c(w), 1e-6, 0.7, out,
                  max_qlen=max(lens[nd:], default=1), num_decode=0 if max(lens) == 1 else nd)
    # fp32 sums over up to 128 terms, then (at 64 tokens a chunk) substitution: 2^-24 times a few hundred; bf16 results 2^-9
    err = lambda a, b: float((a.double().cpu() - b).norm() / b.norm())  # noqa: E731
    assert err(out.view(T, heads, vdim), want) < (2e-5 if dtype == torch.float32 else 4e-3)
    for b in range(B):
        assert err(S[slots[b]], states[b]) < 2e-5, b
    assert torch.equal(S[B].cpu(), S0[B])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim,vdim,heads,kv", [(4, 4, 2, 1), (36, 20, 4, 2), (64, 64, 4, 4), (128, 128, 2, 1), (128, 68, 4, 2)])
@pytest.mark.parametrize("lens,starts,nd", [([1, 1, 5, 64, 65], [5, 0, 0, 0, 9], 2), ([63, 128, 16], [0, 70, 1], 0), ([1] * 4, [0, 3, 1, 8], 4)])
def test_rows32(dim, vdim, heads, kv, lens, starts, nd, dtype):
    run(lens, starts, nd, heads, kv, dim, vdim, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [-15.0, 5.0, 100.0])
def test_rows32_decays(shift):
    """Decays from none to total."""
    run([1, 130], [2, 3], 1, 4, 2, 64, 64, torch.float32, shift)


@pytest.mark.gpu
def test_rows32_one_key_written_again():
    run([100], [0], 0, 2, 1, 64, 64, torch.float32, -15.0, same_key=True)


# a last chunk of one, two, three and four blocks of sixteen tokens, alone and behind a whole chunk, whose results and sums two waves share
@pytest.mark.gpu
@pytest.mark.parametrize("dim,vdim", [(32, 64), (64, 100), (100, 64), (128, 16)])
@pytest.mark.parametrize("lens,starts", [([16, 17, 32, 33, 48, 49], [0, 3, 0, 0, 70, 1]), ([81, 64, 112, 127], [0, 0, 9, 64]),
                                         ([145, 128, 16, 161], [0, 0, 9, 64]), ([129, 191], [5, 0])])  # (beyond 128 rows: places kept)
def test_rows32_blocks_of_the_last_chunk(dim, vdim, lens, starts):
    run(lens, starts, 0, 2, 1, dim, vdim, torch.bfloat16)
