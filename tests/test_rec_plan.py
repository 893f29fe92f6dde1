"""Which form the sequences of a step take in the matrix-state recurrences (hip._rec_plan), at steps where the forms were measured, and the
forms of a mixed step against each other whatever the rule would choose."""
import pytest
import torch

from llmss_amd.ops import hip as H

WALK, CHUNK = (0, False), (0, True)


# us: token by token, chunk by chunk, single rows apart beside either
@pytest.mark.parametrize("kind,nd,B,T,longest,heads,dim,vdim,form", [
    ("decay", 0, 53, 594, 14, 32, 128, 64, WALK),  # 82, 152
    ("decay", 0, 65, 883, 24, 64, 128, 16, WALK),  # 87, 324
    ("delta", 0, 59, 336, 7, 32, 128, 32, WALK),  # 71, 217
    ("delta", 0, 60, 294, 6, 8, 128, 16, WALK),  # 22, 49
    ("ssd", 0, 29, 131, 5, 64, 128, 16, WALK),  # 23, 58
    ("decay", 1, 2, 3, 2, 16, 128, 128, WALK),  # 13.4; apart 19.3
    ("decay", 0, 8, 8192, 1024, 16, 128, 128, CHUNK),  # 1230, 290
    ("decay", 0, 64, 64 * 24, 24, 16, 128, 128, CHUNK),
    ("ssd", 0, 8, 8192, 1024, 64, 128, 64, CHUNK),  # 2160, 208
    ("delta", 0, 8, 8192, 1024, 16, 128, 128, CHUNK),  # 1615, 408
    ("delta", 58, 59, 273, 215, 16, 128, 64, (58, True)),  # 342, 239; apart 352, 88
    ("decay", 64, 64, 64, 1, 16, 128, 128, (64, False)),  # nothing but single rows
])
def test_choice(kind, nd, B, T, longest, heads, dim, vdim, form):
    assert H._rec_plan(kind, nd, B, T, longest, heads, dim, vdim, True, True) == form


def test_forms_that_do_not_take_the_step_are_not_chosen():
    assert H._rec_plan("decay", 0, 8, 8192, 1024, 16, 128, 128, True, False) == WALK
    assert H._rec_plan("decay", 64, 64, 64, 1, 16, 128, 128, False, True) == WALK
    assert H._rec_plan("delta", 58, 59, 273, 215, 16, 128, 64, False, True) == CHUNK
    assert H._rec_plan("decay", 20, 23, 34, 5, 16, 256, 128, True, False) == (20, False)  # 80; single rows apart 37


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["decay", "ssd", "delta"])
@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 36)])
def test_forms_of_a_mixed_step_agree(kind, dim, vdim, monkeypatch):
    lens, past, nd, heads = [1, 1, 1, 65, 1, 20], [4, 0, 9, 0, 0, 3], 3, 4  # a portion of one row among the others, one that continues
    g = torch.Generator().manual_seed(dim)
    T, B = sum(lens), len(lens)
    rows = torch.float32 if kind == "delta" else torch.bfloat16
    q, k, v = (torch.randn(T, heads * n, generator=g).to(rows).cuda() for n in (dim, dim, vdim))
    a, b = (torch.randn(heads, generator=g).cuda() for _ in range(2))
    dt = torch.randn(T, 2 * heads, generator=g).bfloat16().cuda()
    S0 = torch.randn(B, heads, dim, vdim, generator=g).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    ctx = torch.tensor([n + p for n, p in zip(lens, past)]).int().cuda()
    slots = torch.arange(B).int().flip(0).contiguous().cuda()
    gate, w = torch.randn(T, heads * vdim, generator=g).bfloat16().cuda(), torch.ones(vdim).bfloat16().cuda()
    got = []
    for form in (WALK, CHUNK, (nd, False), (nd, True)):
        monkeypatch.setattr(H, "_rec_plan", lambda *a: form)
        S, n = S0.clone(), dict(max_qlen=max(lens), num_decode=nd)
        if kind == "decay":
            y = H.decay_recurrence(q, k, v, torch.full((heads,), 0.9).cuda(), S, cu, ctx, slots, heads, dim, vdim, True, **n)
        elif kind == "ssd":
            y = H.ssd_recurrence(v, k, q, dt[:, :heads], a, b, a, S, cu, ctx, slots, heads, heads, dim, vdim, **n)
        else:
            y = H.delta_mix(q, k, v, dt[:, :heads], dt[:, heads:], a, b, S, cu, ctx, slots, heads, heads, dim, vdim, gate, w, 1e-6, 1.0,
                            torch.empty(T, heads * vdim, dtype=torch.bfloat16, device="cuda"), **n)
        got.append((y.double(), S.double()))
    # two forms that each meet the bounds of the tests against float64: 1e-5 (delta 2e-5), its normed rows in bf16 4e-3
    rel = lambda x, z: float((x - z).norm() / z.norm())  # noqa: E731
    for y, S in got[1:]:
        assert rel(y, got[0][0]) < (8e-3 if kind == "delta" else 2e-5)
        assert rel(S, got[0][1]) < (4e-5 if kind == "delta" else 2e-5)
