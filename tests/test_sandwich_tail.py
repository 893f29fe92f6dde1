"""The next router and the token input in the closing op's launch (csrc/sandwich.hip), against the launches of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def closing(kind, T, W, g):
    """(y, gate logits, their bias) of one kind of sublayer result."""
    from llmss_amd.ops import hip
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    if kind == "plain":
        return rnd(T, W + 8).bfloat16()[:, :W], None, None
    if kind == "gated":
        return rnd(T, W).bfloat16(), rnd(T, 2 * W).bfloat16()[:, W:], rnd(W)
    if kind == "slabs":
        p = hip.PartialSum(rnd(3 * T * W), 3, T, W, None, torch.device("cuda"))
        return p, None, None
    if kind == "pair":
        return hip.PairPending(rnd(T, W).bfloat16(), rnd(T, W).bfloat16(), rnd(W), rnd(W), None), None, None
    if kind == "scaled pair":
        return hip.PairPending(rnd(T, W).bfloat16(), rnd(T, W).bfloat16(), None, None, (0.7, 0.6)), None, None
    if kind == "none":
        return None, None, None
    top = 5  # experts: more than the four in flight
    place = torch.randperm(T * top, generator=g).int().cuda()
    return hip.MoEPending(rnd(T * top, W), place, torch.rand(T, top, generator=g).cuda(), rnd(T, W).bfloat16(), None, None,
                          torch.rand(T, generator=g).cuda()), None, None


KINDS = ["plain", "gated", "slabs", "pair", "scaled pair", "experts", "none"]


def close(a, b, lim):
    # fp32 sums over a row in another order, behind them one rounding to bf16 that may fall the other way
    return ((a.float() - b.float()).abs() <= lim * b.float().abs() + lim * 2.0 ** -3).all()


# outputs: one, a look's 40 and more, the largest number; widths with idle threads, not in whole 512s; one row and the most
@pytest.mark.parametrize("T,W,E,top,gate", [(1, 64, 1, 1, True), (33, 2048, 32, 4, False), (8, 1024, 16, 2, True), (256, 520, 41, 3, True),
                                            (5, 1096, 128, 8, False), (5, 1096, 40, 8, False), (4, 1032, 40, 8, True)])
@pytest.mark.parametrize("kind", KINDS)
def test_route(T, W, E, top, gate, kind, monkeypatch):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(W + E)
    y, r, rb = closing(kind, T, W, g)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x, wpost, wnext, add = rnd(T, W), rnd(W), rnd(W), rnd(W)
    route = ((rnd(E + int(gate), W) * W ** -0.5).bfloat16(), None if E == 32 else rnd(E), top, True, "sigmoid", rnd(E) if gate else None, gate)
    x1, x2 = x.clone(), x.clone()
    lib, calls = hip.lib(), []

    class Seen:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(lib, name)
    with monkeypatch.context() as m:
        m.setattr(hip, "lib", Seen)
        hip.sandwich_add_norm(x.clone(), y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16, route=route)
        assert calls.count("sandwich_tail") == (W >= 768 and E + gate <= 40)  # (narrow rows and many outputs: two launches are the faster ones)
        m.setattr(hip, "TAIL_WIDTH", 0)
        m.setattr(hip, "TAIL_OUTPUTS", 129)
        calls.clear()
        h1, got = hip.sandwich_add_norm(x1, y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16, route=route)
        assert calls.count("sandwich_tail") == 1
    monkeypatch.setattr(hip, "TAIL_ROWS", -1)
    h2, _ = hip.sandwich_add_norm(x2, y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16, route=route)
    assert close(x1, x2, 2.0 ** -17) and close(h1, h2, 2.0 ** -7)
    want = hip.moe_router(h1, *route)  # the same sums in the same order
    assert len(got) == len(want) == 2 + int(gate)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,W,d", [(1, 256, 32), (33, 2048, 32), (256, 1024, 64), (7, 1792, 64)])
@pytest.mark.parametrize("kind", KINDS)
def test_token_side(T, W, d, kind, monkeypatch):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(W + d)
    y, r, rb = closing(kind, T, W, g)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x, wpost, wnext, add = rnd(T, W), rnd(W), rnd(W) if T != 7 else None, rnd(T, W) if d == 64 else None
    ids = torch.randint(-1, 12, (T,), generator=g).cuda()  # (ids past the table's ends: its first and last row)
    side = (ids, rnd(11, d + 16).bfloat16(), 8, (rnd(d, W) * W ** -0.5).bfloat16(), rnd(W, d).bfloat16(), rnd(W))
    x1, x2 = x.clone(), x.clone()
    h1 = hip.sandwich_add_norm(x1, y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16, side=side)
    monkeypatch.setattr(hip, "TAIL_ROWS", -1)
    h2 = hip.sandwich_add_norm(x2, y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16, side=side)
    assert close(x1, x2, 2.0 ** -16) and (wnext is None and h1 is None and h2 is None or close(h1, h2, 2.0 ** -7))


# rows in registers on either side of the sizes where that form begins, and streams that pass the caches by
@pytest.mark.parametrize("T,W", [(2048, 2048), (2049, 1284), (2049, 2048), (6144, 2048), (9600, 1312)])
@pytest.mark.parametrize("kind", ["plain", "gated", "scaled pair", "experts"])
def test_many_rows(T, W, kind):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(T)
    y, r, rb = closing(kind, T, W, g)
    x, wpost, wnext, add = (torch.randn(*s, generator=g).cuda() for s in ((T, W), (W,), (W,), (T, W)))
    v = y
    if kind == "scaled pair":
        v = 0.7 * y.yl.double() + 0.6 * y.yr.double()
    elif kind == "experts":
        v = (y.y.double()[y.place.long()].view(T, y.top, W) * y.wts.double()[..., None]).sum(1) + y.shared_w.double()[:, None] * y.shared.double()
    v = v.double() * (torch.sigmoid(r.double() + rb.double()) if r is not None else 1.0)
    norm = lambda t: t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + 1e-5)  # noqa: E731
    want = x.double() + norm(v) * wpost.double() + add.double()
    h = hip.sandwich_add_norm(x, y, r, rb, wpost, 1e-5, add, wnext, torch.bfloat16)
    # fp32: a sum of W squares and some 20 roundings of terms of up to the largest number's size; one to bf16
    assert ((x.double() - want).abs() <= 2.0 ** -18 * want.abs().amax(-1, keepdim=True)).all()
    hw = norm(want) * wnext.double()
    assert ((h.double() - hw).abs() <= 2.0 ** -8 * hw.abs() + 2.0 ** -16 * hw.abs().amax(-1, keepdim=True)).all()
