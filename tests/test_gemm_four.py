"""Four-wave tiles of middle sizes (csrc/gemm_four.hip): every tile at its edges, gated, with bias and activation, K split in slabs or combined in
the launch, with the rotation and the cache write, against 64 bits; and the rule that chooses them."""
import pytest
import torch

from llmss_amd.ops import hip as H

TILES = {0: (64, 64), 1: (32, 64), 2: (128, 64), 3: (128, 128), 4: (128, 128), 5: (192, 128), 6: (128, 192), 7: (256, 128), 8: (64, 32),
         9: (192, 192), 10: (64, 128), 11: (128, 64), 12: (64, 128), 13: (64, 64)}
FOUR, COMBINE = 2048, 256  # hint bits of the tile code
gpu = pytest.mark.gpu


def rand(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()


def product(x, w):
    """x . w^T in 64 bits, and how far sums in 32 bits may be from it, whatever their order."""
    xd, wd = x.double(), w.double()
    return xd @ wd.t(), (x.shape[1] + 8) * 2.0 ** -24 * (xd.abs() @ wd.abs().t())


ACTS = {"none": lambda z: z, "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"), "gelu": torch.nn.functional.gelu,
        "relu": torch.relu}


@gpu
@pytest.mark.parametrize("code", sorted(TILES))
@pytest.mark.parametrize("dm,dn,K,split", [(0, 0, 64, 1), (1, 8, 128, 1), (-1, -8, 320, 1), (17, 40, 832, 2), (2, 32, 1024, 3)])
def test_edges_of_tiles(code, dm, dn, K, split):
    """Tiles that are whole, a row and a piece of a line past one, and short of one; fewer k-steps than the ring has; an uneven split."""
    bm, bn = TILES[code]
    M, N = bm + dm, 2 * bn + dn
    x, w, b = rand(1, M, K + 8)[:, :K], rand(2, N, K) * K ** -0.5, rand(3, N)
    z, e = product(x, w)
    hint = (code | FOUR | (COMBINE if split > 1 else 0)) << 8
    for act, bias in (("none", None), ("none", b), ("gelu_tanh", b), ("gelu", None), ("relu", b)):
        wide = torch.full((M + 2, N + 16), 7.0, dtype=torch.bfloat16, device="cuda")
        y = wide[1:M + 1, 8:N + 8]
        for _ in range(2):  # (the counters of the combine are clear again)
            H.linear(x, w, bias, act=act, out=y, nt_hint=hint, split_hint=split)
            v = z if bias is None else z + bias.double()
            want, lim = ACTS[act](v), 1.13 * (e + 2.0 ** -22 * v.abs())  # (no function here is steeper)
            assert ((y.double() - want).abs() <= lim + 2.0 ** -8 * (want.abs() + lim) + 2.0 ** -20 * v.abs() + 1e-6).all(), (act, bias is None)
        wide[1:M + 1, 8:N + 8] = 7.0
        assert (wide == 7.0).all()
    if split > 1:
        p = H.linear(x, w, nt_hint=(code | FOUR) << 8, split_hint=split, partial_ok=True)
        assert isinstance(p, H.PartialSum) and p.S == split
        assert ((p.buf[:split * M * N].view(split, M, N).double().sum(0) - z).abs() <= e).all()


@gpu
@pytest.mark.parametrize("code", sorted(c for c, (_, bn) in TILES.items() if bn > 32))
@pytest.mark.parametrize("act", ["none", "gelu_tanh"])
def test_gates(code, act):
    bm, bn = TILES[code]
    M, N, K = bm + 3, bn + 96, 576
    x, w, b = rand(4, M, K), rand(5, N, K) * K ** -0.5, rand(6, N)
    z, e = product(x, w)
    z = z + b.double()
    parts = [t.view(M, N // 32, 2, 16).unbind(2) for t in (z, e)]
    (g, u), (eg, eu) = [[q.reshape(M, -1) for q in p] for p in parts]
    gate = torch.nn.functional.gelu(g, approximate="tanh") if act == "gelu_tanh" else torch.nn.functional.silu(g)
    want = gate * u
    lim = 1.13 * eg * (u.abs() + eu) + gate.abs() * eu + 2.0 ** -18 * (g.abs() * u.abs() + 1e-6)
    for split in (1, 2):
        y = H.linear(x, w, b, act=act, glu=True, nt_hint=(code | FOUR | COMBINE) << 8, split_hint=split)
        assert ((y.double() - want).abs() <= lim + 2.0 ** -8 * (want.abs() + lim)).all()


@gpu
@pytest.mark.parametrize("code", sorted(TILES))
@pytest.mark.parametrize("style,D,rot", [("gptj", 64, 64), ("gptj", 32, 16), ("neox", 32, 32), ("neox", 64, 32), ("gptj", 64, 0)])
def test_rotation_and_cache_write(code, style, D, rot):
    from test_qkv_untuned import check

    nh, nkv, K, M = 6, 2, 512, 2 * TILES[code][0] - 5
    N = (nh + 2 * nkv) * D
    g = torch.Generator().manual_seed(code)
    x, w, b = rand(7, M, K), rand(8, N, K) * K ** -0.5, rand(9, N)
    pos = torch.randint(0, 90, (M,), generator=g).cuda()
    ang = torch.rand(90, max(rot // 2, 4), generator=g).cuda() * 6
    cos, sin = ang.cos(), ang.sin()
    nb = -(-M // 16) + 1
    slots = torch.randperm(nb * 16, generator=g)[:M].cuda()
    slots[M // 3] = -1
    kc, vc = (torch.zeros(nb, nkv, 16, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    y = H.linear_qkv(x, w, b, pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, style, rot > 0, (code | FOUR | code % 2 * COMBINE) << 8, 1 + code % 2)
    if style == "neox" and TILES[code][1] % D:
        assert y is None  # halves of a head in two tiles
        return
    check(y, kc, vc, x, w, b, pos, slots, cos, sin, nh, nkv, D, rot, style)


@gpu
@pytest.mark.parametrize("M,N,K", [(40, 384, 1920), (200, 1024, 8192)])
def test_replays_among_eager_launches(M, N, K):
    """A plan that combines split sums in the launch, replayed among eager launches of the same product."""
    assert H.lib().gemm_plan(M, N, K, False, False, False)[0] >> 8 & (FOUR | COMBINE) == FOUR | COMBINE
    x, w = rand(10, M, K), rand(11, N, K) * K ** -0.5
    y = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    H.linear(x, w, out=y)
    want = y.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        H.linear(x, w, out=y)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(H.linear(x, w), want)


@pytest.mark.parametrize("M,N,K,glu,plan", [
    (64, 2048, 2048, False, "four"), (100, 22016, 4096, True, "four"), (512, 12288, 4096, False, "four"), (1024, 4096, 4096, False, "four"),
    (1773, 4096, 11008, False, "four"), (2300, 2048, 5632, False, "four"), (8192, 12288, 4096, False, "quad"), (8192, 22016, 4096, True, "quad"),
    (4096, 12288, 4096, False, "quad"), (1024, 12288, 4096, False, "quad"), (1024, 4096, 4112, False, "other"), (16, 4096, 4096, False, "other")])
def test_who_takes_which_product(M, N, K, glu, plan):
    """Products of middle sizes and whole k-steps take the four-wave tiles; a gate needs its up in the same wave."""
    nt, split = H.lib().gemm_plan(M, N, K, False, glu, False)
    got = "four" if nt >> 8 & FOUR else "quad" if nt >> 8 == 4 else "other"
    assert got == plan and split == 1 or plan == "other"
    assert not (glu and got == "four" and TILES[nt >> 8 & 15][1] == 32)


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N", [256, 1024, 2048])
@pytest.mark.parametrize("K", [1024, 2048, 5632, 1040])
def test_closing_products_stay_in_32_bits(M, N, K):
    """Where the finished product's K was split, its closing op still gets unsummed slabs."""
    nt, split = H.lib().gemm_closing_plan(M, N, K)
    assert split > 1 or M <= 32  # (up to 32 rows the decode kernel's, unsplit)
    if split > 1:
        assert H.lib().gemm_partial_slabs(M, N, K, False, False, 0, nt, split, 64 << 20) == split


@pytest.mark.parametrize("M,N,K,glu", [(32, 5528, 11328, False), (25, 5752, 7104, False), (28, 5760, 6976, False), (66, 10240, 11392, True),
                                       (121, 10016, 7744, False), (80, 10568, 7744, False)])
def test_long_products_of_few_tiles_split_k(M, N, K, glu):
    """87 - 168 tiles with 100 - 180 steps of K each leave half of the CUs idle and took 1.2 - 1.5 times as long as with K split."""
    nt, _ = H.lib().gemm_plan(M, N, K, False, glu, False)
    bm, bn = TILES[nt >> 8 & 15]
    assert nt >> 8 & FOUR and (nt >> 8 & COMBINE or -(-M // bm) * -(-N // bn) >= 192)
