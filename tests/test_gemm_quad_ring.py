"""256 x 256 products of more tiles than CUs (csrc/gemm_quad.hip): a workgroup takes several tiles, its ring of loads running on from one into
the next, plain, gated and over expert tile lists; a last round that few workgroups have."""
import pytest
import torch

from test_gemm_quad import bound, test_experts_two_matrices as two_matrices
from test_gemm_quad import test_glu as gated

pytestmark = pytest.mark.gpu


# K: fewer steps than reach into another tile (each tile a workgroup), as many as just do, an odd number; M and N: tiles whole and partial, two
# rounds and a bit, four
@pytest.mark.parametrize("M,N,K", [(4200, 4360, 192), (4097, 4096, 256), (4100, 4360, 320), (8200, 4104, 576), (16500, 4096, 1024)])
@pytest.mark.parametrize("bias", [False, True])
def test_many_tiles(M, N, K, bias):
    from llmss_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g, device="cuda").bfloat16() if bias else None
    wide = torch.full((M + 2, N + 16), 7.0, dtype=torch.bfloat16, device="cuda")
    y = wide[1:M + 1, 8:N + 8]
    hip.linear(x, w, b, out=y, nt_hint=4 << 8, split_hint=1)
    assert torch.equal(y, hip.linear(x, w, b, nt_hint=4 << 8, split_hint=1))
    ref = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    assert ((y.double() - ref).abs() <= bound(x, w, ref)).all()
    wide[1:M + 1, 8:N + 8] = 7.0
    assert (wide == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(4100, 4384, 320), (8200, 8192, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_many_gated_tiles(M, N, K, bias):
    gated(M, N, K, bias)


# experts' lists of more tiles than CUs in both products, one expert without a row, partial tiles of each
@pytest.mark.parametrize("E,top,W,F,T", [(5, 2, 1024, 1088, 9001), (9, 3, 1280, 768, 6007)])
@pytest.mark.parametrize("weighted", [True, False])
def test_many_tiles_of_experts(E, top, W, F, T, weighted, monkeypatch):
    two_matrices(E, top, W, F, T, "silu", weighted, monkeypatch)


@pytest.mark.parametrize("kind", ["interleaved", "gelu"])
def test_many_tiles_of_experts_in_one_matrix(kind):
    from llmss_amd.ops import glu_interleave, hip
    E, top, T, W, F, N = 3, 2, 12000, 512, 1024, 1032
    g = torch.Generator(device="cuda").manual_seed(5)
    h = torch.randn(T, W, generator=g, device="cuda").bfloat16()
    gate, up = ((torch.randn(E, F, W, generator=g, device="cuda") * W ** -0.5).bfloat16() for _ in range(2))
    down = (torch.randn(E, N, F, generator=g, device="cuda") * F ** -0.5).bfloat16()
    idx = torch.stack([torch.randperm(E)[:top] for _ in range(T)]).int().cuda()
    w = torch.rand(T, top, generator=g, device="cuda")
    if kind == "gelu":
        y = hip.moe_experts(h, idx, w, None, up, down, 0.0, 0.0, act="gelu")
    else:
        y = hip.moe_experts(h, idx, w, None, glu_interleave(gate, up, 1).contiguous(), down, 0.0, 0.0, act="silu", interleaved=True)
    want = torch.zeros(T, N, dtype=torch.float64, device="cuda")
    for e in range(E):
        for j in range(top):
            r = (idx[:, j] == e).nonzero()[:, 0]
            x = h[r].double()
            a, b = (x @ m[e].double().t() for m in (gate, up))
            v = torch.nn.functional.gelu(b) if kind == "gelu" else torch.nn.functional.silu(a) * b
            want[r] += w[r, j].double()[:, None] * (v @ down[e].double().t())
    # the activations rounded to bf16 once (2^-9 of each, of random sign over F of them), sums in fp32, row by row
    assert ((y.double() - want).norm(dim=1) / want.norm(dim=1)).max().item() < 8e-3


# experts with rests of half a tile and less, which come last and by halves: one row, a matrix instruction's sixteen, 127 - 129 and whole tiles; more
# tiles than CUs in both products, fewer, and only halves
@pytest.mark.parametrize("counts,F,N", [([1000, 128, 2300, 129, 16, 513, 640], 2048, 3080), ([127, 1, 1536, 17, 256 + 255, 0], 288, 264),
                                        ([2048, 384 + 1, 256 + 31], 3072, 2048), ([100, 128, 90, 33, 64, 12, 128, 1], 640, 520),
                                        ([1000, 900, 128, 17, 2], 320, 16640)])  # (sums of 136 MB, past the caches)
@pytest.mark.parametrize("kind", ["two", "interleaved", "gelu"])
def test_half_tiles_of_experts(counts, F, N, kind, monkeypatch):
    from llmss_amd.ops import glu_interleave, hip
    E, W, P = len(counts), 320, sum(counts)
    g = torch.Generator(device="cuda").manual_seed(P)
    h = torch.randn(P, W, generator=g, device="cuda").bfloat16()
    gate, up = ((torch.randn(E, F, W, generator=g, device="cuda") * W ** -0.5).bfloat16() for _ in range(2))
    down = (torch.randn(E, N, F, generator=g, device="cuda") * F ** -0.5).bfloat16()
    idx = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(P)].int()[:, None].cuda()
    w = torch.rand(P, 1, generator=g, device="cuda")
    for name in ("MOE_PP_ROWS", "MOE_PP_ROWS_TWO", "MOE_DEC_ROWS"):
        monkeypatch.setattr(hip, name, 0)
    monkeypatch.setattr(hip, "_moe_plan", lambda *a: (256, 0))
    if kind == "gelu":
        y = hip.moe_experts(h, idx, w, None, up, down, 0.0, 0.0, act="gelu")
    elif kind == "two":
        y = hip.moe_experts(h, idx, w, gate, up, down, 0.0, 0.0, act="silu")
    else:
        y = hip.moe_experts(h, idx, w, None, glu_interleave(gate, up, 1).contiguous(), down, 0.0, 0.0, act="silu", interleaved=True)
    for e in range(E):
        r = (idx[:, 0] == e).nonzero()[:, 0]
        if not len(r):
            continue
        a, b = (h[r].double() @ m[e].double().t() for m in (gate, up))
        v = torch.nn.functional.gelu(b) if kind == "gelu" else torch.nn.functional.silu(a) * b
        want = w[r].double() * (v @ down[e].double().t())
        # the activations rounded to bf16 once (2^-9 of each, of random sign over F of them), sums in fp32, row by row
        assert ((y[r].double() - want).norm(dim=1) / want.norm(dim=1)).max().item() < 8e-3


@pytest.mark.parametrize("P,blocks", [(700, 1), (9000, 1), (33044, 33)])
@pytest.mark.parametrize("E,rows", [(1, 256), (64, 256), (130, 64)])
def test_list_with_its_half_tiles_last(P, blocks, E, rows):
    from llmss_amd.ops import hip
    idx = torch.randint(0, E, (P,), generator=torch.Generator().manual_seed(P + E)).int()
    maxt = -(-P // rows) + min(E, P)
    meta = torch.full((3 + E + 2 * maxt + blocks * E,), -7, dtype=torch.int32, device="cuda")
    order, place = (torch.full((P,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
    d = idx.cuda()
    hip.lib().moe_group_tall(d.data_ptr(), P, E, maxt, meta.data_ptr(), order.data_ptr(), place.data_ptr(), rows, blocks,
                             torch.cuda.current_stream().cuda_stream)
    meta = meta.cpu()
    off = [0] + torch.bincount(idx.long(), minlength=E).cumsum(0).tolist()
    assert meta[1:E + 2].tolist() == off
    tiles = [(e, r, 2 * (off[e + 1] - r) > rows) for e in range(E) for r in range(off[e], off[e + 1], rows)]
    tiles = [t[:2] for t in tiles if t[2]] + [t[:2] for t in tiles if not t[2]]
    tall = sum(2 * (off[e + 1] - r) > rows for e, r in tiles)
    assert meta[0].item() == len(tiles) <= maxt and meta[2 + E + 2 * maxt].item() == tall
    at = 2 + E
    assert list(zip(meta[at:at + len(tiles)].tolist(), meta[at + maxt:at + maxt + len(tiles)].tolist())) == tiles
    assert (order.cpu()[place.cpu().long()] == torch.arange(P)).all()
