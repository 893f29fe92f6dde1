"""Routing and grouping of (token, expert) pairs (csrc/moe.hip) at the edges of their launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# K of one step, a stage of 512 and a step, two stages and a part; outputs at the edges of the row counts (16, 32, 40, 48, then whole waves),
# tokens of one launch a row (33), of 16 a workgroup with a part (259) and of 32 a workgroup with a part (4099)
@pytest.mark.parametrize("T", [33, 259, 4099])
@pytest.mark.parametrize("K,E,gate", [(32, 16, False), (544, 16, True), (1056, 32, False), (2048, 32, True), (544, 40, False), (64, 40, True),
                                      (1056, 47, True), (96, 49, False), (544, 1, True), (2080, 30, True)])
@pytest.mark.parametrize("score", ["sigmoid", "softmax", "chosen"])
def test_router_at_the_edges(T, K, E, gate, score):
    from llmss_amd.ops import hip, reference
    g = torch.Generator().manual_seed(T + K + E)
    # Small whole numbers: products and their fp32 sums are exact in any order, so equal logits are equal everywhere (the lower index
    # wins) and others differ by 2^-8 at least
    h = torch.randint(-2, 3, (T, K), generator=g).bfloat16()
    w = (torch.randint(-2, 3, (E + gate, K), generator=g) * 2.0 ** -8).bfloat16()
    bias = torch.randint(-3, 4, (E,), generator=g) * 2.0 ** -8
    corr = None if score == "chosen" else torch.randint(0, 2, (E,), generator=g).float()
    top = min(E, 5)
    want = reference.moe_router(h, w, corr, top, True, score, bias, gate)
    got = hip.moe_router(h.cuda(), w.cuda(), None if corr is None else corr.cuda(), top, True, score, bias.cuda(), gate)
    assert got[0].cpu().tolist() == want[0].tolist()
    for a, b in zip(got[1:], want[1:]):  # exponentials and quotients of fp32, a few units each; sums of five
        assert (a.cpu() - b).abs().max().item() <= 32 * 2.0 ** -24


# one workgroup with its pairs at hand (132) and read again (9000), workgroups of 1024 with a part (5000, 33044); experts past a wave's lanes
@pytest.mark.parametrize("P,blocks", [(1, 1), (132, 1), (9000, 1), (1025, 2), (5000, 5), (33044, 33)])
@pytest.mark.parametrize("E,rows", [(1, 64), (32, 16), (64, 256), (130, 16)])
def test_grouping(P, blocks, E, rows):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(P + E)
    idx = torch.randint(0, E + 2, (P,), generator=g).int()  # (from E on: no row of its own)
    idx[idx == E // 2] = 0  # one expert without pairs, one with many
    maxt = -(-P // rows) + min(E, P)
    meta = torch.full((2 + E + 2 * maxt + blocks * E,), -7, dtype=torch.int32, device="cuda")
    order, place = (torch.full((P,), -7, dtype=torch.int32, device="cuda") for _ in range(2))
    d = idx.cuda()
    hip.lib().moe_group(d.data_ptr(), P, E, maxt, meta.data_ptr(), order.data_ptr(), place.data_ptr(), rows, blocks,
                        torch.cuda.current_stream().cuda_stream)
    meta, order, place = meta.cpu(), order.cpu(), place.cpu()
    cnt = torch.bincount(idx[idx < E].long(), minlength=E)
    off = [0] + cnt.cumsum(0).tolist()
    assert meta[1:E + 2].tolist() == off
    tiles = [(e, r) for e in range(E) for r in range(off[e], off[e + 1], rows)]
    assert meta[0].item() == len(tiles) <= maxt
    at = 2 + E
    assert list(zip(meta[at:at + len(tiles)].tolist(), meta[at + maxt:at + maxt + len(tiles)].tolist())) == tiles
    own = idx < E
    assert (place[~own] == -1).all()
    p = place[own].long()
    assert p.sort().values.tolist() == list(range(off[E]))  # every row once
    assert (order[p] == torch.arange(P)[own]).all()
    e = idx[own].long()
    o = torch.tensor(off)
    assert ((p >= o[e]) & (p < o[e + 1])).all()
