"""The token input over enough rows for the matrix-core form (1024 and more), against float64: widths and depths at its edges, a
last block of rows that is not full, ids outside the table, with and without the added rows and the next norm."""
import pytest
import torch

from llmss_amd import ops


@pytest.mark.gpu
# (below 1024 rows, and up to 2048 wide: a row per workgroup with its weights in registers)
@pytest.mark.parametrize("T,W,d,add,nxt", [(1, 256, 64, True, True), (3, 1024, 32, False, True), (33, 1280, 32, True, False),
                                           (2, 2048, 64, True, True), (5, 2048, 32, False, True), (2, 1024, 64, False, True),
                                           (2, 2304, 32, False, True), (1024, 256, 32, False, True), (1025, 1024, 32, True, True), (1039, 2048, 64, True, False),
                                           (1040, 2304, 32, False, True), (1100, 4096, 64, True, True), (1024, 4352, 32, False, True),
                                           (1023, 2048, 32, True, True), (1030, 2000, 32, False, True)])
def test_token_side_rows(T, W, d, add, nxt):
    gen = torch.Generator().manual_seed(W + d)
    rn = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    x, table = rn(T, W) * 3, rn(97, 3 * d).bfloat16()
    ids = torch.randint(-2, 99, (T,), generator=gen)
    wg, wp = (rn(d, W) * W ** -0.5).bfloat16(), (rn(W, d) * d ** -0.5).bfloat16()
    wn, wx, extra = 1 + 0.1 * rn(W), 1 + 0.1 * rn(W), rn(T, W) if add else None
    e = table.double()[ids.clamp(0, 96)][:, d:2 * d]
    z = x.double() @ wg.double().T
    y = (0.5 * z * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3))) * e) @ wp.double().T
    norm = lambda v: v / torch.sqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6)  # noqa: E731
    want = x.double() + norm(y) * wn.double() + (extra.double() if add else 0)
    c = lambda t: None if t is None else t.cuda()  # noqa: E731
    X = c(x)
    h = ops.token_side_add(X, c(ids), c(table), d, c(wg), c(wp), c(wn), 1e-6, c(extra), c(wx) if nxt else None, torch.bfloat16)
    # fp32 sums over up to 4352 terms: 2^-24 times a few dozen; the normed rows leave in bf16
    assert float((X.double().cpu() - want).norm() / want.norm()) < 3e-6
    assert float((X.double().cpu() - want).abs().max()) < 1e-3
    if nxt:
        hw = norm(want) * wx.double()
        assert float((h.double().cpu() - hw).norm() / hw.norm()) < 4e-3
    else:
        assert h is None
