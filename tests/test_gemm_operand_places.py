"""Products whose operands the newer plans cannot take - rows more than 4.2 M numbers apart, addresses off 16 bytes - keep the older
rules, and the number of split-K slabs that a caller is told to expect is the one of the plan that the launch runs."""
import pytest
import torch

from llmss_amd.ops import hip as H

WS = 64 << 20
FAR = 1 << 22


def test_slabs_follow_the_operands():
    L = H.lib()

    def slabs(M, N, K, **kw):
        return L.gemm_partial_slabs(M, N, K, False, False, 0, 0, 0, WS, **kw)
    told = {(M, N, K): slabs(M, N, K) for M in (1, 8, 16, 48, 64, 100, 300, 1000) for N in (1024, 2048, 4096, 8192)
            for K in (2048, 4096, 11008)}
    for kw in ({"ldx": FAR}, {"ldw": FAR}, {"ldx": 4100}, {"ldw": 4100}, {"x": 2}, {"w": 2}):
        other = {k: slabs(*k, **kw) for k in told}
        assert other == {k: slabs(*k, ldx=FAR) for k in told}  # one set of older rules, whatever the reason
        assert other != told
    for kw in ({"ldx": FAR - 8}, {"ldx": 4096, "x": 32}, {"ldw": 4096, "w": 16}):
        assert {k: slabs(*k, **kw) for k in told} == told


@pytest.mark.gpu
@pytest.mark.parametrize("M,ld", [(2, 1 << 24), (5, FAR), (40, FAR + 8), (65, FAR), (130, FAR)])
def test_rows_far_apart(M, ld):
    N, K = 512, 1024
    x = torch.empty((M - 1) * ld + K, dtype=torch.bfloat16, device="cuda").as_strided((M, K), (ld, 1))
    x.copy_(torch.randn(M, K, device="cuda"))
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    want = x.float() @ w.float().t()
    got = H.linear(x, w)
    assert ((got.float() - want).norm() / want.norm()).item() < 4e-3  # one rounding to bf16 (2^-9 at most)
    got = H.linear(x, w, partial_ok=True)
    if isinstance(got, H.PartialSum):
        got = got.buf[:got.S * M * N].view(got.S, M, N).sum(0)
    assert ((got.float() - want).norm() / want.norm()).item() < 4e-3
