"""Products without hints or tuned plans, over the rows and widths at which the plan changes: results against fp32, and the
number of split-K slabs the wrapper expects against what the launch leaves."""
import pytest
import torch

from llmss_amd.ops import hip as H

SHAPES = [(1024, 2048), (1600, 1600), (2048, 5632), (4096, 1376), (9248, 512), (16392, 64), (24, 4112)]


def rel(a, b):
    return float((a.float() - b).norm() / b.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 129, 300, 513, 1000, 2100])
def test_products(M):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    for N, K in SHAPES:
        x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
        w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
        b = torch.randn(N, generator=gen, device="cuda").bfloat16()
        want = x.float() @ w.float().t()
        # one rounding to bf16 (2^-9 at most, 0.2 % on average over the numbers' scale) after fp32 sums
        assert rel(H.linear(x, w), want) < 4e-3, (N, K)
        assert rel(H.linear(x, w, b, "relu"), torch.relu(want + b.float())) < 4e-3, (N, K)
        got = H.linear(x, w, b, partial_ok=True)
        if isinstance(got, H.PartialSum):
            slabs = got.buf[:got.S * M * N].view(got.S, M, N)
            assert rel(slabs.sum(0), want) < 1e-5, (N, K)
        else:
            assert rel(got, want + b.float()) < 4e-3, (N, K)
        if N % 32 == 0:
            z = want.view(M, N // 32, 2, 16)  # gate and up rows in alternating groups of 16
            h = (torch.nn.functional.silu(z[:, :, 0]) * z[:, :, 1]).reshape(M, N // 2)
            assert rel(H.linear(x, w, glu=True), h) < 4e-3, (N, K)


@pytest.mark.gpu
def test_rows_of_a_wider_matrix():
    x = torch.randn(200, 3000, device="cuda").bfloat16()[:, 8:1032]
    w = (torch.randn(4096, 1024, device="cuda") / 32).bfloat16()
    for M in (5, 40, 200):
        assert rel(H.linear(x[:M], w), x[:M].float() @ w.float().t()) < 4e-3
