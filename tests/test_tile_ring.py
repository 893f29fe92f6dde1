"""Batched and 32-bit-result products through the ring of k-steps (csrc/gemm_tile.hip): rows and columns about the edges of 64- and
128-row tiles, one to five k-steps, padded strides, results at odd places, bias; what lies around the result stays."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,H", [(1, 8, 64, 3), (63, 72, 128, 2), (65, 64, 192, 1), (511, 136, 64, 4), (512, 128, 128, 2), (513, 130, 64, 3),
                                     (641, 200, 320, 2), (8, 2048, 1024, 1), (700, 1, 64, 1), (130, 1030, 64, 16),
                                     (70, 72, 256, 193), (66, 520, 320, 43), (66, 520, 320, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pad,bias", [(0, False), (8, True), (3, True)])
def test_plain(M, N, K, H, dtype, pad, bias):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, H * K + 8, generator=g).bfloat16().cuda()
    B = (torch.randn(H, N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if bias else None
    C = torch.full((M + 2, H * N + pad), 7.0, dtype=dtype, device="cuda")
    hip.gemm_any(A, B, C[1:, pad // 2:], M, N, K, H, K, A.stride(0), N * K, K, 1, N, C.stride(0), b)
    Ad, Bd = A[:, :H * K].double().view(M, H, K), B.double()
    want = torch.stack([Ad[:, h] @ Bd[h].t() for h in range(H)], 1) + (b.double() if bias else 0.0)
    size = torch.stack([Ad[:, h].abs() @ Bd[h].abs().t() for h in range(H)], 1) + (b.double().abs() if bias else 0.0)
    # sums of K products in 32 bits, one rounding of the result
    lim = (K + 2) * 2.0 ** -24 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * want.abs()
    got = C[1:M + 1, pad // 2:pad // 2 + H * N].double().view(M, H, N)
    assert ((got - want).abs() <= lim).all()
    C[1:M + 1, pad // 2:pad // 2 + H * N] = 7.0
    assert (C == 7.0).all()


# a matrix of 2 GiB and one of 4 GiB, and a few rows more: columns whose rows lie where a 31- or 32-bit offset from its start ends
@pytest.mark.parametrize("N,K", [(2 ** 18 + 3, 4096), (2 ** 19 + 70, 4096), (2 ** 14 + 66, 2 ** 16)])
@pytest.mark.parametrize("M,dtype", [(3, torch.float32), (520, torch.bfloat16)])
def test_plain_large_matrix(N, K, M, dtype):
    from llmss_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16)
    w = torch.empty(N, K, device="cuda", dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g)
    y = torch.empty(M, N, dtype=dtype, device="cuda")
    hip.gemm_any(x, w, y, M, N, K, 1, 0, K, 0, K, 1, 0, N)
    edge = 2 ** 30 // K
    cols = sorted({c for at in (0, edge, 2 * edge, N // 2, N - 4) for c in range(at - 70, at + 70) if 0 <= c < N})
    wd, xd = w[cols].double(), x.double()
    want, size = xd @ wd.t(), xd.abs() @ wd.abs().t()
    lim = (K + 2) * 2.0 ** -24 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * want.abs()
    assert ((y[:, cols].double() - want).abs() <= lim).all()
