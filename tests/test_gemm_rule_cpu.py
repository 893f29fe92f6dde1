"""Which products of up to 64 rows the decode GEMM takes without a hint or tuned plan, at shapes where both sides were measured (us,
older rules against decode kernel): a wave of workgroups that reads X once per narrow tile, or a second, nearly empty wave, must not win."""
import pytest

from llmss_amd.ops import hip as H

DEC = 1024  # the hint bit of the decode kernel


@pytest.mark.parametrize("M,N,K,dec", [
    (20, 23200, 1136, False),  # 18.4 against 52.2: slabs of a wide product
    (64, 23200, 1136, False),  # 21.9, 65.1
    (17, 24992, 288, False),  # 8.6, 22.7
    (17, 10560, 7776, False),  # 37.5, 55.1
    (48, 20672, 2272, False),  # 32.0, 41.8
    (1, 4096, 4096, True),  # 13.6, 9.6
    (1, 1600, 6400, True),
    (16, 4096, 11008, True),
    (20, 4096, 4096, True),
])
def test_choice(M, N, K, dec):
    nt, _ = H.lib().gemm_plan(M, N, K, False)
    assert bool(nt >> 8 & DEC) == dec
