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


WIDE = {15: 96, 11: 128}  # tiles of 64 rows by so many columns


@pytest.mark.parametrize("M,N,K,glu,form", [
    (23, 32000, 4096, False, "dec"),  # LM heads and wide products of 17 - 32 rows: 62.1 against 48.0
    (24, 22016, 4096, False, "dec"),  # 46.4, 35.4
    (20, 16384, 4096, False, "dec"),  # 34.2, 26.0
    (29, 6824, 15616, False, "older"),  # 44.1, 53.4: X once more for every tile
    (64, 22016, 4096, True, 96),  # 53, 39
    (33, 43776, 8160, True, 96),  # 181.9, 177.6; in tiles of 128 columns, a second, nearly empty wave, 223.4
    (45, 35616, 384, True, "older"),  # 10.0, 13.9
    (49, 48128, 320, False, "older"),  # 13.7, 17.6
    (52, 40328, 384, False, "older"),  # 14.4, 18.2
])
def test_choice_of_finished_products(M, N, K, glu, form):
    nt, _ = H.lib().gemm_plan(M, N, K, False, glu=glu, slabs=False)
    tile = nt >> 8
    assert form == ("dec" if tile & DEC else WIDE.get(tile & 15, "older"))
