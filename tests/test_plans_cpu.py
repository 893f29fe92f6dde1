"""Host-side plan logic (no GPU): autotuner candidate lists for the decode GEMM tiles and the workspace slots
that keep concurrently running kernel chains apart (ops/autotune.py, ops/hip.py)."""
import pytest

from llmss_amd.ops import autotune as A


def _tiles(cands):
    return {(nt >> 8) & 15 for nt, _ in cands if nt >> 8}


@pytest.mark.parametrize("M,N,K,glu", [(64, 12288, 4096, False), (64, 22016, 4096, True), (64, 4096, 11008, False),
                                       (512, 1536, 4096, False), (64, 6400, 1600, False)])
def test_candidates_cover_the_round3_tiles(M, N, K, glu):
    c = A.candidates(M, N, K, glu, False)
    assert len(set(c)) == len(c), "duplicate candidates"
    # the gemm_mid decode tiles: 64x192 (13), 64x32 (14), 64x96 (15), 64x48 (7), and the odd / large splits
    assert {7, 13, 14, 15} <= _tiles(c)
    nk = -(-K // 64)
    for nt, s in c:
        assert s >= 1 and (s == 1 or nk // s >= 1)
    if nk // 11 >= 2:
        assert any(s == 11 for _, s in c)


def test_qkv_epilogue_candidates_are_combined_or_unsplit():
    for nt, s in A.qkv_epi_candidates(64, 12288, 4096, 128, False):
        assert s == 1 or (nt >> 8) & 256, (hex(nt), s)  # a split plan must combine in-launch
    # neox RoPE needs head-aligned tiles: no 64x48 / 64x96 / 64x192 plans for D = 128
    neox = _tiles(A.qkv_epi_candidates(64, 12288, 4096, 128, True))
    assert not ({7, 13, 14, 15} & neox)


def test_w8a8_candidates_include_the_fp8_gemm_mid_tiles():
    from llmss_amd.ops.hip import W8A8_FLAG

    c = [nt for nt, _ in A.candidates(64, 10240, 8192, False, True) if nt & W8A8_FLAG]
    tiles = {(nt >> 8) & 15 for nt in c}
    assert {7, 10, 11, 13, 15} <= tiles
    assert not [nt for nt, _ in A.candidates(64, 10240, 8200, False, True) if nt & W8A8_FLAG and (nt >> 8) & 15 >= 7]


def test_workspace_slots_are_disjoint():
    from llmss_amd.ops import hip as H

    a0 = H._GEMM_WS._items[0]
    with H.workspace_slot(1):
        assert H._GEMM_WS._items[H._SLOT.k] is not a0
        with H.workspace_slot(2):
            assert H._SLOT.k == 2
        assert H._SLOT.k == 1
    assert getattr(H._SLOT, "k", 0) == 0


def test_interleaved_ring_candidates_only_where_the_kernel_takes_them():
    """Hint bit 512 (gemm_mid ILV) appears for M >= ILV_MIN_M, K % 64 == 0 and ring depths >= 3 only."""
    ilv = lambda c: [(n, s) for n, s in c if n & (512 << 8)]
    assert ilv(A.candidates(512, 1536, 4096, False, False))
    assert all(((n >> 8) & 48) >= 16 for n, _ in ilv(A.candidates(512, 1536, 4096, False, False)))
    assert not ilv(A.candidates(64, 1536, 4096, False, False))
    assert not ilv(A.candidates(512, 4096, 1376, False, False))  # partial last k-step


def test_w8a8_software_pipelined_candidates_are_4_wave_gemm_mid_tiles():
    """W8A8_ILV (the fp8 gemm_mid k-loop with the next step's reads between the MFMAs) is a candidate for M >= 128
    on the 4-wave gemm_mid tiles only: the 8-wave ones spill its second fragment set (profiles/r6_f8)."""
    from llmss_amd.ops.hip import W8A8_FLAG, W8A8_ILV

    c = [(n, s) for n, s in A.candidates(512, 7168, 8192, True, True) if n & W8A8_FLAG and n & W8A8_ILV]
    tiles = {(n >> 8) & 15 for n, _ in c}
    assert 8 in tiles and 11 in tiles and not tiles & {9, 12} and tiles <= {7, 8, 10, 11, 13, 15}
    assert all(3 <= (n >> 12) & 15 <= 5 for n, _ in c)
    assert not [n for n, _ in A.candidates(64, 7168, 8192, True, True) if n & W8A8_FLAG and n & W8A8_ILV]


@pytest.mark.parametrize("col", ["4", "0"])
def test_model_shapes_include_the_column_chunks_when_forced(monkeypatch, col):
    """The autotuner tunes o / down's column slices (DecoderLM._reduce_cols) whenever the column schedule can run."""
    import torch

    from llmss_amd.models.config import get_preset
    from llmss_amd.models.decoder import DecoderLM
    from llmss_amd.models.weights import random_weights
    from llmss_amd.parallel.dist import TPGroup

    monkeypatch.setenv("LLMSS_TP_COL", col)
    cfg = get_preset("llama2-7b", num_layers=1, hidden_size=256, intermediate_size=512, num_heads=4, head_dim=64,
                     num_kv_heads=4, rotary_dim=64, vocab_size=512, max_position_embeddings=64)
    tp = TPGroup(0, 2, fake=True, sim_comm=(15.0, 150.0))
    m = DecoderLM(cfg, random_weights(cfg, tp=2, rank=0, dtype=torch.float32, seed=0), tp)
    shapes = A.model_shapes(m)
    L = m.w.layers[0]
    if col == "0":
        assert "o_col" not in shapes and "down_col" not in shapes
    else:
        assert shapes["o_col"] == A.GemmShape(L.o.N // 4, L.o.K)
        assert shapes["down_col"] == A.GemmShape(L.down.N // 4, L.down.K)


@pytest.mark.parametrize("M,N,K", [(65536, 4096, 1376), (8192, 4096, 4096), (65536, 1536, 4096), (8192, 1600, 1600)])
def test_prompt_batch_plans_take_the_ping_pong_kernel(M, N, K):
    """Every prompt-batch projection with enough 256x256 tiles runs the ping-pong kernel (tile code 4), including
    K % 64 != 0 (Llama-2-7B's TP=8 down projection, K = 1376: its partial last K-tile reads a zero page; before
    that it fell back to the 128x128 kernel, profiles/r5_prefill_tp8)."""
    from llmss_amd.ops import hip as H

    nt, split = H.lib().gemm_plan(M, N, K, False)
    assert (nt >> 8) & 15 == 4 and split == 1, (hex(nt), split)


@pytest.mark.parametrize("M,N,K,glu,slabs,dec", [
    (1, 12288, 4096, False, False, True), (32, 22016, 4096, True, False, True), (33, 22016, 4096, True, False, False),
    (23, 4096, 11008, False, True, True), (16, 53344, 256, False, False, False), (16, 16384, 1008, False, False, True),
    (15, 1856, 12240, True, False, False), (13, 2848, 6528, True, False, True)])
def test_fp8_products_of_few_rows_take_the_decode_kernel(M, N, K, glu, slabs, dec):
    """Up to 32 rows of fp8 weights: gemm_dec.hip (hint bit 1024), split where the consumer sums slabs that the older plan left
    too; many waves of a short K and SwiGLU of few columns with a long K keep the older kernels."""
    from llmss_amd.ops import hip as H

    nt, split = H.lib().gemm_plan(M, N, K, True, glu, slabs)
    assert bool((nt >> 8) & 1024) == dec, (hex(nt), split)
    if dec:
        assert (split > 1) == slabs and ((nt >> 8) & 15) <= 4


@pytest.mark.parametrize("M,N,K,glu,cut", [(8192, 12288, 4096, False, None), (8192, 5120, 2048, False, None), (5000, 12288, 4096, False, None),
                                           (8261, 2048, 2048, False, "rows"), (1773, 12288, 4096, False, "any"), (3999, 22016, 4096, True, "any"),
                                           (2500, 6144, 2048, False, None), (9999, 10160, 256, False, None), (6783, 10256, 384, False, None),
                                           (1649, 11200, 512, True, "any"), (8261, 2048, 512, False, "rows")])
def test_products_are_cut_where_the_last_wave_of_tiles_is_nearly_empty(M, N, K, glu, cut):
    """Whole waves of 256 x 256 tiles in one launch and the rest in another: never for products that fill their waves, at multiples
    of a tile, by rows or by columns but not both."""
    from llmss_amd.ops import hip as H

    rows, cols = H.lib().gemm_cut(M, N, K, glu)
    assert not (rows and cols) and rows % 256 == 0 and cols % 256 == 0 and rows < M and cols < N
    assert bool(rows or cols) == (cut is not None) and (cut != "rows" or rows == 8192)


@pytest.mark.parametrize("M,N,K,cut,split", [(4106, 15840, 11520, (4096, 0), 1), (6662, 7264, 8448, (6656, 0), 1), (6161, 15888, 10688, (6144, 0), 1),
                                             (8261, 2048, 4096, (8192, 0), 4), (4317, 3952, 9216, (0, 3840), 3), (6851, 2336, 8704, (0, 2304), 4)])
def test_split_rests_cut_elsewhere_only_beside_more_than_64_rows(M, N, K, cut, split):
    """The rest of a cut product may split K (``split``: of the launch that it gets, by the plan of its size), and the product be cut where that
    pays; but up to 64 rows left over, which are priced above what they take, stay where they are (1110 us against 1180 for the first, 631 and
    660, 1858 and 1907)."""
    from llmss_amd.ops import hip as H

    assert tuple(H.lib().gemm_cut(M, N, K, False)) == cut and H.lib().gemm_cut_split(M, N, K, False) == split


@pytest.mark.parametrize("E,pairs,F,K,glu,rows,plan", [
    (142, 70, 768, 128, True, 64, (64, (0, 2))),    # 57 us without the ring, 77 on its tiles of 128 rows
    (36, 96, 1664, 256, True, 64, (64, (1, 2, 3))),  # 65, 70; 57 on those of 64
    (64, 55, 896, 768, True, 64, (64, (0,))),       # 82; 89 on either
    (61, 194, 896, 320, True, 256, (64, (0,))),     # 79, as on 256 rows; 92 on 128
    (16, 38, 512, 1024, True, 64, (64, (3,))),      # 41; 30
    (16, 188, 512, 1024, True, 256, (64, (1, 3))),  # 62; 42
    (32, 64, 768, 2048, True, 64, (128, (3,))),     # 114; 90, 108 on 64 rows
    (32, 103, 768, 2048, True, 64, (128, (3,))),    # 116; 99
])
def test_expert_layers_take_the_ring_where_it_is_the_faster_one(E, pairs, F, K, glu, rows, plan):
    """Rows of a tile and the products that go through the ring of k-steps, at layers where both were measured (us)."""
    from llmss_amd.ops import hip as H

    got = H.lib().moe_plan(E * pairs, E, F, K, K, glu, rows, min(F, K) >= 256)
    assert got[0] == plan[0] and got[1] in plan[1], got


@pytest.mark.parametrize("M,N,K,batch,ring", [
    (3680, 40, 128, 16, False),  # 8.3 us without the ring, 9.9 with it
    (383, 2040, 192, 8, False),  # 14.5, 17.6
    (8, 3936, 64, 40, False),    # 10.3, 14.3
    (71, 1905, 320, 16, False),  # 14.6, 16.7: a wave and a quarter
    (8261, 256, 128, 16, True),  # 45.5, 35.6
    (64, 2048, 2048, 1, True),   # 23.2, 11.6
    (64, 4096, 1024, 24, True), (64, 4096, 130, 1, False),
])
def test_batched_products_take_the_ring_where_it_is_the_faster_one(M, N, K, batch, ring):
    from llmss_amd.ops import hip as H

    assert H.lib().gemm_tile_rings(M, N, K, batch) == ring


@pytest.mark.parametrize("T,top,E,F,N,shared,own", [
    (33, 4, 32, 768, 2048, True, True), (8, 2, 16, 512, 1024, True, True), (8, 8, 64, 64, 512, False, True),
    (13, 4, 64, 576, 3392, False, False),     # 81 us with a grouping launch, 99 without
    (55, 16, 512, 64, 2112, False, False),    # 135, 181
    (17, 4, 160, 64, 3840, False, False),     # 37, 49
])
def test_few_row_experts_find_their_rows_where_that_is_the_faster_way(T, top, E, F, N, shared, own):
    from llmss_amd.ops import hip as H

    assert H._moe_own_rows(T, top, E, F, N, N, True, shared) == own


@pytest.mark.parametrize("block", [2, 16, 48])
@pytest.mark.parametrize("group,head_dim,fp8,alone", [(1, 128, True, 800), (2, 128, True, 800), (1, 64, True, 800), (1, 64, False, 512),
                                                      (4, 128, True, 0), (1, 256, True, 0), (1, 128, False, 0), (2, 64, False, 0),
                                                      (8, 128, False, 0)])
def test_one_partition_only_where_no_mix_of_lengths_is_slower(group, head_dim, fp8, alone, block):
    """Decode attention's partitions: one from 640 (sequence, kv-head) pairs up to the positions that a workgroup walks in time, or where a
    partition of 256 holds them or the pairs fill the chip; elsewhere as many as fill it, of at least 256. They cover the contexts."""
    from llmss_amd.ops import hip as H

    for pairs in (1, 639, 640, 1000, 2047, 2048, 5000):
        for ctx in (1, 256, 257, 400, 512, 513, 800, 801, 2048, 4000):
            n, size = H.decode_splits(pairs, 1, ctx, block, group, head_dim, fp8)
            assert n * size >= ctx and size % block == 0 and (n - 1) * size < ctx
            one = pairs >= 640 and ctx <= min(alone, 256 * block) or ctx <= 256 or pairs >= 2048
            assert (n == 1) == one and n <= -(-2048 // pairs)


@pytest.mark.parametrize("total,B,longest,nh,nkv,D,two", [
    (1900, 2, 950, 32, 32, 128, True), (3406, 19, 315, 8, 2, 128, False), (775, 12, 500, 8, 8, 128, False), (672, 2, 640, 32, 32, 128, False),
    (1202, 6, 296, 64, 64, 64, False), (0, 2, 950, 32, 32, 128, True), (4096, 4, 1024, 64, 64, 64, True), (9000, 9, 1000, 16, 16, 256, False),
    (64, 64, 1, 32, 8, 128, False)])
def test_two_row_groups_a_wave_only_where_the_rows_fill_the_chip(total, B, longest, nh, nkv, D, two):
    """Attention behind prefixes: by the rows of the step, not by the longest portion as if all were as long."""
    from llmss_amd.ops import hip as H

    assert H.lib().attn_extend_two(total, B, longest, nh, nkv, D) == two


@pytest.mark.parametrize("M,N,K,code", [(12, 17472, 3488, 1024), (7, 2592, 4096, 1024), (2, 2272, 3696, 1024), (61, 18688, 4656, 15),
                                        (64, 22016, 4096, None), (40, 8192, 2048, None)])
def test_gated_products_of_few_rows_leave_the_older_kernels(M, N, K, code):
    """Pairs of columns and their split sums cost the older kernels more than plain products: the decode kernel (hint bit 1024) or tiles of
    96 columns (15) where those were the faster ones; None: whatever the model says, unsplit."""
    from llmss_amd.ops import hip as H

    nt, split = H.lib().gemm_plan(M, N, K, False, True, False)
    assert split == 1 and (code is None or (nt >> 8) & (1024 if code == 1024 else 15) == code), (hex(nt), split)


@pytest.mark.parametrize("mode,es", [(1, 2), (2, 4), (3, 2), (0, 2)])
def test_rows_of_expert_results_fit_the_descriptor_that_stores_them(mode, es):
    """A wave of the four-wave kernel stores over 240 rows of an expert tile (csrc/gemm_quad.hip quad_store), every other sixteen, through one
    descriptor of 31 bits: rows past its end would be dropped. Wider results than fit go to another kernel; mode 0: gate and up in two matrices."""
    from llmss_amd.ops import hip as H

    def takes(width):  # numbers of a result row
        if mode == 0:
            return H.lib().moe_pp_glu_ok(256, 3, 1, width, 256)
        return H.lib().moe_pp_quad(mode, 256, 3, 1, width * (2 if mode == 3 else 1), 256)

    last = (2 ** 31 - 1) // (240 * es) // 16 * 16
    assert takes(2048) and takes(last) and 240 * last * es < 2 ** 31
    for width in (last + 16, 2_300_000 * 4 // es, 2 ** 31 // (128 * es) - 16):
        assert 240 * width * es >= 2 ** 31 and not takes(width)


@pytest.mark.parametrize("nt,split", [(0x1300, 3), (0x1300, 1), ((3 | 32 | 1024) << 8, 2)])
def test_closing_products_keep_a_tuned_plan(nt, split):
    """The plan that a tuner or a plan file has set for a size stands, split or not, also where the op behind sums the slabs."""
    from llmss_amd.ops import hip as H

    M, N, K = 40, 1024, 4096
    static = tuple(H.lib().gemm_closing_plan(M, N, K))
    H.lib().gemm_tuned_set(M, N, K, False, 0, nt, split)
    try:
        assert tuple(H.lib().gemm_closing_plan(M, N, K)) == (nt, split) != static
    finally:
        H.lib().gemm_tuned_clear()
    assert tuple(H.lib().gemm_closing_plan(M, N, K)) == static


@pytest.mark.parametrize("sizes", [[(4800, 1600), (1600, 1600), (6400, 1600), (1600, 6400)], [(12288, 4096), (4096, 4096), (22016, 4096), (4096, 11008)],
                                   [(10240, 2048), (2048, 4096), (11264, 2048), (2048, 5632), (2048, 2048), (4352, 2048)]])
def test_prices_of_a_model_are_kept_at_every_number_of_rows(sizes):
    """A step plans every size several times, layer by layer: none may take another's place, whatever the number of rows."""
    from llmss_amd.ops import hip as H

    L = H.lib()

    def walk(M):
        for N, K in sizes:
            L.gemm_plan(M, N, K, False, False, False)
            L.gemm_plan(M, N, K, False, False, True)
            L.gemm_plan(M, N, K, False, True, False)

    for M in list(range(17, 1100)) + list(range(1101, 9000, 97)):
        walk(M)
        before = L.gemm_priced()
        walk(M)
        assert L.gemm_priced() == before, M
