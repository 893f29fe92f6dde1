"""Numerics of every gfx950 HIP kernel against the plain-PyTorch fp32 definitions
(``llmss_amd/ops/reference.py``). Also asserts the native extension is what actually runs."""
import math

import pytest
import torch

from llmss_amd.ops import hip as H
from llmss_amd.ops import reference as R

pytestmark = pytest.mark.gpu
dev = "cuda"
ODD_NT_TILES = (7,)  # gemm_mid 64x48: three 16-column tiles per wave (no SwiGLU epilogue)


def rnd(*s, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(*s, device=dev) * scale).to(dtype)


def close(a, b, atol, rtol=0.02):
    a, b = a.float(), b.float()
    err = (a - b).abs()
    tol = atol + rtol * b.abs()
    bad = ~(err <= tol)
    assert not bool(bad.any()), (f"max err {err.nan_to_num(float('inf')).max().item():.4g} (max |ref| "
                                 f"{b.abs().max().item():.3g}), {int(bad.sum())} bad, first at "
                                 f"{bad.nonzero()[0].tolist()}, rows {bad.nonzero()[:, 0].unique().tolist()[:16]}")


def test_native_loaded():
    lib = H.lib()
    import llmss_amd

    assert lib.__file__.startswith(llmss_amd.__path__[0])


@pytest.mark.parametrize("T,Hd", [(1, 64), (7, 1600), (33, 4096), (5, 8192)])
@pytest.mark.parametrize("rms", [False, True])
def test_add_norm(T, Hd, rms):
    torch.manual_seed(0)
    x, r = rnd(T, Hd), rnd(T, Hd)
    w, b = rnd(Hd, scale=0.5) + 1, (None if rms else rnd(Hd, scale=0.1))
    r_ref = r.clone()
    y, ro = H.add_norm(x, w, b, 1e-5, rms, residual=r)
    y_ref, ro_ref = R.add_norm(x, w, b, 1e-5, rms, r_ref)
    close(ro, ro_ref, 1e-2)
    close(y, y_ref, 3e-2)
    y2, _ = H.add_norm(x, w, b, 1e-5, rms)
    y2_ref, _ = R.add_norm(x, w, b, 1e-5, rms)
    close(y2, y2_ref, 3e-2)


@pytest.mark.parametrize("T,Hd,C", [(7, 1600, 2), (33, 4096, 4), (64, 4096, 8), (5, 5120, 5)])
@pytest.mark.parametrize("rms", [False, True])
def test_add_norm_column_chunked(T, Hd, C, rms):
    """add_norm reading the column-chunked [C, T, Hd / C] layout of the "col" decode schedule
    (DecoderLM._reduce_cols) equals the row-major call on the same values (bitwise: same loads, same order)."""
    torch.manual_seed(0)
    x, r = rnd(T, Hd), rnd(T, Hd)
    w, b = rnd(Hd, scale=0.5) + 1, (None if rms else rnd(Hd, scale=0.1))
    xc = x.view(T, C, Hd // C).permute(1, 0, 2).contiguous()
    r1, r2 = r.clone(), r.clone()
    y, ro = H.add_norm(x, w, b, 1e-5, rms, residual=r1)
    yc, roc = H.add_norm(xc, w, b, 1e-5, rms, residual=r2)
    assert torch.equal(y, yc) and torch.equal(ro, roc)
    y_ref, _ = R.add_norm(x, w, b, 1e-5, rms, r.clone())
    close(yc, y_ref, 3e-2)


def test_embed():
    torch.manual_seed(0)
    wte, wpe = rnd(1000, 256), rnd(64, 256)
    ids = torch.randint(0, 1000, (37,), device=dev)
    pos = torch.randint(0, 64, (37,), device=dev)
    close(H.embed(ids, wte), R.embed(ids, wte), 0)
    close(H.embed(ids, wte, pos, wpe), R.embed(ids, wte, pos, wpe), 1e-2)


@pytest.mark.parametrize("style,D,rot,nh,nkv", [("neox", 128, 128, 8, 2), ("gptj", 256, 64, 4, 4), ("neox", 64, 64, 4, 1)])
def test_rope_cache(style, D, rot, nh, nkv):
    torch.manual_seed(0)
    T, bs, nb = 19, 16, 8
    qkv = rnd(T, (nh + 2 * nkv) * D)
    pos = torch.randint(0, 100, (T,), device=dev)
    cos, sin = R.rope_tables(128, rot, 10000.0, dev)
    kc = torch.zeros(nb, nkv, bs, D, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    slots = torch.randperm(nb * bs, device=dev)[:T]
    slots[3] = -1
    q1, kc1, vc1 = qkv.clone(), kc.clone(), vc.clone()
    H.rope_cache(q1, pos, cos, sin, kc1, vc1, slots, nh, nkv, D, rot, style)
    q2, kc2, vc2 = qkv.clone(), kc.clone(), vc.clone()
    R.rope_cache(q2, pos, cos, sin, kc2, vc2, slots, nh, nkv, D, rot, style)
    close(q1, q2, 2e-2)
    close(kc1, kc2, 2e-2)
    close(vc1, vc2, 0)


@pytest.mark.parametrize("style,T", [("neox", 40), ("gptj", 7), ("neox", 300)])
def test_rope_cache_from_split_k_partials(style, T):
    """QKV GEMM leaves split-K slabs; the rope kernel sums them (+bias) - same result as the unfused path."""
    torch.manual_seed(0)
    D, nh, nkv, K, bs, nb = 128, 8, 2, 4096, 16, 32
    N = (nh + 2 * nkv) * D
    x, w, b = rnd(T, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    pos = torch.randint(0, 100, (T,), device=dev)
    cos, sin = R.rope_tables(128, D, 10000.0, dev)
    slots = torch.randperm(nb * bs, device=dev)[:T]
    p = H.linear(x, w, b, partial_ok=True)
    if T == 40:
        assert isinstance(p, H.PartialSum) and p.S > 1
    kc1, vc1 = [torch.zeros(nb, nkv, bs, D, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    q1 = H.rope_cache(p, pos, cos, sin, kc1, vc1, slots, nh, nkv, D, D, style)
    q2 = H.linear(x, w, b)
    kc2, vc2 = torch.zeros_like(kc1), torch.zeros_like(vc1)
    R.rope_cache(q2, pos, cos, sin, kc2, vc2, slots, nh, nkv, D, D, style)
    close(q1, q2, 2e-2)
    close(kc1, kc2, 2e-2)
    close(vc1, vc2, 2e-2)


@pytest.mark.parametrize("style,D,rot,nh,nkv,bias", [("neox", 128, 128, 8, 2, False), ("gptj", 256, 64, 4, 4, True),
                                                      ("none", 64, 0, 6, 6, True), ("neox", 64, 64, 8, 1, False)])
@pytest.mark.parametrize("tile", [1, 2, 3, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("T", [40, 300])
def test_qkv_gemm_rope_cache_epilogue(style, D, rot, nh, nkv, bias, tile, split, T):
    """QKV GEMM whose epilogue applies RoPE and writes the paged KV cache (one launch) == GEMM + rope_cache:
    q/k/v rows and every cache row, with a skipped slot (-1) and NaN-filled caches whose unwritten rows
    must stay untouched. Plans the epilogue cannot take (neox on tiles narrower than a head) return None."""
    torch.manual_seed(0)
    K, bs, nb = 512, 16, 40
    N = (nh + 2 * nkv) * D
    x, w = rnd(T, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1) if bias else None
    do_rope = style != "none"
    st = "gptj" if style == "gptj" else "neox"
    pos = torch.randint(0, 120, (T,), device=dev)
    cos, sin = R.rope_tables(128, rot if do_rope else 64, 10000.0, dev)
    slots = torch.randperm(nb * bs, device=dev)[:T]
    slots[5] = -1
    kc1 = torch.full((nb, nkv, bs, D), float("nan"), dtype=torch.bfloat16, device=dev)
    vc1 = torch.full_like(kc1, float("nan"))
    d = 16 if tile not in (1, 9) else 0
    hint = (tile | d) << 8
    y = H.linear_qkv(x, w, b, pos, cos, sin, kc1, vc1, slots, nh, nkv, D, rot, st, do_rope, nt_hint=hint,
                     split_hint=split)
    bn = {1: 128, 2: 128, 3: 64, 8: 128, 9: 128, 10: 256, 11: 128, 12: 256}[tile]
    if do_rope and st == "neox" and bn % D:
        assert y is None
        return
    assert y is not None
    q2 = H.linear(x, w, b)
    kc2, vc2 = torch.full_like(kc1, float("nan")), torch.full_like(vc1, float("nan"))
    R.rope_cache(q2, pos, cos, sin, kc2, vc2, slots, nh, nkv, D, rot, st, do_rope=do_rope)
    close(y, q2, 1e-2)
    for a, r in ((kc1, kc2), (vc1, vc2)):
        assert torch.equal(a.isnan(), r.isnan())
        close(a.nan_to_num(0), r.nan_to_num(0), 1e-2)


@pytest.mark.parametrize("version,waves", [(1, 0), (2, 0), (3, 4), (3, 8)])
@pytest.mark.parametrize("D,nh,nkv", [(64, 4, 4), (128, 8, 2), (128, 16, 1), (256, 4, 4), (128, 12, 4), (128, 16, 2),
                                      (64, 6, 3), (256, 8, 2)])
@pytest.mark.parametrize("lens", [(1, 70, 129, 5, 300), (1, 70, 129, 5, 300, 64, 17, 200)])
def test_attn_prefill(D, nh, nkv, version, waves, lens):
    """v1 (register-staged tiles), v2 (LDS-DMA two-slot ring, 2 row blocks per wave, GQA heads sharing a
    K/V tile) and v3 (v2 + light softmax, 4 or 8 waves per workgroup) against the fp32 oracle; qkv as a
    row-strided view, NaN-filled output. Eight sequences make the (sequence, head group) pairs a multiple
    of 8, i.e. the XCD-grouped block order of v2/v3; five do not (plain order)."""
    torch.manual_seed(0)
    lens = list(lens)
    T = sum(lens)
    W = (nh + 2 * nkv) * D
    qkv = rnd(T, W + 64)[:, :W]  # row stride > width (as a fused-QKV view would have)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev)
    sc = 1 / math.sqrt(D)
    H.lib().attn_prefill_set_version(version)
    H.lib().attn_prefill_set_waves(waves)
    try:
        out = torch.full((T, nh * D), float("nan"), dtype=torch.bfloat16, device=dev)
        H.attn_prefill(qkv, cu, max(lens), nh, nkv, D, sc, out=out)
    finally:
        H.lib().attn_prefill_set_version(3)
        H.lib().attn_prefill_set_waves(0)
    ref = R.attn_prefill(qkv.float(), cu.cpu(), nh, nkv, D, sc)
    close(out, ref, 2e-2)


@pytest.mark.parametrize("D,nh,nkv", [(64, 25, 25), (128, 32, 32), (128, 8, 1), (128, 64, 8), (256, 16, 16)])
@pytest.mark.parametrize("B,maxctx", [(1, 1000), (6, 300)])
def test_attn_decode(D, nh, nkv, B, maxctx):
    torch.manual_seed(0)
    bs = 16
    maxb = (maxctx + bs - 1) // bs
    nb = B * maxb + 3
    kc, vc = rnd(nb, nkv, bs, D), rnd(nb, nkv, bs, D)
    perm = torch.randperm(nb, device=dev)[: B * maxb].view(B, maxb).to(torch.int32)
    ctx = torch.randint(1, maxctx + 1, (B,), device=dev, dtype=torch.int32)
    ctx[0] = maxctx
    q = rnd(B, (nh + 2 * nkv) * D)
    sc = 1 / math.sqrt(D)
    out = H.attn_decode(q, kc, vc, perm, ctx, nh, nkv, D, sc, maxctx)
    ref = R.attn_decode(q.float(), kc.float(), vc.float(), perm, ctx, nh, nkv, D, sc)
    close(out, ref, 2e-2)
    out1 = H.attn_decode(q, kc, vc, perm, ctx, nh, nkv, D, sc, maxctx, splits=(1, maxb * bs))
    close(out1, ref, 2e-2)
    try:  # every token-loop variant (1 / 2 / 4 tokens per slot, single or double register set)
        for u in (1, 2, 4, 12, 14):
            H.lib().attn_decode_set_unroll(u)
            close(H.attn_decode(q, kc, vc, perm, ctx, nh, nkv, D, sc, maxctx), ref, 2e-2)
            close(H.attn_decode(q, kc, vc, perm, ctx, nh, nkv, D, sc, maxctx, splits=(1, maxb * bs)), ref, 2e-2)
    finally:
        H.lib().attn_decode_set_unroll(0)


@pytest.mark.parametrize("M", [1, 5, 16, 33, 64, 65, 200, 512])
@pytest.mark.parametrize("N,K", [(4800, 1600), (1376 * 2, 4096), (4096, 1376), (256, 64)])
def test_gemm(M, N, K):
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    ref = R.linear(x.float(), w.float(), b.float())
    close(H.linear(x, w, b), ref, 2e-2)
    close(H.linear(x, w, b, act="gelu_tanh"), R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    if N % 32 == 0:
        close(H.linear(x, w, None, glu=True), R.linear(x.float(), w.float(), None, glu=True), 2e-2)


@pytest.mark.parametrize("tile", [7, 8, 9, 10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("depth", [16, 32, 48])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("M,N,K", [(200, 1536, 4096), (512, 768, 1024), (130, 4800, 1600), (300, 1312, 64 * 5 + 16)])
def test_gemm_mid_interleaved_ring(tile, depth, split, M, N, K):
    """gemm_mid's interleaved ring (hint bit 512, csrc/gemm_mid.hip ILV: second-half fragment reads and the ring
    stage issue between the MFMAs, one mid-k-step barrier) against the fp32 oracle: every tile and ring depth,
    split-K, NaN-filled outputs, SwiGLU; a K with a partial last k-step takes the plain ring (fallback)."""
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    hint = (tile | depth | 512) << 8
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=split, out=y),
          R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    if tile not in ODD_NT_TILES and split == 1:
        y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=x.device)
        close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=split, out=y),
              R.linear(x.float(), w.float(), None, glu=True), 2e-2)
    if split > 1:  # split-K combined inside the launch (hint bit 256) behind the interleaved ring
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
        close(H.linear(x, w, b, nt_hint=hint | (256 << 8), split_hint=split, out=y),
              R.linear(x.float(), w.float(), b.float()), 2e-2)


@pytest.mark.parametrize("M,N,K", [(700, 1312, 64), (513, 768, 128), (300, 512, 192), (1024, 1536, 4096),
                                   (2100, 800, 1600), (257, 288, 256), (600, 544, 320), (1500, 2080, 704),
                                   (600, 1024, 1376), (300, 512, 80), (513, 768, 144), (257, 288, 48)])
def test_gemm_big_edges(M, N, K):
    """The 256x256 ping-pong prefill kernel (gemm.hip gemm_pp_kernel) against the fp32 oracle at K-tile counts
    1-5 and 11 (prologue / last-tile vmcnt edges of its 4-phase, 2-buffer schedule, and the slot reuse of the
    steady state), partial last K-tiles (K % 64 = 16-48: Llama-2-7B's TP=8 down projection has K = 1376; the
    chunks past K read a zero page), ragged M / N, bias + activation and SwiGLU through the swizzled LDS
    epilogue."""
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=4 << 8, split_hint=1, out=y),
          R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=x.device)
    close(H.linear(x, w, None, glu=True, nt_hint=4 << 8, split_hint=1, out=y),
          R.linear(x.float(), w.float(), None, glu=True), 2e-2)


# 128x128, 64x128, 64x64, 256x256, 256x128 / 256x64 (8 waves); gemm_mid (buffer-descriptor staging):
# 8 = 128x128, 9 = 256x128, 10 = 64x256, 11 = 64x128, 12 = 128x256, 13 = 64x192, 14 = 64x32, 15 = 64x96, 7 = 64x48
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("stages", [2, 3, 4, 6])
@pytest.mark.parametrize("split", [1, 3, 8])
@pytest.mark.parametrize("M,N,K", [(64, 1536, 4096), (200, 4800, 1600), (37, 256, 64 * 5 + 16), (700, 1312, 192)])
def test_gemm_tiled_variants(tile, stages, split, M, N, K):
    if tile == 4 and (stages != 2 or split > 1):
        pytest.skip("the 256x256 kernel has one pipeline and no split-K")
    if tile in (5, 6) and stages == 6:
        pytest.skip("8-wave tiles ring at most 3 (256x128) / 4 (256x64) stages (clamped)")
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    hint = (tile | ({2: 0, 3: 16, 4: 32, 6: 48}[stages])) << 8
    ref = R.linear(x.float(), w.float(), b.float(), act="gelu_tanh")
    # NaN-filled outputs: an element the kernel fails to write cannot pass on a recycled buffer
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=split, out=y), ref, 2e-2)
    y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=x.device)
    if tile in ODD_NT_TILES and split == 1:  # an in-kernel SwiGLU pairs 16-column tiles in a wave: refused
        with pytest.raises(RuntimeError):
            H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=split, out=y)
        return
    # (split plans apply SwiGLU in the reduce launch, so every tile takes them)
    close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=split, out=y),
          R.linear(x.float(), w.float(), None, glu=True), 2e-2)


@pytest.mark.parametrize("tile", [1, 2, 3, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("split", [2, 3, 8])
@pytest.mark.parametrize("M,N,K", [(64, 1536, 4096), (200, 4800, 1600), (37, 256, 64 * 5 + 16), (512, 2752, 4096)])
def test_gemm_splitk_combine_in_launch(tile, split, M, N, K):
    """Hint bit 256: the K slices of a tile combine inside the launch (last arriver per tile sums the
    write-through slabs in slice order and runs the epilogue). Bit-identical to the same plan with a
    separate reduce launch; repeated calls check the self-resetting tile counters; NaN-filled outputs
    and a NaN-poisoned workspace check that every element is written from fresh slabs."""
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    d = 16 if tile not in (5, 9) else 0
    hint, comb = (tile | d) << 8, (tile | d | 256) << 8
    H._GEMM_WS.get(64 << 20, x.device).fill_(float("nan"))
    for act, glu, bias in (("gelu_tanh", False, b), ("none", True, None), ("none", False, b)):
        if glu and tile in ODD_NT_TILES:
            continue
        nout = N // 2 if glu else N
        ref = H.linear(x, w, bias, act=act, glu=glu, nt_hint=hint, split_hint=split)
        for _ in range(3):
            y = torch.full((M, nout), float("nan"), dtype=torch.bfloat16, device=dev)
            got = H.linear(x, w, bias, act=act, glu=glu, nt_hint=comb, split_hint=split, out=y)
            if act == "none":  # the same fp32 sums in the same order
                assert torch.equal(got, ref), (act, glu, (got.float() - ref.float()).abs().max().item())
            else:  # GELU compiled into two kernels may contract differently: at most 1 bf16 ulp
                close(got, ref, 0, rtol=1e-2)
        close(got, R.linear(x.float(), w.float(), None if bias is None else bias.float(), act=act, glu=glu), 2e-2)
    # a consumer that could take slabs gets the finished output instead
    p = H.linear(x, w, None, nt_hint=comb, split_hint=split, partial_ok=True)
    assert not isinstance(p, H.PartialSum)
    close(p, R.linear(x.float(), w.float(), None), 2e-2)


@pytest.mark.parametrize("tile", [8, 11, 12])
def test_gemm_mid_k_tail_reads_nothing_past_the_operands(tile):
    """Operands as views at the front of NaN-filled buffers: the partial last k-step of the last rows
    must not pick up the NaNs that follow (0 * NaN would poison the row)."""
    torch.manual_seed(0)
    M, N, K = 130, 384, 64 * 3 + 16
    xb = torch.full((M * K + 4096,), float("nan"), dtype=torch.bfloat16, device=dev)
    wb = torch.full((N * K + 4096,), float("nan"), dtype=torch.bfloat16, device=dev)
    x, w = xb[: M * K].view(M, K), wb[: N * K].view(N, K)
    x.copy_(rnd(M, K))
    w.copy_(rnd(N, K, scale=K ** -0.5))
    for split in (1, 2):
        y = H.linear(x, w, None, nt_hint=(tile | 16) << 8, split_hint=split)
        close(y, R.linear(x.float(), w.float(), None), 2e-2)


@pytest.mark.parametrize("M,N,K,glu,act", [(1773, 12288, 256, False, "none"), (1773, 22016, 1024, True, "none"), (8261, 2048, 512, False, "gelu_tanh"),
                                           (8193, 2048, 1024, False, "relu"), (8261, 6400, 1024, False, "none"), (8261, 2048, 1024, True, "none"),
                                           (8256, 2056, 2048, False, "none"), (964, 16576, 2112, True, "none"), (3558, 9344, 3008, False, "none")])
def test_products_cut_in_two_launches(M, N, K, glu, act):
    """Products of 256 x 256 tiles whose last wave is nearly empty: whole waves and what is left over, by rows or columns, with bias
    and activation on either side, into strided rows; what lies around the output stays as it is."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K + 8)[:, :K], rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    n = N // 2 if glu else N
    wide = torch.full((M + 2, n + 16), 7.0, dtype=torch.bfloat16, device=dev)
    y = wide[1:M + 1, 8:n + 8]
    H.linear(x, w, b, act=act, glu=glu, out=y)
    ref = R.linear(x.float(), w.float(), b.float(), act=act, glu=glu)
    assert any(H.lib().gemm_cut(M, N, K, glu))
    close(y, ref, 2e-2)
    wide[1:M + 1, 8:n + 8] = 7.0
    assert (wide == 7.0).all()


@pytest.mark.parametrize("M,N,K,glu,act,bias", [(8261, 2048, 2048, False, "gelu", True), (1240, 13248, 3392, False, "none", True),
                                                (803, 16512, 3200, True, "none", True), (8261, 2048, 4096, False, "none", False)])
def test_rest_of_a_cut_product_splits_k(M, N, K, glu, act, bias):
    """The rest of a product that is cut in two launches, with few tiles: the second launch's K split, its 32-bit sums combined there, bias,
    activation and gate after their sum; strided rows, what lies around them stays. Each side's error is a rounding of the result in bf16 and of 32-bit sums."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K + 8)[:, :K], rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1) if bias else None
    n = N // 2 if glu else N
    wide = torch.full((M + 2, n + 16), 7.0, dtype=torch.bfloat16, device=dev)
    y = wide[1:M + 1, 8:n + 8]
    assert any(H.lib().gemm_cut(M, N, K, glu)) and H.lib().gemm_cut_split(M, N, K, glu) > 1
    H.linear(x, w, b, act=act, glu=glu, out=y)
    close(y, R.linear(x.float(), w.float(), b.float() if bias else None, act=act, glu=glu), 2e-2)
    wide[1:M + 1, 8:n + 8] = 7.0
    assert (wide == 7.0).all()


@pytest.mark.parametrize("M,N,K,tile", [(33, 256, 1040, False), (64, 2048, 2048, False), (17, 4096, 11008, False), (32, 2816, 12800, False),
                                        (64, 4096, 11008, True), (64, 4096, 11024, True), (59, 6704, 4320, True), (64, 8192, 1040, True)])
def test_slabs_of_few_rows(M, N, K, tile):
    """Products of 17 - 64 rows whose closing op sums the slabs: the planned kernel (column tiles of the decode kernel, or 64 x 64 tiles), odd
    k-steps, against the sums in 32 bits and the norm of their sum with the residual; a rounding of the result in bf16 each."""
    torch.manual_seed(0)
    x, w, r = rnd(M, K + 8)[:, :K], rnd(N, K, scale=K ** -0.5), rnd(M, N)
    g = (1 + 0.1 * torch.randn(N, device=dev)).to(torch.bfloat16)
    nt, split = H.lib().gemm_plan(M, N, K, False, False, True)
    assert split > 1 and bool((nt >> 8) & 1024) != tile
    p = H.linear(x, w, partial_ok=True)
    assert isinstance(p, H.PartialSum) and p.S == split
    total = x.float() @ w.float().t() + r.float()
    y, res = H.add_norm(p, g, None, 1e-5, True, r.clone())
    close(res, total, 2e-2)
    close(y, total * torch.rsqrt(total.pow(2).mean(-1, keepdim=True) + 1e-5) * g.float(), 3e-2)


DEC_BN = {1: 16, 2: 32, 3: 48, 4: 64, 5: 96}  # csrc/gemm_dec.hip tile codes (hint bit 1024 of the tile bits)


@pytest.mark.parametrize("code", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("depth", [0, 16, 32])
@pytest.mark.parametrize("split", [1, 3, 8])
@pytest.mark.parametrize("M,N,K", [(64, 4800, 1600), (1, 1600, 6400), (17, 2752, 4096), (33, 4096, 1376),
                                   (64, 200, 64 * 5 + 16), (5, 96, 16), (48, 1600, 1600)])
def test_gemm_dec(code, depth, split, M, N, K):
    """The K-split-wave decode GEMM (csrc/gemm_dec.hip) against the fp32 oracle: every column width and ring depth,
    M = 1..64 (16 / 32 / 64-row variants), ragged N, partial last k-steps (K % 64 = 16, 32) including a
    single-k-step K, grid splits whose slices leave some waves without k-steps, NaN-filled outputs; bias + GELU,
    SwiGLU and the fp32 split-K slabs a consumer sums (partial_ok)."""
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    hint = (code | depth | 1024) << 8
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=split, out=y),
          R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    if N % 32 == 0 and (DEC_BN[code] % 32 == 0 or min(split, -(-K // 64)) > 1):  # SwiGLU in-kernel or in the reduce
        y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=x.device)
        close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=split, out=y),
              R.linear(x.float(), w.float(), None, glu=True), 2e-2)
    H._GEMM_WS.get(64 << 20, x.device).fill_(float("nan"))
    p = H.linear(x, w, b, nt_hint=hint, split_hint=split, partial_ok=True)
    ref = R.linear(x.float(), w.float(), b.float())
    if isinstance(p, H.PartialSum):
        assert split > 1 and p.S == min(split, -(-K // 64))
        got = p.buf[:p.S * M * N].view(p.S, M, N).sum(0) + b.float()
        close(got, ref, 2e-2)
    else:
        assert split == 1 or -(-K // 64) == 1
        close(p, ref, 2e-2)


@pytest.mark.parametrize("code", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("split", [2, 3, 5])
@pytest.mark.parametrize("M,N,K", [(64, 6400, 1600), (7, 4800, 1600), (33, 2752, 4096), (64, 200, 64 * 5 + 16)])
def test_gemm_dec_combine_in_launch(code, split, M, N, K):
    """The decode GEMM's split-K combined in the launch (hint bit 256): the tile's last K slice sums every slice's
    write-through slab in slice order and runs the epilogue. Bit-identical to the same plan's slabs summed by the
    separate reduce launch (activation-free), across repeated calls (self-resetting tile counters), with NaN-filled
    outputs and a NaN-poisoned workspace; GELU and SwiGLU against the fp32 oracle."""
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    hint, comb = (code | 16 | 1024) << 8, (code | 16 | 1024 | 256) << 8
    H._GEMM_WS.get(64 << 20, x.device).fill_(float("nan"))
    ref = H.linear(x, w, b, nt_hint=hint, split_hint=split)  # slabs + splitk_reduce
    for _ in range(3):
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        got = H.linear(x, w, b, nt_hint=comb, split_hint=split, out=y)
        assert torch.equal(got, ref), (got.float() - ref.float()).abs().max().item()
    close(got, R.linear(x.float(), w.float(), b.float()), 2e-2)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=comb, split_hint=split, out=y),
          R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    if N % 32 == 0 and DEC_BN[code] % 32 == 0:
        y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=dev)
        close(H.linear(x, w, None, glu=True, nt_hint=comb, split_hint=split, out=y),
              R.linear(x.float(), w.float(), None, glu=True), 2e-2)
    p = H.linear(x, w, None, nt_hint=comb, split_hint=split, partial_ok=True)  # finished, not slabs
    assert not isinstance(p, H.PartialSum)


@pytest.mark.parametrize("code", [2, 4])
def test_gemm_dec_k_tail_reads_nothing_past_the_operands(code):
    """As test_gemm_mid_k_tail_...: operands at the front of NaN-filled buffers, a partial last k-step."""
    torch.manual_seed(0)
    M, N, K = 64, 384, 64 * 3 + 16
    xb = torch.full((M * K + 4096,), float("nan"), dtype=torch.bfloat16, device=dev)
    wb = torch.full((N * K + 4096,), float("nan"), dtype=torch.bfloat16, device=dev)
    x, w = xb[: M * K].view(M, K), wb[: N * K].view(N, K)
    x.copy_(rnd(M, K))
    w.copy_(rnd(N, K, scale=K ** -0.5))
    for split in (1, 2):
        y = H.linear(x, w, None, nt_hint=(code | 16 | 1024) << 8, split_hint=split)
        close(y, R.linear(x.float(), w.float(), None), 2e-2)


@pytest.mark.parametrize("code,M,N,K,split", [(1, 1, 96, 16, 1), (1, 16, 200, 128 * 5, 2), (2, 5, 1376, 1600, 3), (2, 17, 4096, 1376, 1),
                                              (3, 32, 200, 128 * 9 + 112, 4), (4, 23, 2752, 4096, 1), (4, 32, 640, 128 * 3 + 16, 2)])
def test_gemm_dec_fp8(code, M, N, K, split):
    """The decode GEMM over e4m3 weights against the dequantised product in fp32: 16 / 32-row variants, ragged N, partial last
    k-steps, slices without k-steps, strided rows of x; GELU, SwiGLU and slabs. Weights are exact in bf16, so what
    is off is the order of fp32 sums and the output's rounding (2^-9). A NaN weight stays in its own column: the bytes
    past a row's end are the next row's."""
    torch.manual_seed(0)
    x = rnd(M, K + 24)[:, :K]
    q, sc = H.quant_fp8_rows(rnd(N, K, scale=K ** -0.5))
    w = q.view(torch.float8_e4m3fn).float() * sc[:, None]
    b = rnd(N, scale=0.1)
    hint, bn = (code | 32 | 1024) << 8, DEC_BN[code]
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    close(H.linear(x, q, b, act="gelu_tanh", w_scale=sc, nt_hint=hint, split_hint=split, out=y),
          R.linear(x.float(), w, b.float(), act="gelu_tanh"), 2e-2)
    if N % 32 == 0 and (bn % 32 == 0 or min(split, -(-K // 64)) > 1):
        close(H.linear(x, q, None, glu=True, w_scale=sc, nt_hint=hint, split_hint=split), R.linear(x.float(), w, None, glu=True), 2e-2)
    H._GEMM_WS.get(64 << 20, x.device).fill_(float("nan"))
    p = H.linear(x, q, b, w_scale=sc, nt_hint=hint, split_hint=split, partial_ok=True)
    if isinstance(p, H.PartialSum):
        p = p.buf[:p.S * M * N].view(p.S, M, N).sum(0) + b.float()
    close(p, R.linear(x.float(), w, b.float()), 2e-2)
    q[1::2, 0] = 0x7F
    y = H.linear(x, q, None, w_scale=sc, nt_hint=hint, split_hint=split)
    assert torch.isfinite(y[:, 0::2]).all() and torch.isnan(y[:, 1::2]).all()


@pytest.mark.parametrize("M,N,K,glu", [(1, 4096, 4096, False), (16, 12288, 4096, False), (23, 22016, 4096, True), (32, 4096, 11008, False),
                                       (33, 4096, 4096, False), (3, 1856, 12240, True), (2, 53344, 256, False), (9, 328, 528, False)])
def test_fp8_products_of_few_rows_by_any_plan(M, N, K, glu):
    """What the plan of an fp8 product chooses on both sides of its lines, against the dequantised product."""
    torch.manual_seed(0)
    x = rnd(M, K)
    q, sc = H.quant_fp8_rows(rnd(N, K, scale=K ** -0.5))
    ref = R.linear(x.float(), q.view(torch.float8_e4m3fn).float() * sc[:, None], None, glu=glu)
    close(H.linear(x, q, None, glu=glu, w_scale=sc), ref, 2e-2)
    if not glu:
        p = H.linear(x, q, None, w_scale=sc, partial_ok=True)
        close(p.buf[:p.S * M * N].view(p.S, M, N).sum(0) if isinstance(p, H.PartialSum) else p, ref, 2e-2)


@pytest.mark.parametrize("code", [1, 2, 4, 5])
@pytest.mark.parametrize("split", [1, 2, 3])
@pytest.mark.parametrize("style,D,rot,nh,nkv", [("none", 64, 0, 25, 25), ("gptj", 256, 64, 4, 4), ("neox", 64, 64, 8, 1)])
def test_gemm_dec_qkv_epilogue(code, split, style, D, rot, nh, nkv):
    """The decode GEMM with the QKV RoPE / paged-KV-write epilogue (GPT-2-XL's unrotated heads, GPT-J's interleaved
    partial rotation) == GEMM + rope_cache, unsplit or split and combined in the launch; neox RoPE on a tile narrower
    than a head is refused."""
    torch.manual_seed(0)
    T, K, bs, nb = 64, 512, 16, 40
    N = (nh + 2 * nkv) * D
    x, w = rnd(T, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    do_rope = style != "none"
    st = "gptj" if style == "gptj" else "neox"
    pos = torch.randint(0, 120, (T,), device=dev)
    cos, sin = R.rope_tables(128, rot if do_rope else 64, 10000.0, dev)
    slots = torch.randperm(nb * bs, device=dev)[:T]
    slots[5] = -1
    kc1 = torch.full((nb, nkv, bs, D), float("nan"), dtype=torch.bfloat16, device=dev)
    vc1 = torch.full_like(kc1, float("nan"))
    hint = (code | 16 | 1024) << 8
    y = H.linear_qkv(x, w, b, pos, cos, sin, kc1, vc1, slots, nh, nkv, D, rot, st, do_rope, nt_hint=hint,
                     split_hint=split)
    if do_rope and st == "neox" and DEC_BN[code] % D:
        assert y is None
        return
    assert y is not None
    q2 = H.linear(x, w, b)
    kc2, vc2 = torch.full_like(kc1, float("nan")), torch.full_like(vc1, float("nan"))
    R.rope_cache(q2, pos, cos, sin, kc2, vc2, slots, nh, nkv, D, rot, st, do_rope=do_rope)
    close(y, q2, 1e-2)
    for a, r in ((kc1, kc2), (vc1, vc2)):
        assert torch.equal(a.isnan(), r.isnan())
        close(a.nan_to_num(0), r.nan_to_num(0), 1e-2)


@pytest.mark.parametrize("M", [1, 8, 64, 100])
def test_gemm_fp8(M):
    torch.manual_seed(0)
    N, K = 1024, 2048
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    q, s = H.quant_fp8_rows(w)
    q_ref, s_ref = R.quant_fp8_rows(w)
    close(s, s_ref, 1e-6)
    a, b = q.cpu().view(torch.float8_e4m3fn).float(), q_ref.cpu().view(torch.float8_e4m3fn).float()
    assert ((a - b).abs() <= 0.125 * b.abs() + 2 ** -9).all()  # at most one e4m3 ulp of rounding difference
    ref = R.linear(x.float(), q, None, w_scale=s)
    close(H.linear(x, q, None, w_scale=s), ref, 2e-2)
    xb = rnd(300, K)  # prefill size: W8A8 on the MX-fp8 MFMA (per-token fp8 activations)
    xq, xs = H.quant_fp8_rows(xb)
    close(H.linear(xb, q, None, w_scale=s), R.linear(R.dequant_fp8(xq, xs), q, None, w_scale=s), 3e-2)
    wd = H.dequant_fp8_rows(q, s)
    close(wd, R.dequant_fp8(q, s), 1e-6, rtol=1e-2)


def test_sample_greedy_and_filters():
    torch.manual_seed(0)
    B, V = 8, 50257
    logits = rnd(B, V + 15, scale=3.0)
    temp = torch.zeros(B, device=dev)
    topk = torch.zeros(B, dtype=torch.int32, device=dev)
    topp = torch.ones(B, device=dev)
    seeds = torch.arange(B, dtype=torch.int64, device=dev)
    out = H.sample(logits, temp, topk, topp, seeds, vocab=V)
    assert torch.equal(out, logits[:, :V].float().argmax(-1))
    # top-k = 3: samples must lie in the top-3 set
    temp.fill_(1.0)
    topk.fill_(3)
    top3 = logits[:, :V].float().topk(3, -1).indices
    for s in range(20):
        seeds.fill_(s * 7919)
        o = H.sample(logits, temp, topk, topp, seeds + torch.arange(B, device=dev), vocab=V)
        assert bool((top3 == o[:, None]).any(-1).all())
    # top-p tiny -> argmax
    topk.fill_(0)
    topp.fill_(1e-6)
    o = H.sample(logits, temp, topk, topp, seeds, vocab=V)
    lf = logits[:, :V].float()
    assert torch.equal(lf.gather(1, o[:, None])[:, 0], lf.max(-1).values)  # a max-logit token (bf16 ties)


def test_sample_distribution():
    torch.manual_seed(0)
    V = 8
    base = torch.tensor([[2.0, 1.0, 0.5, 0.0, -1.0, -2.0, -3.0, 0.2]], device=dev)
    logits = base.repeat(4096, 1).to(torch.bfloat16)
    temp = torch.full((4096,), 0.7, device=dev)
    topk = torch.zeros(4096, dtype=torch.int32, device=dev)
    topp = torch.ones(4096, device=dev)
    seeds = torch.arange(4096, dtype=torch.int64, device=dev) * 1000003
    o = H.sample(logits, temp, topk, topp, seeds)
    freq = torch.bincount(o, minlength=V).float() / 4096
    p = torch.softmax(logits[0].float() / 0.7, -1)
    assert (freq - p).abs().max() < 0.03, (freq, p)


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (64, 4096, 11008), (100, 1600, 6400)])
@pytest.mark.parametrize("rms", [True, False])
def test_splitk_partials_fused_into_add_norm(M, N, K, rms):
    torch.manual_seed(0)
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    b = rnd(N, scale=0.1)
    res = rnd(M, N)
    nw, nb = rnd(N, scale=0.2) + 1, (None if rms else rnd(N, scale=0.1))
    y_ref = H.linear(x, w, b)
    out_ref, r_ref = H.add_norm(y_ref, nw, nb, 1e-5, rms, residual=res.clone())
    p = H.linear(x, w, b, partial_ok=True)
    r2 = res.clone()
    out, r_out = H.add_norm(p, nw, nb, 1e-5, rms, residual=r2)
    close(r_out, r_ref, 2e-2)
    close(out, out_ref, 3e-2)


@pytest.mark.parametrize("S", [3, 5, 6, 9, 11, 12])
@pytest.mark.parametrize("rms", [True, False])
def test_split_slab_sums_at_any_split_count(S, rms):
    """Split counts without a compile-time add_norm variant (2 / 4 / 8 have one) sum their slabs in load groups
    (csrc/norm.hip PS = -1, csrc/gemm.hip slab_sum): GPT-2-XL's o / down plans leave 5 slabs. add_norm over the
    slabs and the split-K reduce (activation / SwiGLU epilogues) vs fp32."""
    torch.manual_seed(S)
    M, N, K = 64, 1600, 6400
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    res = rnd(M, N)
    nw, nb = rnd(N, scale=0.2) + 1, (None if rms else rnd(N, scale=0.1))
    hint = (14 | 32) << 8  # gemm_mid 64x32, 4 stages
    p = H.linear(x, w, b, nt_hint=hint, split_hint=S, partial_ok=True)
    assert isinstance(p, H.PartialSum) and p.S == S
    y32 = R.linear(x.float(), w.float(), b.float())
    out, r_out = H.add_norm(p, nw, nb, 1e-5, rms, residual=res.clone())
    r_ref = (y32.to(torch.bfloat16).float() + res.float()).to(torch.bfloat16)
    close(r_out, r_ref, 2e-2)
    out_ref, _ = R.add_norm(r_ref, nw, nb, 1e-5, rms)
    close(out, out_ref, 3e-2)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=S), R.linear(x.float(), w.float(), b.float(),
                                                                                 act="gelu_tanh"), 2e-2)
    close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=S), R.linear(x.float(), w.float(), None, glu=True),
          2e-2)


@pytest.mark.parametrize("V", [32000, 50257, 1000])
def test_sample_topk_topp_sets(V):
    """Every sampled token must lie in the reference top-k -> top-p kept set."""
    torch.manual_seed(1)
    B = 16
    logits = rnd(B, V, scale=2.0)
    temp = torch.full((B,), 0.8, device=dev)
    topk = torch.tensor([0, 1, 5, 50, 0, 50, 100, 0] * 2, dtype=torch.int32, device=dev)
    topp = torch.tensor([0.9, 1.0, 1.0, 0.95, 0.5, 0.8, 1.0, 1.0] * 2, device=dev)
    allowed = []
    for b in range(B):
        x = logits[b].float() / 0.8
        keep = torch.ones(V, dtype=torch.bool, device=dev)
        k = int(topk[b])
        if 0 < k < V:
            keep &= x >= torch.topk(x, k).values[-1]
        if float(topp[b]) < 1.0:
            pr = torch.softmax(x.masked_fill(~keep, float("-inf")), -1)
            sp, _ = pr.sort(descending=True)
            cum = sp.cumsum(0)
            n = int((cum - sp < float(topp[b])).sum())
            keep &= pr >= sp[n - 1] * (1 - 1e-5)
        allowed.append(keep)
    for s in range(25):
        seeds = torch.arange(B, dtype=torch.int64, device=dev) * 7777 + s
        o = H.sample(logits, temp, topk, topp, seeds)
        for b in range(B):
            assert allowed[b][o[b]], (b, int(o[b]), int(topk[b]), float(topp[b]))


def test_autotune_installs_plan():
    from llmss_amd import _native
    from llmss_amd.ops.autotune import GemmShape, tune_shape

    lib = _native()
    torch.manual_seed(0)
    M, N, K = 48, 1536, 1024
    nt, s, t, t_default = tune_shape(M, GemmShape(N, K), dev, weight_budget=64 << 20, iters=2,
                                     cands=[(0x300, 2), (0x1200, 1), (3 + 32, 4)])
    assert t <= t_default and (nt == 0 or nt in (0x300, 0x1200, 35))
    try:
        lib.gemm_tuned_set(M, N, K, False, 0, 0x1300, 4)
        assert lib.gemm_tuned_get(M, N, K, False, 0) == (0x1300, 4)
        assert lib.gemm_plan(M, N, K, False)[1] == 4
        x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
        close(H.linear(x, w), R.linear(x.float(), w.float()), 2e-2)
        p = H.linear(x, w, partial_ok=True)
        assert isinstance(p, H.PartialSum) and p.S == 4
    finally:
        lib.gemm_tuned_clear()


def _kept_sets(logits, temp, k, p):
    """Exact kept token sets (reference semantics: temperature -> top-k (ties kept) -> top-p)."""
    out = []
    for row in logits.float().cpu():
        x = row.double() / temp
        if 0 < k < x.numel():
            x = x.masked_fill(x < torch.topk(x, k).values[-1], float("-inf"))
        if p < 1.0:
            pr = torch.softmax(x, -1)
            sp, _ = pr.sort(descending=True)
            keep = (sp.cumsum(0) - sp) < p * sp.sum()
            thr = sp[keep].min()
            x = x.masked_fill(pr < thr, float("-inf"))
        out.append(set(torch.nonzero(x > float("-inf")).flatten().tolist()))
    return out


@pytest.mark.parametrize("V", [32000, 50257, 1000])
@pytest.mark.parametrize("k,p,temp", [(50, 1.0, 1.0), (0, 0.6, 0.8), (40, 0.9, 1.0), (7, 0.3, 1.3)])
def test_sample_kept_set_exact(V, k, p, temp):
    torch.manual_seed(V + k)
    B = 6
    logits = rnd(B, V, scale=2.5)
    sets = _kept_sets(logits, temp, k, p)
    tt = torch.full((B,), temp, device=dev)
    tk = torch.full((B,), k, dtype=torch.int32, device=dev)
    tp = torch.full((B,), p, device=dev)
    seen = [set() for _ in range(B)]
    for s in range(64):
        seeds = torch.arange(B, dtype=torch.int64, device=dev) * 7919 + s * 104729
        o = H.sample(logits, tt, tk, tp, seeds).tolist()
        o2 = H.sample(logits, tt, tk, tp, seeds).tolist()
        assert o == o2  # deterministic for identical inputs (TP ranks rely on it)
        for b in range(B):
            assert o[b] in sets[b], (b, o[b], len(sets[b]))
            seen[b].add(o[b])
    for b in range(B):
        if len(sets[b]) <= 3:
            assert seen[b] == sets[b]


@pytest.mark.parametrize("V", [32000, 50304, 1000])
@pytest.mark.parametrize("k,p,scale", [(0, 0.95, 0.3), (0, 0.5, 0.5), (2000, 0.9, 0.3), (40, 0.95, 0.05)])
def test_sample_flat_rows(V, k, p, scale):
    """Near-flat logits put hundreds of tokens into the boundary bin of the top-p / top-k selection (the
    sorted-candidate path of sample_v3_kernel): every draw in the exact kept set, identical on a repeat. Scales are
    chosen so the boundary bin holds at most SV3_MAXC = 2048 tokens; beyond that the kernel keeps the whole bin by
    design (a superset of the exact set)."""
    torch.manual_seed(V + k)
    B = 4
    logits = rnd(B, V, scale=scale)
    sets = _kept_sets(logits, 1.0, k, p)
    tt = torch.ones(B, device=dev)
    tk = torch.full((B,), k, dtype=torch.int32, device=dev)
    tp = torch.full((B,), p, device=dev)
    for s in range(16):
        seeds = torch.arange(B, dtype=torch.int64, device=dev) * 7919 + s * 104729
        o = H.sample(logits, tt, tk, tp, seeds).tolist()
        assert o == H.sample(logits, tt, tk, tp, seeds).tolist()
        for b in range(B):
            assert o[b] in sets[b], (b, o[b], len(sets[b]))


@pytest.mark.parametrize("tile,stages", [(1, 2), (1, 3), (2, 2), (2, 4), (3, 3), (3, 4)])
@pytest.mark.parametrize("per_cu", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(512, 1536, 4096), (300, 2752, 1376), (64, 4096, 11008), (130, 544, 208)])
def test_gemm_streamk(tile, stages, per_cu, M, N, K):
    """Stream-K tiled GEMM: tiles split across workgroups, combined in-kernel by the last arriver."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    hint = (tile | {2: 0, 3: 16, 4: 32}[stages] | 128) << 8
    for _ in range(2):  # second launch reuses the self-reset arrival counters
        close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=per_cu),
              R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=per_cu),
          R.linear(x.float(), w.float(), None, glu=True), 2e-2)


@pytest.mark.parametrize("tile,stages", [(3, 2), (3, 3), (3, 4), (2, 2), (2, 3), (1, 2)])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("M,N,K", [(64, 1024, 2048), (37, 544, 2064), (128, 4096, 1376)])
def test_gemm_fp8_tiled(tile, stages, split, M, N, K):
    """W8A16 tiled GEMM: fp8 weight tiles staged in LDS, expanded to bf16 fragments, scale in the epilogue."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    q, s = H.quant_fp8_rows(w)
    hint = (tile | {2: 0, 3: 16, 4: 32}[stages]) << 8
    close(H.linear(x, q, b, act="gelu_tanh", w_scale=s, nt_hint=hint, split_hint=split),
          R.linear(x.float(), q, b.float(), act="gelu_tanh", w_scale=s), 2e-2)
    close(H.linear(x, q, None, glu=True, w_scale=s, nt_hint=hint, split_hint=split),
          R.linear(x.float(), q, None, glu=True, w_scale=s), 2e-2)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,hint,split", [(256, 0x21, 4), (512, 0x12, 2), (200, (1 | 16 | 128) << 8, 2),
                                          (96, (3 | 128) << 8, 3), (64, 0x300, 4), (64, 0x1300, 1),
                                          (512, (5 | 16) << 8, 8), (300, (6 | 32) << 8, 12),
                                          (256, (5 | 128) << 8, 4)])
def test_partial_capable_calls_never_lose_output(fp8, M, hint, split):
    """partial_ok=True must return split-K slabs only when the kernel leaves them (stream-K and fp8
    prefill panels finish their output in place): regression for a null-output fault."""
    torch.manual_seed(0)
    N, K = 1280, 2048
    x, w = rnd(M, K), rnd(N, K, scale=K ** -0.5)
    sc = None
    if fp8:
        w, sc = H.quant_fp8_rows(w)
    ref = R.linear(x.float(), w if fp8 else w.float(), None, w_scale=sc)
    r = H.linear(x, w, None, w_scale=sc, nt_hint=hint, split_hint=split, partial_ok=True)
    if isinstance(r, H.PartialSum):
        r = r.buf[: r.S * M * N].view(r.S, M, N).sum(0)
    close(r, ref, 2e-2)


@pytest.mark.parametrize("tile,depth", [(1, 3), (1, 2), (2, 4), (2, 3), (3, 4), (3, 2), (4, 0)])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("M,N,K", [(256, 1280, 2048), (300, 544, 2064), (129, 4096, 1376), (700, 800, 1024)])
def test_gemm_w8a8_mx_fp8(tile, depth, split, M, N, K):
    """W8A8 on the MX-fp8 MFMA: exact vs fp32 math on the same fp8 operands (per-token x, per-row w)."""
    if tile == 4 and (K % 128 or split > 1):
        pytest.skip("the 256x256 fp8 tile needs K % 128 == 0 and has no split-K")
    torch.manual_seed(0)
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    q, s = H.quant_fp8_rows(w)
    xq, xs = H.quant_fp8_rows(x)
    xd = R.dequant_fp8(xq, xs)  # the activations the kernel actually multiplies
    y = H.linear_w8a8(x, q, s, b, act="gelu_tanh", tile=tile, depth=depth, split=split)
    close(y, R.linear(xd, q, b.float(), act="gelu_tanh", w_scale=s), 2e-2)
    yg = H.linear_w8a8(x, q, s, None, glu=True, tile=tile, depth=depth, split=split)
    close(yg, R.linear(xd, q, None, glu=True, w_scale=s), 2e-2)
    # and close to the bf16-activation result: per-token fp8 activation error only (~3% relative RMS)
    ya, yr = H.linear(x, q, b, w_scale=s).float(), R.linear(x.float(), q, b.float(), w_scale=s)
    assert ((ya - yr).norm() / yr.norm()).item() < 0.05


@pytest.mark.parametrize("K", [1024, 4096, 8192, 11008])
def test_quant_fp8_activation_rows(K):
    """Per-token activation quantisation (strided rows, one pass) == the two-pass weight quantiser."""
    torch.manual_seed(1)
    xf = rnd(37, K + 64)
    x = xf[:, 32:32 + K] if K <= 8192 else xf[:, :K].contiguous()  # strided rows (one-pass kernel) or long rows
    q = torch.empty(37, K, dtype=torch.uint8, device=dev)
    s = torch.empty(37, dtype=torch.float32, device=dev)
    H.lib().quant_fp8_rows_ld(x.data_ptr(), x.stride(0), q.data_ptr(), s.data_ptr(), 37, K, H._stream())
    q_ref, s_ref = H.quant_fp8_rows(x.contiguous())
    assert torch.equal(q, q_ref) and torch.equal(s, s_ref)


@pytest.mark.parametrize("M", [64, 256, 512])
def test_w8a8_decode_plan_in_graph(M):
    """A tuned W8A8 plan (fp8 activations quantised into the reusable scratch, MX-fp8
    MFMA) runs inside a captured HIP graph and replays exactly the eager values; both match fp32 math on
    the same fp8 operands. The plan goes through the tuned table exactly as a decode step consults it."""
    from llmss_amd import _native

    torch.manual_seed(2)
    N, K = 1024, 4096
    w = rnd(N, K, scale=K ** -0.5)
    q, s = H.quant_fp8_rows(w)
    b = rnd(N, scale=0.1)
    x = rnd(M, K)
    lib = _native()
    nt = H.W8A8_FLAG | (3 << 8) | (3 << 12)
    lib.gemm_tuned_set(M, N, K, False, 1, nt, 2)
    try:
        eager = H.linear(x, q, b, w_scale=s)
        y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        g = torch.cuda.CUDAGraph()
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            H.linear(x, q, b, w_scale=s, out=y)
        torch.cuda.current_stream().wait_stream(st)
        with torch.cuda.graph(g, capture_error_mode="thread_local"):
            H.linear(x, q, b, w_scale=s, out=y)
        x2 = rnd(M, K)
        x.copy_(x2)
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
    finally:
        lib.gemm_tuned_clear()
    xq, xs = H.quant_fp8_rows(x2)
    ref = R.linear(R.dequant_fp8(xq, xs), q, b.float(), w_scale=s)
    close(y, ref, 2e-2)
    assert not torch.equal(eager, y)  # the replay read the new activations


def _row_stats(h):
    hf = h.float()
    return torch.stack([hf.sum(1), hf.pow(2).sum(1)], 1).contiguous()


@pytest.mark.parametrize("variant,nt", [(1, 1), (1, 2), (2, 1), (2, 2)])
@pytest.mark.parametrize("split", [1, 4])
@pytest.mark.parametrize("M", [17, 33, 64])
def test_gemm_streaming_kernels_up_to_64_rows(variant, nt, split, M):
    """The weight-streaming kernels (four 16-row MFMA tiles per wave at M = 49-64) are autotuner candidates
    up to M = 64: explicit hints vs the fp32 oracle, with bias / GELU / SwiGLU epilogues and split-K."""
    torch.manual_seed(0)
    N, K = 2752, 4096
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    hint = nt + 16 * variant
    close(H.linear(x, w, b, nt_hint=hint, split_hint=split), R.linear(x.float(), w.float(), b.float()), 2e-2)
    close(H.linear(x, w, b, act="gelu_tanh", nt_hint=hint, split_hint=split),
          R.linear(x.float(), w.float(), b.float(), act="gelu_tanh"), 2e-2)
    close(H.linear(x, w, None, glu=True, nt_hint=hint, split_hint=split),
          R.linear(x.float(), w.float(), None, glu=True), 2e-2)


@pytest.mark.parametrize("tile,depth", [(11, 3), (11, 4), (10, 3), (13, 4), (8, 3), (12, 3), (9, 3), (14, 4), (15, 3), (7, 4)])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("M,N,K", [(64, 1280, 2048), (37, 4096, 1024), (300, 544, 3072), (512, 2752, 4096)])
def test_gemm_w8a8_mid_tiles(tile, depth, split, M, N, K):
    """W8A8 through the gemm_mid kernels (fp8 MFMA on the buffer-descriptor ring, scales in registers before the
    epilogue): exact vs fp32 math on the same fp8 operands; slabs left to a consumer carry the scales."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    q, s = H.quant_fp8_rows(w)
    xq, xs = H.quant_fp8_rows(x)
    xd = R.dequant_fp8(xq, xs)
    y = H.linear_w8a8(x, q, s, b, act="gelu_tanh", tile=tile, depth=depth, split=split)
    close(y, R.linear(xd, q, b.float(), act="gelu_tanh", w_scale=s), 2e-2)
    if tile not in ODD_NT_TILES:
        yg = H.linear_w8a8(x, q, s, None, glu=True, tile=tile, depth=depth, split=split)
        close(yg, R.linear(xd, q, None, glu=True, w_scale=s), 2e-2)
    p = H.linear_w8a8(x, q, s, None, tile=tile, depth=depth, split=split, partial_ok=True)
    if isinstance(p, H.PartialSum):
        res = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
        _, r = H.add_norm_partial(p, torch.ones(N, dtype=torch.bfloat16, device=dev), None, 1e-5, True, res)
        close(r, R.linear(xd, q, None, w_scale=s), 2e-2)
    else:
        close(p, R.linear(xd, q, None, w_scale=s), 2e-2)


@pytest.mark.parametrize("up_tile", [8, 11, 10, 13, 9, 12])
@pytest.mark.parametrize("M,F,K", [(512, 1024, 2048), (129, 512, 1024), (64, 256, 1024)])
def test_w8a8_swiglu_mx_output_feeds_the_down_projection(up_tile, M, F, K):
    """A W8A8 SwiGLU GEMM writes its output as MX-fp8 (e4m3 + one e8m0 scale per 32 outputs)
    and the down projection consumes it on the MX-fp8 MFMA with per-lane block scales, so no bf16 intermediate and no
    quantisation launch sit between them.
    * producer: bit-identical to the CPU MX quantisation (ops/reference.py quant_mx_fp8) of the same kernel's bf16
      output, for every tile whose outputs hold whole 32-column blocks (BN % 64 == 0);
    * consumer: every gemm_mid tile, plain and software-pipelined k-loops, split-K slabs and all, == fp32 math on the
      dequantised MX activations."""
    torch.manual_seed(0)
    x = rnd(M, K)
    wu, wd = rnd(2 * F, K, scale=K ** -0.5), rnd(768, F, scale=F ** -0.5)
    qu, su = H.quant_fp8_rows(wu)
    qd, sd = H.quant_fp8_rows(wd)
    y = H.linear_w8a8(x, qu, su, None, glu=True, tile=up_tile, depth=3, split=1)
    mx = H.linear_w8a8(x, qu, su, None, glu=True, tile=up_tile, depth=3, split=1, mx_out=True)
    assert isinstance(mx, H.MxAct) and mx.q.shape == (M, F) and mx.s.shape == (M, F // 32)
    rq, rs = R.quant_mx_fp8(y.float().cpu())
    assert torch.equal(mx.s.cpu(), rs) and torch.equal(mx.q.cpu(), rq)
    ref = R.linear(R.dequant_mx_fp8(rq, rs), qd.cpu(), None, w_scale=sd.cpu()).float()
    for tile, depth, split, ilv in [(8, 3, 1, False), (8, 4, 1, True), (11, 4, 3, True), (10, 3, 1, False),
                                    (13, 5, 2, True), (14, 4, 1, False), (15, 3, 3, True), (7, 4, 1, False),
                                    (9, 3, 2, False), (12, 3, 1, False)]:
        yd = H.linear_w8a8(mx, qd, sd, None, tile=tile, depth=depth, split=split, ilv=ilv)
        close(yd.float().cpu(), ref, 2e-2)
        p = H.linear_w8a8(mx, qd, sd, None, tile=tile, depth=depth, split=split, ilv=ilv, partial_ok=True)
        if isinstance(p, H.PartialSum):
            p = p.buf[: p.S * M * 768].view(p.S, M, 768).sum(0)
        close(p.float().cpu(), ref, 2e-2)


@pytest.mark.parametrize("tile,depth", [(8, 3), (8, 4), (8, 5), (11, 4), (9, 3), (12, 3), (13, 5), (15, 3)])
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("M,N,K", [(512, 2752, 4096), (300, 544, 3072), (129, 1024, 640)])
def test_gemm_w8a8_mid_tiles_software_pipelined(tile, depth, split, M, N, K):
    """The fp8 gemm_mid k-loop with k-step t+1's fragment reads and the ring issue between k-step t's MFMAs
    (W8A8_ILV): bit-identical to the plain loop (same MFMA order per accumulator) and to fp32 math on the same fp8
    operands, through short K ranges per split (1-2 steps: the pipeline's prologue and tail alone) too."""
    torch.manual_seed(0)
    x, w, b = rnd(M, K), rnd(N, K, scale=K ** -0.5), rnd(N, scale=0.1)
    q, s = H.quant_fp8_rows(w)
    xq, xs = H.quant_fp8_rows(x)
    xd = R.dequant_fp8(xq, xs)
    for glu in ([False] if tile in ODD_NT_TILES else [False, True]):
        kw = dict(act="none" if glu else "gelu_tanh", glu=glu, tile=tile, depth=depth, split=split)
        y = H.linear_w8a8(x, q, s, None if glu else b, ilv=True, **kw)
        assert torch.equal(y, H.linear_w8a8(x, q, s, None if glu else b, **kw))
        close(y, R.linear(xd, q, None if glu else b.float(), act=kw["act"], glu=glu, w_scale=s), 2e-2)
    # through the nt_hint encoding a tuned plan carries
    hint = H.W8A8_FLAG | H.W8A8_ILV | (tile << 8) | (depth << 12)
    close(H.linear(x, q, b, w_scale=s, nt_hint=hint, split_hint=split), R.linear(xd, q, b.float(), w_scale=s), 2e-2)


@pytest.mark.parametrize("ch,nbytes,us", [(32, 4 << 20, 40.0), (16, 64 << 10, 12.0), (64, 32 << 20, 120.0)])
def test_comm_model_holds_its_channels_for_the_modelled_time(ch, nbytes, us):
    """The many-CU modelled collective of the simulated TP shard (csrc/comm_model.hip): each call lasts the modelled
    time (its traffic done within it, or the time stretched by the traffic), timed over 10 calls in a HIP graph."""
    lib = H.lib()
    buf = torch.empty(ch * 2 * lib.comm_model_slice(ch, nbytes), dtype=torch.uint8, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    lib.comm_model(buf.data_ptr(), ch, nbytes, us, st)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        for _ in range(10):
            lib.comm_model(buf.data_ptr(), ch, nbytes, us, torch.cuda.current_stream().cuda_stream)
    g.replay()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    g.replay()
    e.record()
    e.synchronize()
    per = s.elapsed_time(e) * 1e3 / 10
    assert us * 0.98 <= per <= us * 1.5 + 10, per
