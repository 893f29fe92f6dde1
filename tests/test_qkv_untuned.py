"""The query / key / value product of untuned models: one launch by the decode kernel's unsplit plan or by a prompt's tiles, and the two
launches that it stands for, against 64 bits; rows that are kept further apart read as others are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def check(y, kc, vc, x, w, b, pos, slots, cos, sin, nh, nkv, D, rot, style):
    """Rows [T, N] and caches of zeros before, after the product, the rotation (rot 0: none) and the cache write."""
    T, K = x.shape
    xd, wd, n = x.double(), w.double(), (nh + nkv) * D
    z, e = xd @ wd.t(), (K + 2) * 2.0 ** -24 * (xd.abs() @ wd.abs().t())  # sums in 32 bits, whatever their order
    if b is not None:
        z, e = z + b.double(), e + 2.0 ** -23 * b.double().abs()
    r = 2.0 ** -8  # a rounding to bf16
    lim = e + r * (z.abs() + e)
    if rot:  # turned in 32 bits, before or after a rounding, and rounded
        heads, err = z[:, :n].view(T, -1, D), lim[:, :n].view(T, -1, D)
        i, j = (slice(0, rot, 2), slice(1, rot, 2)) if style == "gptj" else (slice(0, rot // 2), slice(rot // 2, rot))
        c, s = (t.double()[pos][:, None] for t in (cos, sin))
        p, q, ep, eq = heads[..., i].clone(), heads[..., j].clone(), err[..., i].clone(), err[..., j].clone()
        for at, first, second, ef, es in ((i, p * c, -q * s, ep, eq), (j, q * c, p * s, eq, ep)):
            v = first + second
            ev = c.abs() * ef + s.abs() * es + 2.0 ** -22 * (first.abs() + second.abs())
            heads[..., at], err[..., at] = v, ev + r * (v.abs() + ev)
    assert ((y.double() - z).abs() <= lim * (1 + 2.0 ** -20) + 1e-30).all()
    live = slots >= 0
    at = (slots[live] // kc.shape[2], slice(None), slots[live] % kc.shape[2])
    for cache, rows in ((kc, y[:, nh * D:n]), (vc, y[:, n:])):
        assert torch.equal(cache[at], rows[live].reshape(-1, nkv, D))
        cache[at] = 0.0
        assert not cache.any()


# rows of the decode kernel and past it, and of tiles below 256 x 256; an even and a packed cache, one key head, turned heads (Llama's
# halves lie side by side in the loaded weights), rows a multiple of 4 KB wide
@pytest.mark.parametrize("preset,over", [("tiny-gpt2", dict(hidden_size=1024, num_heads=16, num_kv_heads=16, head_dim=64)),
                                         ("tiny-bigcode", dict(hidden_size=512, num_heads=8, num_kv_heads=1, head_dim=64)),
                                         ("tiny-gptj", dict(hidden_size=512, num_heads=8, num_kv_heads=8, head_dim=64, rotary_dim=32)),
                                         ("tiny-llama", dict(hidden_size=512, num_heads=8, num_kv_heads=2, head_dim=64, rotary_dim=64)),
                                         ("tiny-llama", dict(hidden_size=1024, num_heads=16, num_kv_heads=8, head_dim=64, rotary_dim=64))])
@pytest.mark.parametrize("M", [1, 7, 16, 33, 64, 65, 128, 300, 2100])
def test_one_launch_and_two(preset, over, M, monkeypatch):
    from llmss_amd.models.config import get_preset
    from llmss_amd.models.decoder import DecoderLM, StepInput
    from llmss_amd.models.weights import random_weights
    from llmss_amd.ops import hip
    cfg = get_preset(preset, intermediate_size=512, max_position_embeddings=128, **over)
    m = DecoderLM(cfg, random_weights(cfg, device="cuda", dtype=torch.bfloat16, seed=3, std=0.05))
    L = m.w.layers[0]
    g = torch.Generator().manual_seed(M)
    y = torch.randn(M, cfg.hidden_size, generator=g).bfloat16().cuda()
    nb = max(12, -(-M // 16) + 1)
    slots = torch.randperm(16 * nb, generator=g)[:M].cuda()
    slots[M // 2] = -1
    inp = StepInput("decode", torch.zeros(M, dtype=torch.long, device="cuda"), torch.randint(0, 128, (M,), generator=g).cuda(), slots)
    plan = m._qkv_plan(M, L.qkv.N, L.qkv.K)
    calls, real = [], hip.linear_qkv
    monkeypatch.setattr(hip, "linear_qkv", lambda *a: calls.append(real(*a)) or calls[-1])
    rot = m.cfg.rotary_dim if m.cfg.position == "rope" else 0
    for one in (True, False):
        m.qkv_epi = one
        kv = m.allocate_kv_cache(nb, 16)[0]
        qkv = m._qkv_rope_cache(L, y, inp, *kv)
        check(qkv, *kv, y, L.qkv.w, L.qkv.b, inp.positions, slots, m.w.cos, m.w.sin, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, rot,
              m.cfg.rope_style)
    assert len(calls) == (plan is not None)
    fused = bool(calls) and calls[0] is not None
    if M <= 64:
        assert plan is not None or preset != "tiny-gpt2"
    else:  # (those of 2048 and 3072 columns split K below)
        assert fused == (M >= 128 and (L.qkv.N < 2048 or M == 2100))
    if fused and M >= 128:
        rows = calls[0]
        assert rows.stride(0) == L.qkv.N + (hip.QKV_PAD if L.qkv.N == 2048 else 0)
        args = (cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.head_dim ** -0.5)
        cu = torch.tensor([0, M - 50, M]).int().cuda()
        assert torch.equal(hip.attn_prefill(rows, cu, M - 50, *args), hip.attn_prefill(rows.contiguous(), cu, M - 50, *args))
        bt, ctx = torch.randint(0, nb, (2, nb), generator=g).int().cuda(), torch.tensor([M + 10, 60]).int().cuda()
        kv = [t.normal_() for t in kv]
        got, want = (hip.attn_extend(t, *kv, bt, cu, ctx, M - 50, *args) for t in (rows, rows.contiguous()))
        assert torch.equal(got, want)


# 256 x 256 tiles: whole and partial ones, rows or columns left over to other tiles (up to 64 rows: the decode kernel), heads of half a wave's
# columns to all of a tile's, one key head, pairs turned in part or not at all, rows that are not cached
@pytest.mark.parametrize("M,K,nh,nkv,D,rot", [(1, 64, 2, 1, 128, 128), (300, 128, 3, 3, 64, 64), (257, 192, 2, 2, 256, 64), (520, 64, 5, 1, 64, 0),
                                              (8261, 256, 8, 4, 128, 128), (8230, 1024, 8, 4, 128, 128), (8230, 256, 16, 8, 64, 64),
                                              (4352, 1024, 32, 2, 128, 32)])
def test_tiles_of_prompts(M, K, nh, nkv, D, rot):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(M)
    N = (nh + 2 * nkv) * D
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if M % 2 else None
    pos = torch.randint(0, 90, (M,), generator=g).cuda()
    ang = torch.rand(90, max(rot // 2, 4), generator=g).cuda() * 6
    cos, sin = ang.cos(), ang.sin()
    nb = -(-M // 16) + 1
    slots = torch.randperm(nb * 16, generator=g)[:M].cuda()
    slots[M // 3] = -1
    for one in (True, False):
        kc, vc = (torch.zeros(nb, nkv, 16, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        if one:
            y = hip.linear_qkv(x, w, b, pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, "gptj", rot > 0, 4 << 8, 1)
            assert y is not None
        else:
            y = hip.linear(x, w, b, nt_hint=4 << 8, split_hint=1)
            y = hip.rope_cache(y, pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, "gptj", rot > 0)
        check(y, kc, vc, x, w, b, pos, slots, cos, sin, nh, nkv, D, rot, "gptj")
    # halves that turn against each other are not this form's
    assert rot == 0 or hip.linear_qkv(x, w, b, pos, cos, sin, None, None, None, nh, nkv, D, rot, "neox", True, 4 << 8, 1) is None
