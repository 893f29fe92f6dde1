"""The query / key / value product of untuned models: one launch by the decode kernel's unsplit plan, with the values of the two."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows of the decode kernel and past it; an even and a packed cache, one key head, turned heads (Llama's
# halves lie side by side in the loaded weights)
@pytest.mark.parametrize("preset,over", [("tiny-gpt2", dict(hidden_size=1024, num_heads=16, num_kv_heads=16, head_dim=64)),
                                         ("tiny-bigcode", dict(hidden_size=512, num_heads=8, num_kv_heads=1, head_dim=64)),
                                         ("tiny-gptj", dict(hidden_size=512, num_heads=8, num_kv_heads=8, head_dim=64, rotary_dim=32)),
                                         ("tiny-llama", dict(hidden_size=512, num_heads=8, num_kv_heads=2, head_dim=64, rotary_dim=64))])
@pytest.mark.parametrize("M", [1, 7, 16, 33, 64, 65])
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
    slots = torch.randperm(16 * 12, generator=g)[:M].cuda()
    slots[M // 2] = -1
    inp = StepInput("decode", torch.zeros(M, dtype=torch.long, device="cuda"), torch.randint(0, 128, (M,), generator=g).cuda(), slots)
    plan = m._qkv_plan(M, L.qkv.N, L.qkv.K)
    calls, real = [], hip.linear_qkv
    monkeypatch.setattr(hip, "linear_qkv", lambda *a: calls.append(real(*a)) or calls[-1])
    res = []
    for one in (True, False):
        m.qkv_epi = one
        kv = m.allocate_kv_cache(12, 16)[0]
        res.append((m._qkv_rope_cache(L, y, inp, *kv), *kv))
    assert len(calls) == (plan is not None)
    assert (plan is not None) == (M <= 64) if preset == "tiny-gpt2" else plan is None or M <= 64
    fused = bool(calls) and calls[0] is not None
    for a, b in zip(*res):
        if fused:  # turned from the fp32 sums or from their bf16 rows, the sums split or not: a rounding each, of a number and its partner
            lim = 2.0 ** -7 * (a.double().abs() + (b.double().abs().amax() if cfg.position == "rope" else 0.0)) + 1e-5
            assert ((a.double() - b.double()).abs() <= lim).all()
        else:
            assert torch.equal(a, b)


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
    res = []
    for one in (True, False):
        kc, vc = (torch.zeros(nb, nkv, 16, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        if one:
            y = hip.linear_qkv(x, w, b, pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, "gptj", rot > 0, 4 << 8, 1)
            assert y is not None
        else:
            y = hip.rope_cache(hip.linear(x, w, b, nt_hint=4 << 8, split_hint=1), pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, "gptj", rot > 0)
        res.append((y, kc, vc))
    for a, c in zip(*res):  # bf16 rows turned in fp32, from sums that may be in another order: a rounding each, of a number and its partner
        assert ((a.double() - c.double()).abs() <= 2.0 ** -7 * (c.double().abs() + (c.double().abs().amax() if rot else 0.0)) + 1e-5).all()
    assert (res[0][1][nb - 1].abs().sum() > 0) == (res[1][1][nb - 1].abs().sum() > 0)
    # halves that turn against each other are not this form's
    assert rot == 0 or hip.linear_qkv(x, w, b, pos, cos, sin, None, None, None, nh, nkv, D, rot, "neox", True, 4 << 8, 1) is None
