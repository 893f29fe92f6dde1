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
