"""End-to-end GPU parity against HF transformers checkpoints (fp32 HF on CPU as the oracle):
prefill logits and greedy continuations of all five families through the native bf16 kernels, fp8
(W8A16 / W8A8) Llama against its bf16 twin, and generate.py's no-cache (recompute) mode against its
cached mode on the GPU."""
import ast
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu

VOCAB = 1000


def _hf(name):
    from transformers import (GPT2Config, GPT2LMHeadModel, GPTBigCodeConfig, GPTBigCodeForCausalLM, GPTJConfig,
                              GPTJForCausalLM, LlamaConfig, LlamaForCausalLM)

    torch.manual_seed(0)
    kw = dict(vocab_size=VOCAB, bos_token_id=VOCAB - 1, eos_token_id=VOCAB - 1)
    if name == "gpt2":
        return GPT2LMHeadModel(GPT2Config(n_embd=256, n_layer=3, n_head=4, n_positions=256, initializer_range=0.05,
                                          **kw))
    if name == "gptj":
        return GPTJForCausalLM(GPTJConfig(n_embd=512, n_layer=2, n_head=2, n_positions=256, rotary_dim=64,
                                          initializer_range=0.05, **kw))
    if name == "bigcode":
        return GPTBigCodeForCausalLM(GPTBigCodeConfig(n_embd=512, n_layer=2, n_head=4, n_positions=256,
                                                      multi_query=True, initializer_range=0.05, **kw))
    if name == "bigcode_mha":
        return GPTBigCodeForCausalLM(GPTBigCodeConfig(n_embd=256, n_layer=2, n_head=4, n_positions=256,
                                                      multi_query=False, initializer_range=0.05, **kw))
    return LlamaForCausalLM(LlamaConfig(hidden_size=512, num_hidden_layers=2, num_attention_heads=4,
                                        num_key_value_heads=2, intermediate_size=1024, max_position_embeddings=256,
                                        initializer_range=0.05, **kw))


def _prompts():
    g = torch.Generator().manual_seed(5)
    return [torch.randint(0, VOCAB - 1, (n,), generator=g).tolist() for n in (9, 31, 64, 17)]


@pytest.mark.parametrize("name", ["gpt2", "gptj", "bigcode", "bigcode_mha", "llama"])
def test_native_bf16_matches_hf(tmp_path, name):
    from llmss_amd.engine import LLMEngine, SamplingParams, build_model
    from llmss_amd.models.decoder import StepInput

    hf = _hf(name).eval()
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    dev = torch.device("cuda", 0)
    m = build_model(str(tmp_path), None, "bf16", dev)
    ps = _prompts()
    # all-position prefill logits of the packed batch vs HF per prompt
    ids = torch.tensor([t for p in ps for t in p], device=dev)
    pos = torch.cat([torch.arange(len(p)) for p in ps]).to(dev)
    cu = torch.tensor([0] + torch.tensor([len(p) for p in ps]).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    kv = m.allocate_kv_cache(32, 16)
    inp = StepInput("prefill", ids, pos, torch.full_like(ids, -1), cu_seqlens=cu, max_seqlen=max(map(len, ps)))
    got = m(inp, kv)[:, :VOCAB].float().cpu()
    with torch.no_grad():
        ref = torch.cat([hf(torch.tensor([p])).logits[0] for p in ps])
    scale = ref.abs().max()
    err = (got - ref).abs().max() / scale
    cos = torch.nn.functional.cosine_similarity(got, ref, dim=-1).min()
    assert err < 3e-2 and cos > 0.999, (name, float(err), float(cos))
    # greedy continuations through the engine (paged decode, HIP graphs) vs HF generate
    eng = LLMEngine(m, max_num_seqs=4, block_size=16, autotune=False)
    out = eng.generate(ps, SamplingParams(max_new_tokens=10, is_greedy=True, ignore_eos=True))
    # margin-aware greedy agreement: every token must match HF's greedy token, except at a position where HF's
    # own top-2 logit margin is within bf16 noise (a few times the measured prefill error): there a flip is a
    # tie-break, and the rest of that sequence is conditioned on a different token, so comparison stops
    noise = max(4 * float(err) * float(scale), 1e-3)
    compared = ties = 0
    for p, o in zip(ps, out):
        with torch.no_grad():
            r = hf.generate(torch.tensor([p]), max_new_tokens=10, do_sample=False, min_new_tokens=10,
                            pad_token_id=0)[0, len(p):].tolist()
            lg = hf(torch.tensor([p + r])).logits[0, len(p) - 1:len(p) + len(r) - 1]
        top2 = lg.topk(2, dim=-1).values
        margin = (top2[:, 0] - top2[:, 1]).tolist()
        for i, (a, b) in enumerate(zip(o, r)):
            if a == b:
                compared += 1
                continue
            assert margin[i] < noise, (name, "greedy token differs at a clear margin", i, margin[i], noise, o, r)
            ties += 1
            break
    assert compared >= 0.75 * 10 * len(ps), (name, compared, ties, out)


def test_fp8_llama_end_to_end_vs_bf16(tmp_path):
    from llmss_amd.engine import LLMEngine, SamplingParams, build_model
    from llmss_amd.models.decoder import StepInput

    hf = _hf("llama").eval()
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    dev = torch.device("cuda", 0)
    ps = _prompts()
    outs = {}
    for fp8 in (False, True):
        m = build_model(str(tmp_path), None, "bf16", dev, fp8=fp8)
        assert (m.w.layers[0].qkv.w.dtype == torch.uint8) == fp8  # e4m3 weight bytes + per-channel scales
        ids = torch.tensor([t for p in ps for t in p], device=dev)
        pos = torch.cat([torch.arange(len(p)) for p in ps]).to(dev)
        cu = torch.tensor([0] + torch.tensor([len(p) for p in ps]).cumsum(0).tolist(), dtype=torch.int32, device=dev)
        inp = StepInput("prefill", ids, pos, torch.full_like(ids, -1), cu_seqlens=cu, max_seqlen=max(map(len, ps)),
                        last_idx=(cu[1:] - 1).long())
        lg = m(inp, m.allocate_kv_cache(32, 16))[:, :VOCAB].float().cpu()
        eng = LLMEngine(m, max_num_seqs=4, block_size=16, autotune=False)
        gen = eng.generate(ps, SamplingParams(max_new_tokens=12, is_greedy=True, ignore_eos=True))
        outs[fp8] = (lg, gen)
        del eng, m
        torch.cuda.empty_cache()
    (lb, gb), (lf, gf) = outs[False], outs[True]
    cos = torch.nn.functional.cosine_similarity(lb, lf, dim=-1).min()
    err = (lb - lf).abs().max() / lb.abs().max()
    print(f"fp8 vs bf16 logits: min cosine {float(cos):.5f}, max err / max |logit| {float(err):.4f}")
    assert cos > 0.99 and err < 0.15, (float(cos), float(err))
    first = sum(a[0] == b[0] for a, b in zip(gb, gf))
    assert first >= 3, (gb, gf)


def _to(obj, dev):
    """A copy of a weights container (dataclasses / lists / dicts of tensors) on ``dev``."""
    import dataclasses

    if isinstance(obj, torch.Tensor):
        return obj.to(dev)
    if dataclasses.is_dataclass(obj):
        return dataclasses.replace(obj, **{f.name: _to(getattr(obj, f.name), dev) for f in dataclasses.fields(obj)
                                           if f.init})
    if isinstance(obj, list):
        return [_to(o, dev) for o in obj]
    if isinstance(obj, dict):
        return {k: _to(v, dev) for k, v in obj.items()}
    return obj


def test_fp8_w8a8_prefill_and_decode_vs_fake_quant_oracle(tmp_path, monkeypatch):
    """The W8A8 path end to end (per-token e4m3 activations on the MX-fp8 matrix cores), not W8A16.
    Prefill: 153 prompt tokens, so every fp8 GEMM runs W8A8 (untuned calls above 128 rows), its activations quantised
    by add_norm's fp8 twin (qkv, up) or the quantisation kernel (o, down). Decode: 4 rows with W8A8 plans forced into
    the tuned table for every fp8 shape. Oracle: the same quantised weights in the CPU reference model with every fp8
    linear's input fake-quantised per token (ops/reference.py fake_quant_fp8_act): an fp32 oracle of W8A8. Parity
    against an fp8 reference is unpinned (the reference has no fp8); this is the repo's own oracle.
    * Every fp8 GEMM of both steps, on the exact bf16 input it received in the model: GPU W8A8 == oracle within
      1e-2 of max |y| (fp32 accumulation order and the bf16 output rounding are all that differ).
    * End to end, e4m3 activations are chaotic: one bf16 rounding moved across a quantisation boundary moves a value
      by an e4m3 step (6-12 %). The oracle itself moves by that much when its intermediates are fp32 instead of bf16
      (its noise floor, measured here); the GPU logits must sit within 1.5x that floor of the oracle, and closer to
      it than to the W8A16 oracle (weights dequantised, bf16 activations)."""
    import dataclasses
    import functools

    import llmss_amd.ops as O
    from llmss_amd.engine import build_model
    from llmss_amd.models.decoder import DecoderLM, StepInput
    from llmss_amd.models.weights import Linear
    from llmss_amd.ops import hip as H
    from llmss_amd.ops import reference as R

    hf = _hf("llama").eval()
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    dev = torch.device("cuda", 0)
    m = build_model(str(tmp_path), None, "bf16", dev, fp8=True)
    L = m.w.layers[0]
    lins = (L.qkv, L.o, L.up, L.down)
    assert all(lin.w.dtype == torch.uint8 for lin in lins)
    g = torch.Generator().manual_seed(11)
    lens = [40, 50, 30, 33]
    T, B = sum(lens), len(lens)
    ps = [torch.randint(0, VOCAB - 1, (n,), generator=g).tolist() for n in lens]
    assert all(H.w8a8_planned(T, lin.N, lin.K, lin.glu) for lin in lins)  # untuned M > 128: W8A8
    lib = H.lib()
    plan = H.W8A8_FLAG | (3 << 8) | (3 << 12)  # 64x64 W8A8 tile, 3-stage ring
    for lin in lins:
        lib.gemm_tuned_set(B, lin.N, lin.K, lin.glu, 1, plan, 1)
    assert all(H.w8a8_planned(B, lin.N, lin.K, lin.glu) for lin in lins)
    bs, per = 16, 4  # 4 blocks of 16 per sequence

    def run(model, d):
        ids = torch.tensor([t for p in ps for t in p], device=d)
        pos = torch.cat([torch.arange(n) for n in lens]).to(d)
        slots = torch.cat([torch.arange(n) + i * per * bs for i, n in enumerate(lens)]).to(d)
        cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=d)
        kv = model.allocate_kv_cache(B * per, bs)
        lp = model(StepInput("prefill", ids, pos, slots, cu_seqlens=cu, max_seqlen=max(lens),
                             last_idx=(cu[1:] - 1).long()), kv)[:, :VOCAB].float().cpu()
        nxt = torch.tensor([7, 99, 500, 3], device=d)  # fixed next tokens: the decode inputs do not hinge on a tie
        bt = torch.arange(B * per, dtype=torch.int32).view(B, per).to(d)
        inp = StepInput("decode", nxt, torch.tensor(lens, device=d), torch.tensor(
            [i * per * bs + n for i, n in enumerate(lens)], device=d), block_tables=bt,
            ctx_lens=torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=d), max_ctx=per * bs)
        ld = model(inp, kv)[:, :VOCAB].float().cpu()
        return lp, ld

    recs = []
    call = Linear.__call__

    def recording(self, x, act="none", partial_ok=False):
        if self.w_scale is not None and x.is_cuda:
            recs.append((self, x.clone(), act))
        return call(self, x, act, partial_ok)

    monkeypatch.setattr(Linear, "__call__", recording)
    try:
        gp, gd = run(m, dev)
        assert len(recs) == 2 * len(m.w.layers) * 4 and {x.shape[0] for _, x, _ in recs} == {T, B}
        worst = 0.0
        for lin, x, act in recs:  # each fp8 GEMM on its exact model input: W8A8 kernel vs the fake-quant oracle
            y = H.linear(x, lin.w, lin.b, act, lin.glu, lin.w_scale).float().cpu()
            ref = R.linear(x.cpu(), lin.w.cpu(), None if lin.b is None else lin.b.cpu(), act, lin.glu,
                           lin.w_scale.cpu(), a8=True).float()
            worst = max(worst, float((y - ref).abs().max() / ref.abs().max()))
    finally:
        lib.gemm_tuned_clear()
    monkeypatch.setattr(Linear, "__call__", call)
    print(f"per-GEMM W8A8 vs fake-quant oracle on identical inputs: max rel err {worst:.5f}")
    assert worst <= 1e-2, worst

    wc = _to(m.w, "cpu")
    mc = DecoderLM(m.cfg, wc)
    w16 = run(mc, "cpu")
    monkeypatch.setattr(O.ref, "linear", functools.partial(R.linear, a8=True))
    w8 = run(mc, "cpu")

    def to32(o):  # the oracle with fp32 intermediates: its own sensitivity to the bf16 rounding points
        if isinstance(o, torch.Tensor):
            return o.float() if o.dtype == torch.bfloat16 else o
        if dataclasses.is_dataclass(o):
            return dataclasses.replace(o, **{f.name: to32(getattr(o, f.name)) for f in dataclasses.fields(o) if f.init})
        return [to32(v) for v in o] if isinstance(o, list) else o

    w8f = run(DecoderLM(m.cfg, to32(wc)), "cpu")

    def err(a, b):
        return float((a - b).abs().max() / b.abs().max())

    e8 = (err(gp, w8[0]), err(gd, w8[1]))
    e16 = (err(gp, w16[0]), err(gd, w16[1]))
    floor = (err(w8f[0], w8[0]), err(w8f[1], w8[1]))
    print(f"W8A8 GPU vs fake-quant oracle: prefill {e8[0]:.4f} decode {e8[1]:.4f}; oracle noise floor (fp32 vs bf16 "
          f"intermediates) {floor[0]:.4f} / {floor[1]:.4f}; GPU vs the W8A16 oracle {e16[0]:.4f} / {e16[1]:.4f}")
    for k in range(2):
        assert e8[k] <= 1.5 * floor[k], (e8, floor)
        assert e8[k] < e16[k], (e8, e16)  # the oracle tells W8A8 from W8A16


def test_fp8_mlp_mx_handoff_vs_fake_quant_oracle(tmp_path, monkeypatch):
    """At model level: with W8A8 gemm_mid plans for every fp8 GEMM (forced into the tuned table,
    prefill 153 rows and decode 4 rows), DecoderLM._mlp has the gate/up epilogue write its SwiGLU output as MX-fp8 and
    the down projection consume it - no bf16 intermediate, no quantisation launch. Oracle: the CPU reference with
    per-token fake-quant activations for qkv / o / gate-up and MX fake-quant (ops/reference.py fake_quant_mx_act) for
    the down projection's input. As in the W8A8 test above, e4m3 activations are chaotic end to end: the GPU logits
    must sit within 1.5x the oracle's own fp32-vs-bf16 noise floor of it, and closer to it than to the W8A16 oracle."""
    import dataclasses

    import llmss_amd.ops as O
    from llmss_amd.engine import build_model
    from llmss_amd.models.decoder import DecoderLM, StepInput
    from llmss_amd.ops import hip as H
    from llmss_amd.ops import reference as R

    hf = _hf("llama").eval()
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    dev = torch.device("cuda", 0)
    m = build_model(str(tmp_path), None, "bf16", dev, fp8=True)
    L = m.w.layers[0]
    F = L.down.K
    g = torch.Generator().manual_seed(12)
    lens = [40, 50, 30, 33]
    T, B = sum(lens), len(lens)
    ps = [torch.randint(0, VOCAB - 1, (n,), generator=g).tolist() for n in lens]
    lib = H.lib()
    plans = {id(L.qkv): 11, id(L.o): 11, id(L.up): 8, id(L.down): 11}  # 64x128 / 128x128 gemm_mid W8A8 tiles
    for M in (T, B):
        for lin in (L.qkv, L.o, L.up, L.down):
            lib.gemm_tuned_set(M, lin.N, lin.K, lin.glu, 1, H.W8A8_FLAG | (plans[id(lin)] << 8) | (3 << 12), 1)
    assert H.mx_mlp_ok(T, L.up, L.down) and H.mx_mlp_ok(B, L.up, L.down)
    bs, per = 16, 4
    n_mx = [0]
    w8a8 = H.linear_w8a8

    def counting(*a, **k):
        n_mx[0] += bool(k.get("mx_out"))
        return w8a8(*a, **k)

    def run(model, d):
        ids = torch.tensor([t for p in ps for t in p], device=d)
        pos = torch.cat([torch.arange(n) for n in lens]).to(d)
        slots = torch.cat([torch.arange(n) + i * per * bs for i, n in enumerate(lens)]).to(d)
        cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=d)
        kv = model.allocate_kv_cache(B * per, bs)
        lp = model(StepInput("prefill", ids, pos, slots, cu_seqlens=cu, max_seqlen=max(lens),
                             last_idx=(cu[1:] - 1).long()), kv)[:, :VOCAB].float().cpu()
        bt = torch.arange(B * per, dtype=torch.int32).view(B, per).to(d)
        inp = StepInput("decode", torch.tensor([7, 99, 500, 3], device=d), torch.tensor(lens, device=d), torch.tensor(
            [i * per * bs + n for i, n in enumerate(lens)], device=d), block_tables=bt,
            ctx_lens=torch.tensor([n + 1 for n in lens], dtype=torch.int32, device=d), max_ctx=per * bs)
        return lp, model(inp, kv)[:, :VOCAB].float().cpu()

    monkeypatch.setattr(H, "linear_w8a8", counting)
    try:
        gp, gd = run(m, dev)
    finally:
        lib.gemm_tuned_clear()
    assert n_mx[0] == 2 * len(m.w.layers), n_mx  # every layer's MLP, prefill and decode, took the MX hand-off
    assert torch.isfinite(gp).all() and torch.isfinite(gd).all()

    ref_linear = R.linear  # O.ref is the reference module: patching O.ref.linear replaces R.linear

    def oracle_linear(x, w, bias=None, act="none", glu=False, w_scale=None, a8=False):
        mx = w_scale is not None and not glu and w.shape[1] == F  # the down projection's input
        return ref_linear(x, w, bias, act, glu, w_scale, a8="mx" if mx else True)

    wc = _to(m.w, "cpu")
    w16 = run(DecoderLM(m.cfg, wc), "cpu")
    monkeypatch.setattr(O.ref, "linear", oracle_linear)
    w8 = run(DecoderLM(m.cfg, wc), "cpu")

    def to32(o):
        if isinstance(o, torch.Tensor):
            return o.float() if o.dtype == torch.bfloat16 else o
        if dataclasses.is_dataclass(o):
            return dataclasses.replace(o, **{f.name: to32(getattr(o, f.name)) for f in dataclasses.fields(o) if f.init})
        return [to32(v) for v in o] if isinstance(o, list) else o

    w8f = run(DecoderLM(m.cfg, to32(wc)), "cpu")

    def err(a, b):
        return float((a - b).abs().max() / b.abs().max())

    e8 = (err(gp, w8[0]), err(gd, w8[1]))
    e16 = (err(gp, w16[0]), err(gd, w16[1]))
    floor = (err(w8f[0], w8[0]), err(w8f[1], w8[1]))
    print(f"MX hand-off GPU vs oracle: prefill {e8[0]:.4f} decode {e8[1]:.4f}; oracle noise floor {floor[0]:.4f} / "
          f"{floor[1]:.4f}; GPU vs W8A16 oracle {e16[0]:.4f} / {e16[1]:.4f}")
    for k in range(2):
        assert e8[k] <= 1.5 * floor[k], (e8, floor)
        assert e8[k] < e16[k], (e8, e16)


def test_fp8_decode_graphs_survive_a_prefill_that_grows_the_scratch(tmp_path):
    """Decode graphs are captured at engine start with the W8A8 / MX-fp8 activation scratch sized for <= 4 rows; the
    first prompt batch (320 rows) then grows it. The graphs keep the old addresses, so the old buffers must stay
    allocated (ops/hip.py _retire): greedy tokens with graphs equal the eager engine's, and the grown buffers were
    retired, not freed."""
    from llmss_amd.engine import LLMEngine, SamplingParams, build_model
    from llmss_amd.ops import hip as H

    hf = _hf("llama").eval()
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    dev = torch.device("cuda", 0)
    m = build_model(str(tmp_path), None, "bf16", dev, fp8=True)
    L = m.w.layers[0]
    lib = H.lib()
    plans = {id(L.qkv): 11, id(L.o): 11, id(L.up): 8, id(L.down): 11}  # W8A8 gemm_mid tiles, MX hand-off in the MLP
    g = torch.Generator().manual_seed(21)
    ps = [torch.randint(0, VOCAB - 1, (n,), generator=g).tolist() for n in (100, 90, 70, 60)]
    sp = SamplingParams(max_new_tokens=12, is_greedy=True, ignore_eos=True)
    for slotted, cls in ((H._QSCRATCH, H._QuantScratch), (H._PRESCRATCH, H._PreQScratch), (H._MXSCRATCH, H._MxScratch)):
        for it in slotted._items:  # start from empty scratch (earlier tests may have grown it past 320 rows)
            H._retire(it.q, it.s)
        slotted._items = [cls() for _ in slotted._items]
    outs = {}
    try:
        for graphs in (True, False):
            for M in (1, 2, 4):
                for lin in (L.qkv, L.o, L.up, L.down):
                    lib.gemm_tuned_set(M, lin.N, lin.K, lin.glu, 1, H.W8A8_FLAG | (plans[id(lin)] << 8) | (3 << 12), 1)
            eng = LLMEngine(m, max_num_seqs=4, block_size=16, autotune=False, use_graphs=graphs)
            n0 = len(H._RETIRED)
            outs[graphs] = eng.generate(ps, sp)
            if graphs:
                assert eng.graphs and len(H._RETIRED) > n0  # the prompt batch outgrew the captured scratch
            del eng
    finally:
        lib.gemm_tuned_clear()
    assert outs[True] == outs[False]


def test_generate_cli_recompute_mode_on_gpu(tmp_path):
    from helpers import make_tokenizer

    hf = _hf("gpt2")
    hf.save_pretrained(str(tmp_path), safe_serialization=True)
    make_tokenizer(str(tmp_path), 101)  # ids < 101 of the 1000-entry vocabulary
    prompts = ["hello world", "this is a tiny"]
    outs = []
    for cache in ([], ["--use_cache"]):
        r = subprocess.run([sys.executable, "generate.py", "--pretrained_model_path", str(tmp_path), "--prompts",
                            *prompts, "--max_new_tokens", "8", "--is_greedy", "--device", "cuda", *cache],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        lines = r.stdout.strip().splitlines()
        assert lines[0].startswith("elapsed time: ") and lines[1] == f"prompts: {prompts}"
        outs.append(ast.literal_eval(lines[2][len("continuations: "):]))
        assert "cuda" in r.stdout  # the timing line names the device the run used
    assert outs[0] == outs[1]  # recompute (no cache) == paged-cache decode
