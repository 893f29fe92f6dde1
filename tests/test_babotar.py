"""Babotar through the framework (config reader, checkpoint loader, engine, scheduler, paged cache, state slots,
kernels) against the plain float64 definition in babotar_oracle.py. Every scenario runs on the CPU path in fp32 and,
on a GPU box, through the HIP kernels in fp32 and bf16. Small configurations made here, with sizes that differ
between layers and values that obvious choices would make equal or 1: grouped and single heads, value sizes unlike
key sizes, partial and full rotation with and without frequency scaling, one to four streams or none, convolutions
of one to four taps or none, layers without a feed-forward, no head mixing, no biases."""
import json
import os

import numpy as np
import pytest
import torch

import babotar_oracle as oracle
from llmss_amd.engine import LLMEngine, SamplingParams, build_model
from llmss_amd.models.config import ModelConfig
from llmss_amd.models.weights import babotar_state_dict

gpu = pytest.mark.gpu
RUNS = [pytest.param("cpu", "float32", id="cpu-fp32"), pytest.param("cuda", "float32", marks=gpu, id="gpu-fp32"),
        pytest.param("cuda", "bfloat16", marks=gpu, id="gpu-bf16")]


def left(heads, kv, dim, vdim, scale, softcap=None, rot=None):
    d = dict(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, scale=scale)
    if softcap:
        d["softcap"] = softcap
    if rot:
        d["rot"] = rot
    return d


def par(a, r, ls=1.0, rs=1.0, ff=None):
    return dict(type="parallel", mixer=dict(left=a, right=r, left_scale=ls, right_scale=rs),
                mlp=dict(kind="dense", ff=ff) if ff else None)


def lig(heads, dim, vdim, decay, ff=None):
    return dict(type="lightning", mixer=dict(heads=heads, dim=dim, vdim=vdim, decay=decay),
                mlp=dict(kind="dense", ff=ff) if ff else None)


YARN = dict(factor=4.0, original=32, fast=8.0, slow=1.0)
CONFIGS = {
    # three streams, four-tap input convolution; grouped heads on both sides; a decay layer first and one without a
    # feed-forward; partial rotation with scaled frequencies, then full rotation without
    "mixed": dict(architecture="Babotar", vocab=97, width=40, max_positions=160, norm=dict(eps=1e-5),
                  residual_mult=0.6, streams=3, canon=dict(taps=4), layers=[
        lig(3, 8, 12, [0.6, 0.9, 0.995], ff=56),
        par(left(4, 2, 8, 12, 0.3, softcap=20.0, rot=dict(base=500.0, dims=4, scaling=YARN)),
            dict(heads=4, kv_heads=2, dim=8, vdim=6, conv=3), 0.8, 1.2, ff=48),
        lig(2, 16, 4, [0.8, 0.99]),
        par(left(2, 1, 16, 8, 0.2, rot=dict(base=10000.0, dims=16)),
            dict(heads=2, kv_heads=2, dim=12, vdim=10, conv=2), 1.1, 0.7, ff=24),
    ]),
    # the ordinary residual (no streams, no multiplier), no input convolution, single heads, no rotation, no cap,
    # a convolution of one tap
    "plain": dict(architecture="Babotar", vocab=61, width=24, max_positions=160, norm=dict(eps=1e-6), layers=[
        par(left(1, 1, 8, 8, 0.35), dict(heads=1, kv_heads=1, dim=8, vdim=8, conv=1), ff=32),
        lig(1, 8, 8, [0.9], ff=16),
        par(left(3, 3, 8, 4, 0.3, softcap=5.0), dict(heads=3, kv_heads=1, dim=4, vdim=8, conv=4)),
    ]),
    # one stream with learned weights, two-tap input convolution; head sizes the kernels tile (64, 128, above 128)
    "wide": dict(architecture="Babotar", vocab=83, width=64, max_positions=160, norm=dict(eps=1e-6),
                 residual_mult=1.5, streams=1, canon=dict(taps=2), layers=[
        par(left(4, 2, 64, 128, 0.125, softcap=40.0, rot=dict(base=30000.0, dims=32, scaling=YARN)),
            dict(heads=2, kv_heads=1, dim=128, vdim=64, conv=4), 0.9, 0.9, ff=128),
        lig(2, 160, 72, [0.9, 0.999], ff=64),
    ]),
}
CONFIGS.update({
    # odd sizes everywhere (no dimension a multiple of 8), five streams, a rotation of two dimensions
    "odd": dict(architecture="Babotar", vocab=51, width=36, max_positions=160, norm=dict(eps=1e-5),
                residual_mult=0.9, streams=5, canon=dict(taps=2), layers=[
        par(left(6, 3, 6, 5, 0.4, softcap=8.0, rot=dict(base=50.0, dims=2, scaling=YARN)),
            dict(heads=3, kv_heads=3, dim=5, vdim=7, conv=3), 1.0, 1.0, ff=27),
        lig(5, 3, 9, [0.5, 0.7, 0.9, 0.95, 0.99], ff=19),
    ]),
    # no attention at all: nothing is paged, everything a sequence keeps lives in its state slot
    "decays": dict(architecture="Babotar", vocab=43, width=32, max_positions=160, norm=dict(eps=1e-5),
                   streams=2, layers=[lig(2, 8, 8, [0.7, 0.97], ff=40), lig(4, 4, 12, [0.5, 0.8, 0.9, 0.999])]),
})
DROP = {"plain": (".talk", ".q.b", ".k.b", ".v.b")}  # checkpoints without head mixing and without biases


class Case:
    def __init__(self, name, tmp, device, dtype, seed=0):
        self.cfg = CONFIGS[name]
        mc = ModelConfig.from_hf_dict(self.cfg)
        self.sd = {k: v for k, v in babotar_state_dict(mc, seed=seed).items()
                   if not k.endswith(DROP.get(name, ("\0",)))}
        d = tmp / f"{name}-{seed}"
        d.mkdir(exist_ok=True)
        from safetensors.torch import save_file

        save_file({k: v.contiguous() for k, v in self.sd.items()}, str(d / "model.safetensors"))
        (d / "config.json").write_text(json.dumps(self.cfg))
        self.path, self.device, self.dtype = str(d), device, dtype
        self.model = build_model(self.path, dtype=dtype, device=device)
        self.V = self.cfg["vocab"]
        self._ref = {}

    def engine(self, tokens=512, slots=4, block=16, **kw):
        return LLMEngine(self.model, max_num_seqs=slots, block_size=block, num_blocks=-(-tokens // block),
                         max_model_len=min(tokens, self.cfg["max_positions"]), max_batched_tokens=tokens,
                         use_graphs=kw.pop("use_graphs", False), autotune=False, **kw)

    def ref(self, tokens):
        key = tuple(tokens)
        if key not in self._ref:
            self._ref[key] = oracle.forward(self.cfg, self.sd, list(tokens))[0].float()
        return self._ref[key]

    def close(self, got, want, what=""):
        got, want = got.float().cpu(), want.float()
        d = (got - want) - (got - want).mean(-1, keepdim=True)
        err = d.pow(2).mean(-1).sqrt() / want.std(-1).clamp_min(1e-3)
        tol = 2e-4 if self.dtype == "float32" else 6e-2
        assert float(err.max()) < tol, f"{what}: relative error {float(err.max()):.3g} at row {int(err.argmax())}"


def toks(n, V, seed):
    return np.random.default_rng(seed).integers(0, V, n).tolist()


@pytest.fixture(scope="module")
def cases(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("babotar")
    made = {}

    def get(name, device, dtype):
        k = (name, device, dtype)
        if k not in made:
            made[k] = Case(name, tmp, device, dtype)
        return made[k]
    return get


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_whole_prompt_every_position(cases, name, device, dtype):
    c = cases(name, device, dtype)
    t = toks(45, c.V, 1)
    eng = c.engine()
    got = eng.replay_step([(0, t, list(range(len(t))))], end=[0])
    c.close(got, c.ref(t), "whole prompt")
    for n in (1, 2, 3):  # the first tokens of a sequence on their own, in the slot the last request left
        got = eng.replay_step([(n, t[:n], list(range(n)))], end=[n])
        c.close(got, c.ref(t[:n]), f"first {n} token(s)")


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_residual_stream_after_every_layer(cases, name, device, dtype):
    c = cases(name, device, dtype)
    t = toks(19, c.V, 2)
    want = oracle.forward(c.cfg, c.sd, t)[1]
    seen = {}
    c.model.tap = lambda i, x: seen.__setitem__(i, x.detach().float().cpu().clone())
    try:
        c.engine().replay_step([(0, t, [len(t) - 1])], end=[0])
    finally:
        c.model.tap = None
    assert sorted(seen) == list(range(len(want)))
    tol = 2e-4 if dtype == "float32" else 5e-2
    for i, w in enumerate(want):
        rel = (seen[i] - w.float()).abs().max() / w.abs().max()
        assert float(rel) < tol, f"layer {i}: {float(rel):.3g}"


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_prefill_against_token_by_token_decoding(cases, name, device, dtype):
    c = cases(name, device, dtype)
    t = toks(40, c.V, 3)
    eng = c.engine()
    rows = [eng.replay_step([(0, [tok], [0])]) for tok in t]  # every token decoded alone, from position 0 on
    eng.replay_step([], end=[0])
    c.close(torch.cat(rows), c.ref(t), "token by token")


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", ["mixed", "wide"])
@pytest.mark.parametrize("cuts", [(2, 2, 2, 3, 5, 16, 17, 2, 1, 1, 9), (15, 1, 16, 1, 17, 6), (33, 2, 21),
                                  (1, 2, 70, 2, 33, 1, 1, 30)])
def test_portions_of_several_sizes(cases, cuts, name, device, dtype):
    c = cases(name, device, dtype)
    t = toks(sum(cuts), c.V, 4)
    eng = c.engine()
    got, at = [], 0
    for n in cuts:
        got.append(eng.replay_step([(7, t[at:at + n], list(range(n)))]))
        at += n
    eng.replay_step([], end=[7])
    c.close(torch.cat(got), c.ref(t), f"portions {cuts}")


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", ["mixed", "plain", "wide"])
def test_mixed_batch_of_unequal_requests_equals_each_alone(cases, name, device, dtype):
    c = cases(name, device, dtype)
    seqs = {0: toks(50, c.V, 5), 1: toks(23, c.V, 6), 2: toks(9, c.V, 7), 3: toks(37, c.V, 8)}
    # per step: how many tokens of each request (0 = sits the step out); single tokens ride beside portions
    plan = [{0: 17, 1: 2}, {0: 1, 1: 5, 2: 9}, {0: 1, 1: 16, 3: 30}, {0: 31, 3: 1}, {3: 1, 1: 0}, {3: 5}]
    eng = c.engine(tokens=256)
    at = {k: 0 for k in seqs}
    got = {k: [] for k in seqs}
    for step in plan:
        entries, end = [], []
        for k, n in step.items():
            if n == 0:
                continue
            entries.append((k, seqs[k][at[k]:at[k] + n], list(range(n))))
            at[k] += n
            if at[k] == len(seqs[k]):
                end.append(k)
        out = eng.replay_step(entries, end)
        r = 0
        for k, tk, _ in entries:
            got[k].append(out[r:r + len(tk)])
            r += len(tk)
    assert at == {k: len(v) for k, v in seqs.items()}
    for k, t in seqs.items():
        c.close(torch.cat(got[k]), c.ref(t), f"request {k} in the mixed batch")


@pytest.mark.parametrize("device,dtype", RUNS)
def test_pages_and_state_slots_are_used_again(cases, device, dtype):
    c = cases("mixed", device, dtype)
    eng = c.engine(tokens=64, slots=2, block=16)  # 4 pages, 2 sequences with their state slots
    assert eng.sched.num_free_blocks() == 4
    used = set()
    for r in range(6):  # every round takes the pages and the slots that finished requests gave back
        a, b = toks(30 + r, c.V, 10 + r), toks(17, c.V, 20 + r)
        o1 = eng.replay_step([(2 * r, a[:20], [19]), (2 * r + 1, b, [16])], end=[2 * r + 1])
        used.add(eng.sched.state_slot(2 * r))
        assert eng.sched.num_free_blocks() == 2
        o2 = eng.replay_step([(2 * r, a[20:], list(range(len(a) - 20)))], end=[2 * r])
        assert eng.sched.num_free_blocks() == 4 and eng.sched.num_running() == 0
        c.close(o1, torch.stack([c.ref(a)[19], c.ref(b)[16]]), f"round {r}, first step")
        c.close(o2, c.ref(a)[20:], f"round {r}, second step")
    assert used <= {0, 1}
    with pytest.raises(RuntimeError):  # a third live request has no slot
        eng.replay_step([(100, [1], []), (101, [1], []), (102, [1], [])])
    with pytest.raises(RuntimeError):  # more tokens than the pool has pages for; nothing is taken
        eng.replay_step([(200, [1] * 40, []), (201, [1] * 40, [])])
    assert eng.sched.num_free_blocks() == 4 and eng.sched.num_running() == 0


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", ["mixed", "wide"])
def test_long_decoding_across_pages(cases, name, device, dtype):
    c = cases(name, device, dtype)
    t = toks(120, c.V, 30)
    eng = c.engine()
    got = [eng.replay_step([(0, t[:5], [4])])]
    got += [eng.replay_step([(0, [tok], [0])]) for tok in t[5:]]
    c.close(torch.cat(got), c.ref(t)[4:], "long decoding")


@pytest.mark.parametrize("device,dtype", RUNS)
@pytest.mark.parametrize("name", list(CONFIGS))
def test_greedy_generation_through_the_engine(cases, name, device, dtype):
    c = cases(name, device, dtype)
    prompts = [toks(11, c.V, 40), toks(3, c.V, 41), toks(26, c.V, 42)]
    eng = LLMEngine(c.model, max_num_seqs=4, block_size=16, num_blocks=32, max_model_len=128, max_batched_tokens=24,
                    prefill_chunk=7, autotune=False)  # its own scheduler cuts the prompts and batches the decodes
    out = eng.generate(prompts, SamplingParams(max_new_tokens=12, is_greedy=True, ignore_eos=True))
    for p, o in zip(prompts, out):
        want = oracle.greedy(c.cfg, c.sd, p, 12)
        if dtype == "float32":
            assert o == want
        else:  # bf16 may flip a near-tie; the tokens before the first difference must then be a true near-tie
            k = next((i for i, (x, y) in enumerate(zip(o, want)) if x != y), None)
            if k is not None:
                lg = oracle.forward(c.cfg, c.sd, p + want[:k])[0][-1]
                assert float(lg[want[k]] - lg[o[k]]) < 0.05 * float(lg.std())


@pytest.mark.parametrize("device,dtype", RUNS)
def test_preempted_requests_start_over_from_an_empty_state(cases, device, dtype):
    """A pool too small for all requests: the scheduler preempts (pages and state slot go back) and recomputes."""
    c = cases("mixed", device, dtype)
    prompts = [toks(20, c.V, 80), toks(18, c.V, 81), toks(22, c.V, 82)]
    eng = LLMEngine(c.model, max_num_seqs=3, block_size=8, num_blocks=9, max_model_len=64, max_batched_tokens=32,
                    autotune=False)
    out = eng.generate(prompts, SamplingParams(max_new_tokens=14, is_greedy=True, ignore_eos=True))
    assert eng.stats["preemptions"] > 0
    if dtype == "float32":
        for p, o in zip(prompts, out):
            assert o == oracle.greedy(c.cfg, c.sd, p, 14)


def test_config_reader_rejects_what_the_design_does_not_have():
    bad = json.loads(json.dumps(CONFIGS["plain"]))
    bad["layers"][0]["type"] = "convolution"
    with pytest.raises(ValueError):
        ModelConfig.from_hf_dict(bad)
    bad = json.loads(json.dumps(CONFIGS["plain"]))
    bad["layers"][1]["mixer"]["decay"] = [0.5, 0.6]  # two decays for one head
    with pytest.raises(ValueError):
        ModelConfig.from_hf_dict(bad)
    bad = json.loads(json.dumps(CONFIGS["mixed"]))
    bad["layers"][1]["mixer"]["left"]["kv_heads"] = 3  # does not divide the heads
    with pytest.raises(ValueError):
        ModelConfig.from_hf_dict(bad)
    bad = json.loads(json.dumps(CONFIGS["plain"]))
    bad["layers"][0]["mlp"]["kind"] = "moe"
    with pytest.raises(ValueError):
        ModelConfig.from_hf_dict(bad)


def test_loader_checks_shapes_against_the_config(cases, tmp_path):
    c = cases("plain", "cpu", "float32")
    cfg = json.loads(json.dumps(c.cfg))
    cfg["layers"][1]["mixer"]["vdim"] = 12
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    os.symlink(os.path.join(c.path, "model.safetensors"), tmp_path / "model.safetensors")
    with pytest.raises(ValueError):
        build_model(str(tmp_path), dtype="float32", device="cpu")


def test_cache_holds_pages_for_attention_and_state_for_recurrences(cases):
    c = cases("mixed", "cpu", "float32")
    kv = c.model.allocate_kv_cache(4, 16, num_slots=3)
    assert kv[0][0] is None and kv[0][2]["S"].shape == (3, 3, 8, 12)
    assert kv[1][0].shape == (4, 16, 2 * 8) and kv[1][1].shape == (4, 16, 2 * 12)
    assert kv[1][2]["S"].shape == (3, 4, 8, 6) and kv[1][2]["tail"].shape == (3, 2, 2 * 2 * 8 + 4 * 6)
    assert c.model.canon_tail.shape == (4, 3, 3, 40)
    assert c.model.kv_bytes_per_block(16) == 16 * 4 * (2 * (8 + 12) + 1 * (16 + 8))
    assert c.model.needs_state and c.model.state_bytes_per_slot() > 0
    with pytest.raises(ValueError):
        c.model.allocate_kv_cache(4, 16)


def test_trace_runner_replays_steps_on_the_cpu_path(cases, tmp_path):
    import subprocess
    import sys

    c = cases("plain", "cpu", "float32")
    t = toks(21, c.V, 50)
    steps = [dict(step=0, entries=[dict(id="a", tokens=t[:9], want=[0, 8])], end=[]),
             dict(step=1, entries=[dict(id="b", tokens=t[:2], want=[])], end=[]),
             dict(step=2, entries=[dict(id="a", tokens=t[9:], want=[11]), dict(id="b", tokens=t[2:3], want=[0])],
                  end=["a", "b"])]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", c.path, "--dtype", "float32",
                        "--out", str(tmp_path), "--max-tokens", "64", "--device", "cpu"],
                       input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [ln for ln in r.stdout.splitlines() if ln.startswith("done")] == ["done 0", "done 1", "done 2"]
    g0 = torch.from_numpy(np.fromfile(tmp_path / "0.f32", dtype="<f4").reshape(2, c.V))
    g2 = torch.from_numpy(np.fromfile(tmp_path / "2.f32", dtype="<f4").reshape(2, c.V))
    c.close(g0, c.ref(t)[[0, 8]], "step 0")
    c.close(g2, torch.stack([c.ref(t)[20], c.ref(t[:3])[2]]), "step 2")


def test_registry_facade_runs_the_design(cases):
    """MODEL_REGISTRY["babotar"](config, weights): HF-style calls with a growing paged past and a state slot."""
    from llmss_amd.models.registry import MODEL_REGISTRY, Weights
    from llmss_amd.utils.checkpoint import weight_files

    c = cases("mixed", "cpu", "float32")
    cfg = ModelConfig.from_pretrained(c.path)
    lm = MODEL_REGISTRY[cfg.model_type](cfg, Weights(weight_files(c.path), "cpu", torch.float32), max_blocks=16)
    t = toks(21, c.V, 60)
    out = lm(torch.tensor([t[:13]]), use_cache=True)
    c.close(out.logits[0], c.ref(t[:13]), "prompt through the facade")
    out2 = lm(torch.tensor([t[13:]]), past_key_values=out.past_key_values, use_cache=True)
    c.close(out2.logits[0], c.ref(t)[13:], "continuation through the facade")
    lm.release(out2.past_key_values)
    assert len(lm._free_state) == 16


@gpu
def test_decode_graphs_and_autotuned_projections_decode_right(cases):
    """Serving defaults on a GPU: GEMM plans timed per decode bucket, decode steps replayed from captured graphs
    (state slots ride in the graphs' static buffers), pipelined decode."""
    c = cases("wide", "cuda", "bfloat16")
    assert c.model.gemm_shapes()
    eng = LLMEngine(c.model, max_num_seqs=4, block_size=16, num_blocks=32, max_model_len=96, max_batched_tokens=64)
    assert eng.graphs
    prompts = [toks(9, c.V, 70), toks(17, c.V, 71), toks(2, c.V, 72)]
    outs = eng.generate(prompts, SamplingParams(max_new_tokens=10, is_greedy=True, ignore_eos=True))
    for p, out in zip(prompts, outs):
        want = oracle.greedy(c.cfg, c.sd, p, 10)
        k = next((i for i, (x, y) in enumerate(zip(out, want)) if x != y), None)
        if k is not None:
            lg = oracle.forward(c.cfg, c.sd, p + want[:k])[0][-1]
            assert float(lg[want[k]] - lg[out[k]]) < 0.05 * float(lg.std())


@gpu
def test_fp32_decode_graphs_reproduce_the_oracle_exactly(cases):
    c = cases("mixed", "cuda", "float32")
    eng = LLMEngine(c.model, max_num_seqs=4, block_size=16, num_blocks=32, max_model_len=96, max_batched_tokens=64,
                    autotune=False)
    assert eng.graphs
    prompts = [toks(9, c.V, 73), toks(30, c.V, 74), toks(1, c.V, 75)]
    outs = eng.generate(prompts, SamplingParams(max_new_tokens=20, is_greedy=True, ignore_eos=True))
    for p, out in zip(prompts, outs):
        assert out == oracle.greedy(c.cfg, c.sd, p, 20)


@pytest.mark.parametrize("width,ff,dtype,fused", [(64, 48, "bfloat16", True), (64, 32, "bfloat16", True), (96, 32, "bfloat16", False),
                                                  (64, 40, "bfloat16", False), (40, 48, "bfloat16", False), (64, 48, "float32", False)])
def test_rows_of_gate_and_up_alternate_where_the_epilogue_gates(width, ff, dtype, fused):
    """bf16, whole pieces and groups of 16, at least as many columns as K; the feed-forward gives the same either way."""
    from llmss_amd.models.layered import create_model
    from llmss_amd.models.weights import random_babotar_weights

    d = dict(architecture="Babotar", vocab=61, width=width, max_positions=64, norm=dict(eps=1e-6), layers=[lig(1, 8, 8, [0.9], ff=ff)])
    mc = ModelConfig.from_hf_dict(d)
    m = create_model(mc, random_babotar_weights(mc, dtype=getattr(torch, dtype), seed=3))
    W = m.w.layers[0].mlp
    assert W.interleaved == fused
    h = torch.randn(5, width, generator=torch.Generator().manual_seed(1)).to(getattr(torch, dtype))
    from llmss_amd.models.layered import DenseFeedForward

    got = DenseFeedForward.forward(m, W, mc.layer_specs[0].mlp, h).float()
    gu = W.gu.view(-1, 2, 16, width).transpose(0, 1).reshape(2 * ff, width) if fused else W.gu[:2 * ff]
    g, u = (h.float() @ gu.float().T).chunk(2, -1)
    want = (torch.nn.functional.gelu(g, approximate="tanh") * u) @ W.down.float().T
    # the gated row's rounding to bf16 and the result's (2^-9 each), the products' before the gate without the epilogue
    assert float((got - want).norm() / want.norm()) < (1e-5 if dtype == "float32" else 1.5e-2)
