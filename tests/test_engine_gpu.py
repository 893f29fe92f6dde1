"""End-to-end model/engine checks on the GPU: HIP forward vs the CPU fp32 reference forward,
HIP-graph decode vs eager decode, and continuous batching determinism."""
import gc

import pytest
import torch

from llmss_amd.engine import LLMEngine, SamplingParams
from llmss_amd.models.config import get_preset
from llmss_amd.models.decoder import DecoderLM, StepInput
from llmss_amd.models.weights import random_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nccl_world():
    """A one-member torch nccl process group for this file's tests; destroyed with its watchdog thread after the last of them."""
    import torch.distributed as dist

    assert not dist.is_initialized()
    dist.init_process_group("nccl", store=dist.HashStore(), rank=0, world_size=1, device_id=torch.device("cuda", 0))
    yield
    gc.collect()  # graphs that hold captured collectives go before their communicator
    torch.cuda.synchronize()
    dist.destroy_process_group()


def _to_gpu(w):
    from llmss_amd.models.weights import Linear, LayerWeights, ModelWeights

    def t(x, keep32=False):
        if x is None:
            return None
        return x.to("cuda", torch.float32 if keep32 else torch.bfloat16).contiguous()

    def lin(l):
        return Linear(t(l.w), t(l.b), None, l.glu)

    layers = [LayerWeights(t(L.ln1_w), t(L.ln1_b), t(L.ln2_w), t(L.ln2_b), lin(L.qkv), lin(L.o), lin(L.up), lin(L.down))
              for L in w.layers]
    return ModelWeights(t(w.wte), t(w.wpe), layers, t(w.lnf_w), t(w.lnf_b), lin(w.head),
                        t(w.cos, True), t(w.sin, True), rope_interleaved=w.rope_interleaved)


@pytest.mark.parametrize("name", ["tiny-gpt2", "tiny-gptj", "tiny-bigcode", "tiny-llama"])
def test_forward_matches_reference(name):
    over = {}
    if name == "tiny-gptj":
        over = dict(head_dim=64, hidden_size=256, num_heads=4, num_kv_heads=4, rotary_dim=16)
    else:
        over = dict(head_dim=64, hidden_size=256, num_heads=4, num_kv_heads=4 if name != "tiny-llama" else 2,
                    rotary_dim=64 if name == "tiny-llama" else 0)
        if name == "tiny-bigcode":
            over["num_kv_heads"] = 1
    cfg = get_preset(name, **over)
    wc = random_weights(cfg, device="cpu", dtype=torch.float32, seed=1, std=0.05)
    m_cpu = DecoderLM(cfg, wc)
    m_gpu = DecoderLM(cfg, _to_gpu(wc))
    T = 40
    ids = torch.randint(0, cfg.vocab_size, (T,))
    cu = torch.tensor([0, 25, T], dtype=torch.int32)
    pos = torch.cat([torch.arange(25), torch.arange(T - 25)])
    last = torch.tensor([24, T - 1])
    kv_c = m_cpu.allocate_kv_cache(16, 16)
    kv_g = m_gpu.allocate_kv_cache(16, 16)
    slots = torch.arange(T)
    ref = m_cpu(StepInput("prefill", ids, pos, slots, cu_seqlens=cu, max_seqlen=25, last_idx=last), kv_c)
    out = m_gpu(StepInput("prefill", ids.cuda(), pos.cuda(), slots.cuda(), cu_seqlens=cu.cuda(), max_seqlen=25,
                          last_idx=last.cuda()), kv_g)
    V = cfg.vocab_size
    _assert_logits_close(out[:, :V].float().cpu(), ref[:, :V])
    # single-sequence decode step after a prefill of 25 tokens
    dec_ids = torch.randint(0, V, (1,))
    kv_c = m_cpu.allocate_kv_cache(16, 16)
    kv_g = m_gpu.allocate_kv_cache(16, 16)
    ids1 = ids[:25]
    m_cpu(StepInput("prefill", ids1, torch.arange(25), torch.arange(25), cu_seqlens=torch.tensor([0, 25], dtype=torch.int32),
                    max_seqlen=25), kv_c)
    m_gpu(StepInput("prefill", ids1.cuda(), torch.arange(25).cuda(), torch.arange(25).cuda(),
                    cu_seqlens=torch.tensor([0, 25], dtype=torch.int32).cuda(), max_seqlen=25), kv_g)
    bt = torch.tensor([[0, 1]], dtype=torch.int32)
    ctx = torch.tensor([26], dtype=torch.int32)
    d_in = dict(kind="decode", input_ids=dec_ids[:1], positions=torch.tensor([25]), slots=torch.tensor([25]),
                block_tables=bt, ctx_lens=ctx, max_ctx=32)
    ref = m_cpu(StepInput(**d_in), kv_c)
    d_g = {k: (v.cuda() if torch.is_tensor(v) else v) for k, v in d_in.items()}
    out = m_gpu(StepInput(**d_g), kv_g)
    _assert_logits_close(out[:, :V].float().cpu(), ref[:, :V])


def _assert_logits_close(got, ref):
    """bf16 kernels vs the fp32 reference: per-row cosine > 0.999 and relative L2 error < 2%."""
    cos = torch.nn.functional.cosine_similarity(got, ref.float(), dim=-1).min().item()
    rel = ((got - ref).norm() / ref.norm()).item()
    assert cos > 0.999 and rel < 0.02, (cos, rel)


def _near_tie(m, ids, tol):
    """Top-2 logit margin of the next token after ``ids`` (one prefill on the GPU model) is below ``tol``."""
    T = len(ids)
    x = torch.tensor(ids, device="cuda")
    lg = m(StepInput("prefill", x, torch.arange(T, device="cuda"), torch.full((T,), -1, device="cuda"),
                     cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device="cuda"), max_seqlen=T,
                     last_idx=torch.tensor([T - 1], device="cuda")), m.allocate_kv_cache(8, 16))
    top2 = lg[0, :m.cfg.vocab_size].float().topk(2).values
    return (top2[0] - top2[1]).item() < tol


def test_engine_graph_vs_eager_and_batching():
    cfg = get_preset("tiny-llama", hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=256)
    w = random_weights(cfg, device="cuda", dtype=torch.bfloat16, seed=3, std=0.05)
    m = DecoderLM(cfg, w)
    prompts = [[int(x) for x in torch.randint(0, cfg.vocab_size, (n,))] for n in (5, 17, 33, 2, 60)]
    sp = SamplingParams(max_new_tokens=24, is_greedy=True, ignore_eos=True)
    e_graph = LLMEngine(m, max_num_seqs=8, block_size=16, use_graphs=True)
    out_g = e_graph.generate(prompts, sp)
    del e_graph
    e_eager = LLMEngine(m, max_num_seqs=8, block_size=16, use_graphs=False)
    out_e = e_eager.generate(prompts, sp)
    assert out_g == out_e
    # one-at-a-time == batched (continuous batching must not change greedy results); a lone prompt may run a
    # different GEMM kernel, so a flip is allowed only where the top-2 logit margin is within bf16 noise, and
    # that sequence is compared no further
    singles = [e_eager.generate([p], sp)[0] for p in prompts]
    for p, s1, s2 in zip(prompts, singles, out_e):
        k = next((i for i, (a, b) in enumerate(zip(s1, s2)) if a != b), None)
        if k is not None:
            assert _near_tie(m, p + s2[:k], 0.05), ("batched and single greedy runs differ at a clear margin", k)
    # sampled decoding is reproducible with fixed seeds
    sps = [SamplingParams(max_new_tokens=16, temperature=0.8, top_k=20, top_p=0.9, seed=11 + i, ignore_eos=True)
           for i in range(len(prompts))]
    a = e_eager.generate(prompts, sps)
    sps = [SamplingParams(max_new_tokens=16, temperature=0.8, top_k=20, top_p=0.9, seed=11 + i, ignore_eos=True)
           for i in range(len(prompts))]
    b = e_eager.generate(prompts, sps)
    assert a == b


def test_tp_allreduce_overlap_streams(nccl_world):
    """Row-chunked all-reduce on the comm stream (RCCL) overlapped with the next chunk's GEMMs must give
    the same hidden states as one all-reduce. A one-member RCCL group makes the collective the
    identity, so the multi-stream path runs for real on a single GPU."""
    import torch.distributed as dist

    from llmss_amd.parallel.dist import TPGroup

    tp = TPGroup(0, 2, group=dist.group.WORLD)  # rank-0 shard of a TP=2 plan, "real" communicator
    assert tp.is_real
    for fam, par in (("tiny-llama", False), ("tiny-gptj", True)):
        cfg = get_preset(fam, hidden_size=256, num_heads=4, head_dim=64, rotary_dim=64 if not par else 16,
                         intermediate_size=512, max_position_embeddings=256,
                         **({"num_kv_heads": 2} if not par else {}))
        assert cfg.parallel_block == par
        m = DecoderLM(cfg, random_weights(cfg, 2, 0, device="cuda", dtype=torch.bfloat16, seed=1, std=0.05), tp)
        T = 120
        kv = m.allocate_kv_cache(16, 16)
        pos = torch.cat([torch.arange(50), torch.arange(70)]).to("cuda")
        inp = StepInput(kind="prefill", input_ids=torch.randint(0, cfg.vocab_size, (T,), device="cuda"),
                        positions=pos, slots=torch.arange(T, device="cuda"),
                        cu_seqlens=torch.tensor([0, 50, T], dtype=torch.int32, device="cuda"), max_seqlen=70)
        m.overlap_rows = 1 << 30
        ref = m.hidden_states(inp, kv)
        m.overlap_rows = 32
        out = m.hidden_states(inp, kv)
        torch.cuda.synchronize()
        assert m._comm_stream is not None
        err = (out.float() - ref.float()).abs().max().item()
        assert err < 5e-2, err


def test_rccl_collectives_inside_decode_graphs(nccl_world):
    """Capture smoke test (torch process-group mode, LLMSS_COMM=torch): the TP decode step with its
    all-reduces + all-gather through torch's RCCL process group captures into HIP graphs and replays ==
    eager. The communicator has ONE member, so its in-place all-reduces move no data and need not leave a
    node in the graph: this proves capture works, not that a multi-rank collective is in the graph (that is
    measured by bench.py's comm probe on the driver's multi-GPU node)."""
    import torch.distributed as dist

    from llmss_amd.parallel.dist import TPGroup

    class OneMemberTP(TPGroup):  # TP=2 shard plan over a 1-rank communicator (collectives run, sum = identity)
        def all_gather_last_dim(self, t):
            out = torch.empty((t.shape[0],) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
            dist.all_gather_into_tensor(out, t.contiguous(), group=self.group)
            return torch.cat([out, out], -1)

    tp = OneMemberTP(0, 2, group=dist.group.WORLD)
    cfg = get_preset("tiny-llama", hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=256)
    m = DecoderLM(cfg, random_weights(cfg, 2, 0, device="cuda", dtype=torch.bfloat16, seed=3, std=0.05), tp)
    prompts = [[int(x) for x in torch.randint(0, cfg.vocab_size, (n,))] for n in (5, 17, 33)]
    sp = SamplingParams(max_new_tokens=12, is_greedy=True, ignore_eos=True)
    e_graph = LLMEngine(m, max_num_seqs=4, block_size=16, use_graphs=True, autotune=False)
    assert e_graph.use_graphs and len(e_graph.graphs) > 0  # capture with RCCL collectives succeeded
    out_g = e_graph.generate(prompts, sp)
    del e_graph
    e_eager = LLMEngine(m, max_num_seqs=4, block_size=16, use_graphs=False, autotune=False)
    assert e_eager.generate(prompts, sp) == out_g


@pytest.mark.skip(reason="captures a collective right behind eager ones without the wait for the process group's watchdog that "
                         "the engine's captures have (TPGroup.settle): the watchdog may query an event of the stream that the "
                         "capture holds (hipErrorCapturedEvent), which ended the test process in one of eight runs")
def test_graph_capture_while_rccl_watchdog_polls(nccl_world):
    """Capture smoke regression (torch process-group mode): with the RCCL process group's watchdog thread
    tracking earlier collectives, a capture in torch's default (global) mode aborted the process when the
    watchdog queried an event mid-capture ("operation not permitted when stream is capturing"). Engine and
    autotuner capture thread-locally. One member: the captured in-place all-reduce is empty (HIP warns
    "The CUDA Graph is empty"); the test is about the watchdog, not the collective."""
    import torch.distributed as dist

    from llmss_amd.ops import autotune as A

    t = torch.ones(1 << 16, device="cuda")
    for i in range(60):
        for _ in range(4):  # eager collectives: work items the watchdog polls
            dist.all_reduce(t)
        A._time(lambda j: dist.all_reduce(t), 4)  # captures with a collective inside
    torch.cuda.synchronize()
    assert torch.isfinite(t).all()


def _one_member_tp():
    import torch.distributed as dist

    from llmss_amd.parallel.dist import TPGroup

    class OneMemberTP(TPGroup):  # TP=2 shard plan over a 1-rank communicator (collectives run, sum = identity)
        def all_gather_last_dim(self, t):
            out = torch.empty((t.shape[0],) + tuple(t.shape[1:]), dtype=t.dtype, device=t.device)
            dist.all_gather_into_tensor(out, t.contiguous(), group=self.group)
            return torch.cat([out, out], -1)

    return OneMemberTP(0, 2, group=dist.group.WORLD)


@pytest.mark.parametrize("fam", ["tiny-llama", "tiny-gptj"])
def test_decode_microbatch_overlap(fam, nccl_world):
    """Two-micro-batch decode (each half's RCCL all-reduces on the comm stream while the other half
    computes) == the single-batch decode step, for sequential (Llama) and parallel (GPT-J) blocks."""
    tp = _one_member_tp()
    par = fam == "tiny-gptj"
    cfg = get_preset(fam, hidden_size=256, num_heads=4, head_dim=64, rotary_dim=16 if par else 64,
                     intermediate_size=512, max_position_embeddings=256, **({} if par else {"num_kv_heads": 2}))
    m = DecoderLM(cfg, random_weights(cfg, 2, 0, device="cuda", dtype=torch.bfloat16, seed=4, std=0.05), tp)
    bs, nseq, per = 16, 24, 4  # 24 sequences, 4 blocks (64 tokens) each
    kv = m.allocate_kv_cache(nseq * per, bs)
    lens = [5 + (7 * i) % 40 for i in range(nseq)]
    ids = torch.randint(0, cfg.vocab_size, (sum(lens),), device="cuda")
    pos = torch.cat([torch.arange(n) for n in lens]).cuda()
    slots = torch.cat([torch.arange(n) + i * per * bs for i, n in enumerate(lens)]).cuda()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device="cuda")
    m.hidden_states(StepInput("prefill", ids, pos, slots, cu_seqlens=cu, max_seqlen=max(lens)), kv)
    bt = torch.arange(nseq * per, dtype=torch.int32, device="cuda").view(nseq, per)
    L = torch.tensor(lens, device="cuda")
    dec = StepInput("decode", torch.randint(0, cfg.vocab_size, (nseq,), device="cuda"), L.clone(),
                    L + torch.arange(nseq, device="cuda") * per * bs, block_tables=bt,
                    ctx_lens=(L + 1).to(torch.int32), max_ctx=per * bs)
    m.tbo_min = 0
    ref = m.hidden_states(dec, kv)
    m.tbo_min = 2
    assert m.overlap_split(nseq) == 12
    out = m.hidden_states(dec, kv)  # rewrites the same KV slots with the same values
    torch.cuda.synchronize()
    err = (out.float() - ref.float()).abs().max().item()
    assert err < 5e-2, err


@pytest.mark.parametrize("fam", ["tiny-llama", "tiny-gptj"])
def test_prefill_microbatch_overlap(fam, nccl_world):
    """Prefill split into two micro-batches at a sequence boundary (each half's RCCL all-reduces on the comm
    stream while the other half computes) == the single prefill step: hidden states and the paged KV."""
    tp = _one_member_tp()
    par = fam == "tiny-gptj"
    cfg = get_preset(fam, hidden_size=256, num_heads=4, head_dim=64, rotary_dim=16 if par else 64,
                     intermediate_size=512, max_position_embeddings=256, **({} if par else {"num_kv_heads": 2}))
    m = DecoderLM(cfg, random_weights(cfg, 2, 0, device="cuda", dtype=torch.bfloat16, seed=6, std=0.05), tp)
    bs, per = 16, 4
    lens = [37, 5, 64, 18, 51, 9]
    ids = torch.randint(0, cfg.vocab_size, (sum(lens),), device="cuda")
    pos = torch.cat([torch.arange(n) for n in lens]).cuda()
    slots = torch.cat([torch.arange(n) + i * per * bs for i, n in enumerate(lens)]).cuda()
    cu_host = [0] + [int(c) for c in torch.tensor(lens).cumsum(0)]
    inp = StepInput("prefill", ids, pos, slots, cu_seqlens=torch.tensor(cu_host, dtype=torch.int32, device="cuda"),
                    max_seqlen=max(lens), cu_host=cu_host)
    kv_a, kv_b = m.allocate_kv_cache(len(lens) * per, bs), m.allocate_kv_cache(len(lens) * per, bs)
    m.tbo_prefill_min = 0
    ref = m.hidden_states(inp, kv_a)
    m.tbo_prefill_min = 16
    assert m.prefill_split(inp) == (3, 106)
    out = m.hidden_states(inp, kv_b)
    torch.cuda.synchronize()
    assert (out.float() - ref.float()).abs().max().item() < 5e-2
    for (ka, va), (kb, vb) in zip(kv_a, kv_b):  # half-batch GEMMs may pick other split-K plans: bf16 tolerance
        assert (ka.float() - kb.float()).abs().max().item() < 5e-2 and (va.float() - vb.float()).abs().max() < 5e-2


def test_decode_microbatch_overlap_in_graphs(nccl_world):
    """The micro-batch decode schedule (two streams, event joins, RCCL) captures into HIP graphs and
    replays exactly like eager; also with the modelled-comm fake group used by bench --sim-comm."""
    from llmss_amd.parallel.dist import TPGroup

    cfg = get_preset("tiny-llama", hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=256)
    w = random_weights(cfg, 2, 0, device="cuda", dtype=torch.bfloat16, seed=3, std=0.05)
    prompts = [[int(x) for x in torch.randint(0, cfg.vocab_size, (n,))] for n in (5, 17, 33, 9, 12, 40, 3, 21)]
    sp = SamplingParams(max_new_tokens=10, is_greedy=True, ignore_eos=True)
    for tp in (_one_member_tp(), TPGroup(0, 2, fake=True, sim_comm=(3.0, 100.0))):
        m = DecoderLM(cfg, w, tp)
        m.tbo_min = 4
        e_graph = LLMEngine(m, max_num_seqs=8, block_size=16, use_graphs=True, autotune=False)
        assert e_graph.use_graphs and len(e_graph.graphs) > 0
        assert 4 in e_graph.decode_batch_sizes()  # halves of the 8-row bucket
        out_g = e_graph.generate(prompts, sp)
        del e_graph
        e_eager = LLMEngine(m, max_num_seqs=8, block_size=16, use_graphs=False, autotune=False)
        assert e_eager.generate(prompts, sp) == out_g


def _async_engine_run(m, prompts, sps, async_decode, eos=None, abort_after=None):
    # one graph bucket: every decode step runs M = 8 rows, so a row's numerics never depend on how
    # many other rows are live (sync and async modes shrink the batch at different steps)
    eng = LLMEngine(m, max_num_seqs=8, block_size=4, use_graphs=True, autotune=False, eos_token_id=eos,
                    graph_buckets=[8])
    eng.async_decode = async_decode
    rids = [eng.add_request(p, sp) for p, sp in zip(prompts, sps)]
    n = 0
    while eng.has_unfinished():
        eng.step()
        n += 1
        if abort_after is not None and n == abort_after:
            eng.abort(rids[0])
    out = {r.id: (list(r.output_ids), r.finish_reason) for r in eng.pop_finished()}
    return [out[r] for r in rids]


def test_async_decode_matches_sync():
    """Pipelined decode (next step launched before the current one is collected, device-side input
    ids, dropped rows for EOS stops) produces exactly the tokens of the synchronous engine: staggered
    max_new_tokens, KV block boundaries every 4 tokens, sampling, EOS stops and an abort."""
    cfg = get_preset("tiny-llama", hidden_size=256, num_heads=4, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=256, vocab_size=64)
    m = DecoderLM(cfg, random_weights(cfg, device="cuda", dtype=torch.bfloat16, seed=5, std=0.08))
    g = torch.Generator().manual_seed(0)
    prompts = [torch.randint(0, 64, (n,), generator=g).tolist() for n in (3, 9, 5, 14, 6, 2, 11, 7)]
    sps = [SamplingParams(max_new_tokens=4 + 3 * i, temperature=0.9, top_k=20, top_p=0.9, seed=100 + i)
           for i in range(len(prompts))]
    ref = _async_engine_run(m, prompts, sps, False)
    assert _async_engine_run(m, prompts, sps, True) == ref
    # EOS: the most frequent generated token stops sequences mid-stream
    toks = [t for o, _ in ref for t in o]
    eos = max(set(toks), key=toks.count)
    ref_e = _async_engine_run(m, prompts, sps, False, eos=eos)
    assert any(r == "eos" for _, r in ref_e)
    assert _async_engine_run(m, prompts, sps, True, eos=eos) == ref_e
    # abort mid-run: every other request is unaffected
    a = _async_engine_run(m, prompts, sps, False, abort_after=4)
    b = _async_engine_run(m, prompts, sps, True, abort_after=4)
    assert a[0][1] == b[0][1] == "abort"
    assert a[1:] == b[1:] == ref[1:]


@pytest.mark.parametrize("kv_heads", [1, 2])
def test_gqa_decode_on_mfma_extend_kernel(kv_heads):
    """GQA / MQA decode attention routed through the MFMA extend kernel (DecoderLM.gqa_mfma) == the VALU
    split-K decode kernel, on a decode step after a prefill; and the engine's timed choice decodes the same
    greedy tokens as the eager VALU path up to near-ties."""
    cfg = get_preset("tiny-llama", hidden_size=512, num_heads=8, num_kv_heads=kv_heads, head_dim=64, rotary_dim=64,
                     intermediate_size=512, max_position_embeddings=512)
    m = DecoderLM(cfg, random_weights(cfg, device="cuda", dtype=torch.bfloat16, seed=9, std=0.05))
    B, T0 = 6, 37
    kv = m.allocate_kv_cache(64, 16)
    ids = torch.randint(0, cfg.vocab_size, (B * T0,), device="cuda")
    pos = torch.arange(T0, device="cuda").repeat(B)
    slots = torch.cat([torch.arange(T0, device="cuda") + 16 * 4 * i for i in range(B)])
    cu = torch.arange(0, B * T0 + 1, T0, dtype=torch.int32, device="cuda")
    m(StepInput("prefill", ids, pos, slots, cu_seqlens=cu, max_seqlen=T0, last_idx=cu[1:].long() - 1), kv)
    bt = torch.stack([torch.arange(4 * i, 4 * i + 4, dtype=torch.int32) for i in range(B)]).cuda()
    dec = dict(kind="decode", input_ids=torch.randint(0, cfg.vocab_size, (B,), device="cuda"),
               positions=torch.full((B,), T0, device="cuda"), slots=torch.tensor([64 * i + T0 for i in range(B)],
                                                                                 device="cuda"),
               block_tables=bt, ctx_lens=torch.full((B,), T0 + 1, dtype=torch.int32, device="cuda"), max_ctx=64)
    m.gqa_mfma = set()
    ref = m(StepInput(**dec), kv).float()
    m.gqa_mfma = {B}
    got = m(StepInput(**dec), kv).float()
    m.gqa_mfma = set()
    _assert_logits_close(got.cpu(), ref.cpu())
    cos = torch.nn.functional.cosine_similarity(got, ref, dim=-1).min().item()
    assert cos > 0.9999, cos


def test_fp8_norm_twin_matches_separate_quantisation():
    """add_norm's per-token fp8 twin (fp8_out) feeds the W8A8 GEMMs exactly what their own quantisation launch
    would: a W8A8 prefill (M > 128 rows) gives bit-identical logits with and without the fused twin."""
    cfg = get_preset("tiny-llama", hidden_size=512, num_heads=8, num_kv_heads=2, head_dim=64, rotary_dim=64,
                     intermediate_size=1024, max_position_embeddings=512)
    m = DecoderLM(cfg, random_weights(cfg, device="cuda", dtype=torch.bfloat16, seed=4, std=0.05, fp8=True))
    assert m.w.layers[0].qkv.w_scale is not None
    T = 200
    ids = torch.randint(0, m.cfg.vocab_size, (T,), device="cuda")
    inp = StepInput("prefill", ids, torch.arange(T, device="cuda"), torch.full((T,), -1, device="cuda"),
                    cu_seqlens=torch.tensor([0, T], dtype=torch.int32, device="cuda"), max_seqlen=T,
                    last_idx=torch.tensor([T - 1], device="cuda"))
    kv = m.allocate_kv_cache(16, 16)
    m._norm_quant = False
    ref = m(inp, kv).float()
    m._norm_quant = True
    got = m(inp, kv).float()
    assert torch.equal(got, ref)


def test_pipelined_decode_across_kv_block_boundaries():
    """The pipelined decode launches step t+1 before collecting step t, also when a sequence enters a new KV
    block (the block is reserved ahead of the scheduler: Scheduler.reserve). Greedy tokens equal the
    un-pipelined engine's, with 4-token pages so nearly every fourth step crosses a boundary."""
    cfg = get_preset("tiny-llama", head_dim=64, hidden_size=256, num_heads=4, num_kv_heads=2, rotary_dim=64)
    w = _to_gpu(random_weights(cfg, device="cpu", dtype=torch.float32, seed=3, std=0.05))
    prompts = [[(5 * i + j) % cfg.vocab_size for j in range(3 + 2 * i)] for i in range(6)]
    sp = SamplingParams(max_new_tokens=23, is_greedy=True, ignore_eos=True)
    outs = []
    for pipelined in (True, False):
        eng = LLMEngine(DecoderLM(cfg, w), max_num_seqs=8, block_size=4, num_blocks=96, max_model_len=64,
                        autotune=False)
        eng.async_decode = pipelined
        outs.append(eng.generate(prompts, sp))
        if pipelined:
            assert eng.stats.get("spec_block_reserves", 0) > 0
    assert outs[0] == outs[1]

