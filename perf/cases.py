"""What users of this framework have it do, as cases that can be timed and checked.

Five model families in the sizes of the repository's own benchmarks, random weights under checkpoint names, bf16:
gpt2 (GPT-2-XL layers), llama (Llama-2-7B layers; also with fp8 weights and an fp8 cache), and three per-layer designs -
babotar (linear attention with constant decay, sink attention beside a gated delta rule, residual streams), fizelix
(pooled window attention, state space, experts, a looped stretch) and nolavik (gated delta rule, attention beside a
selective scan, latent attention, experts).

What a pass does (``do``):

* ``prompts``: one step over whole prompts, as the engine runs admitted requests: the rows after the final norm, the
  logits of every prompt's last token, and the per-sequence states that later steps start from.
* ``decode``: one step of single tokens behind cached contexts, in a HIP graph, as the engine replays them.
* ``mixed``: portions that continue cached prefixes beside single tokens (chunked prefill).
* ``answers``: prompts in one step, then ``steps`` single-token steps in a HIP graph with given tokens - a burst of
  short requests answered. This is how the designs with per-sequence state decode here: a single step could not be
  repeated, because it moves the state on.

Every step goes through the model surface the engine itself uses (``create_model``, ``allocate_kv_cache``, ``StepInput``,
``hidden_states``, ``logits``). Weights, cache pages and captured graphs are what a serving process keeps.
"""
import math
import random

import torch

F64 = torch.float64
BLOCK = 16  # cache positions per page
VOCAB = 32000
EPS = 1e-6


# ------------------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one user, one conversation: the smallest step, latency and launches
        dict(name="gpt2_decode_1", family="gpt2", do="decode", width=1600, layers=4, batch=1, longest=100, ragged=False),
        # the benchmark's decode step: 64 sequences at the mean context of 128 + 128 tokens
        dict(name="llama_decode_64", family="llama", do="decode", width=4096, layers=2, batch=64, longest=192, ragged=False),
        # quantised serving of longer conversations, an odd batch
        dict(name="llama_decode_fp8", family="llama", do="decode", width=4096, layers=2, batch=23, longest=1777, ragged=True,
             fp8=True),
        # the benchmark's prompt step
        dict(name="llama_prompts_64x128", family="llama", do="prompts", width=4096, layers=2, batch=64, longest=128,
             ragged=False),
        # one document, an odd length: attention's share grows
        dict(name="llama_prompt_3999", family="llama", do="prompts", width=4096, layers=2, batch=1, longest=3999,
             ragged=False),
        # chunked prefill: two portions behind cached prefixes ride along with running conversations
        dict(name="llama_mixed", family="llama", do="mixed", width=4096, layers=2, batch=2, longest=1900, ragged=True,
             decodes=31),
        # prompt steps of the per-layer designs at the size their benchmarks quote
        dict(name="babotar_prompts", family="babotar", do="prompts", width=2048, batch=8, longest=1024, ragged=False),
        dict(name="fizelix_prompts", family="fizelix", do="prompts", width=2048, batch=8, longest=1024, ragged=False),
        dict(name="nolavik_prompts", family="nolavik", do="prompts", width=2048, batch=7, longest=1433, ragged=True),
        # short requests answered: decode steps of the designs with per-sequence state
        dict(name="babotar_answers", family="babotar", do="answers", width=2048, batch=64, longest=24, ragged=False, steps=8),
        dict(name="fizelix_answers", family="fizelix", do="answers", width=2048, batch=33, longest=31, ragged=True, steps=8),
        dict(name="nolavik_answers", family="nolavik", do="answers", width=1024, batch=8, longest=16, ragged=False, steps=8),
    ]


def draw(rng: random.Random):
    def spread(lo, hi):  # evenly over the logarithm
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))
    family = rng.choice(["gpt2", "llama", "babotar", "babotar", "fizelix", "fizelix", "nolavik", "nolavik"])
    c = dict(family=family, ragged=rng.random() < 0.5)
    if family in ("gpt2", "llama"):
        c.update(width=1600 if family == "gpt2" else 4096, layers=4 if family == "gpt2" else 2,
                 do=rng.choice(["decode", "prompts", "mixed"]))
        top = 1000 if family == "gpt2" else 3999
        if c["do"] == "decode":
            c.update(batch=spread(1, 64), longest=spread(16, min(top, 1777)))
            if family == "llama" and rng.random() < 0.3:
                c.update(fp8=True, batch=spread(1, 23))
        else:
            tokens = spread(32, 8192)
            c["longest"] = min(top, spread(16, tokens))
            c["batch"] = max(1, min(64, tokens // c["longest"]))
            if c["do"] == "mixed":
                c.update(batch=min(2, c["batch"]), longest=max(64, min(c["longest"], 1900)), decodes=spread(1, 31))
    else:
        c.update(width=rng.choice([1024, 2048]), do=rng.choice(["prompts", "answers"]))
        if c["do"] == "prompts":
            tokens = spread(64, 8192)
            c["longest"] = min(2048, spread(16, tokens))
            c["batch"] = max(1, min(64, tokens // c["longest"]))
        else:
            c.update(batch=spread(1, 64), longest=spread(2, 31), steps=8)
    return c


def lengths(case):
    """Prompt (or context) length of every sequence."""
    n, top = case["batch"], case["longest"]
    if not case["ragged"]:
        return [top] * n
    return [max(1, top - (top * 2 * i * i) // (3 * n * n)) for i in range(n)]


def tolerance(case):
    """Two correct bf16 implementations differ by the roundings of the rows between the operations: 0.4 % each, a few
    dozen of them on the way to the logits (0.5 to 1 % off the same in 64 bits, a state after a few layers 1.2 %)."""
    return {"rel": 0.02, "max": 0.5}


# ------------------------------------------------------------------------------------------------ model descriptions
def describe(case):
    """The config.json dictionary of the case's model."""
    w = case["width"]
    if case["family"] == "gpt2":
        return dict(model_type="gpt2", n_embd=w, n_layer=case["layers"], n_head=w // 64, n_positions=1024, vocab_size=50257)
    if case["family"] == "llama":
        return dict(model_type="llama", hidden_size=w, num_hidden_layers=case["layers"], num_attention_heads=w // 128,
                    num_key_value_heads=w // 128, intermediate_size=11008, vocab_size=VOCAB, max_position_embeddings=4096,
                    rms_norm_eps=EPS)
    heads, kv, norm = w // 128, w // 512, dict(eps=EPS)
    if case["family"] == "babotar":
        mlp = dict(kind="dense", ff=w * 11 // 4)
        left = dict(heads=heads, kv_heads=kv, dim=128, vdim=128, scale=128 ** -0.5, softcap=30.0,
                    rot=dict(base=10000.0, dims=64, scaling=dict(factor=4.0, original=4096, fast=16.0, slow=2.0)))
        right = dict(heads=heads, kv_heads=heads // 2, dim=64 if w == 1024 else 128, vdim=128, conv=4)
        par = dict(type="parallel", mlp=mlp, mixer=dict(left=left, right=right, left_scale=1.0, right_scale=1.0))
        decay = [1.0 - 2.0 ** (-3 - 5 * i / (heads - 1)) for i in range(heads)]
        lig = dict(type="lightning", mlp=mlp, mixer=dict(heads=heads, dim=128, vdim=128, decay=decay))
        return dict(architecture="Babotar", vocab=VOCAB, width=w, max_positions=4096, norm=norm, residual_mult=1.0, streams=2,
                    canon=dict(taps=4), layers=[par, par, lig, par])
    experts = dict(kind="moe", router=dict(experts=w // 64, top=w // 512), expert=dict(ff=512 if w == 1024 else 768))
    if case["family"] == "fizelix":
        experts["shared"] = dict(ff=1024)
        dense = dict(kind="dense", ff=2 * w)
        att = dict(heads=heads, kv_heads=kv, dim=128, vdim=128, scale=128 ** -0.5, mask=dict(size=512, pool=16),
                   rot=dict(base=10000.0, dims=64))
        ssd = dict(heads=w // 32, vdim=64, state=128, groups=1, conv=4, norm_groups=1)
        return dict(architecture="Fizelix", vocab=VOCAB, width=w, norm=norm, embedding=dict(scale=1.0), logit_scale=1.0,
                    token_side=dict(dim=32), loop=dict(start=1, stop=3, times=2),
                    layers=[dict(type="attention", mixer=att, mlp=dense), dict(type="mamba2", mixer=ssd, mlp=experts),
                            dict(type="attention", mixer=att, mlp=experts), dict(type="attention", mixer=att, mlp=dense)])
    experts["shared"] = dict(ff=512 if w == 1024 else 768)
    delta = dict(type="delta", mlp=experts, mixer=dict(heads=heads, kv_heads=heads // 2, dim=128, vdim=128, conv=4))
    left = dict(heads=heads, kv_heads=kv, dim=128, vdim=128, scale=128 ** -0.5,
                rot=dict(base=500000.0, dims=128, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192)))
    right = dict(inner=2 * w, state=16, dt_rank=w // 16, conv=4)
    par = dict(type="parallel", mlp=experts, mixer=dict(left=left, right=right, left_scale=0.7, right_scale=0.6))
    lat = dict(type="latent_attention", mlp=experts,
               mixer=dict(heads=heads, dim=128, rot_dim=64, vdim=128, q_rank=w * 3 // 8, kv_rank=192, scale=192 ** -0.5,
                          rot=dict(base=10000.0, dims=64)))
    return dict(architecture="Nolavik", vocab=VOCAB, width=w, norm=norm, loop=dict(start=0, stop=2, times=1),
                layers=[delta, par, lat, delta])


def runs(d):
    """Layer indices in the order they run (a looped stretch repeats)."""
    n, lp = len(d["layers"]), d.get("loop")
    if not lp:
        return list(range(n))
    a, b = lp["start"], lp["stop"]
    return list(range(a)) + list(range(a, b)) * lp["times"] + list(range(b, n))


def shapes(d):
    """Checkpoint tensor names of a model and their shapes."""
    if d.get("model_type") == "gpt2":
        w, out = d["n_embd"], {"wte.weight": (d["vocab_size"], d["n_embd"]), "wpe.weight": (d["n_positions"], d["n_embd"])}
        for i in range(d["n_layer"]):
            p = f"h.{i}."
            for n, a, b in (("attn.c_attn", w, 3 * w), ("attn.c_proj", w, w), ("mlp.c_fc", w, 4 * w), ("mlp.c_proj", 4 * w, w)):
                out.update({p + n + ".weight": (a, b), p + n + ".bias": (b,)})
            for n in ("ln_1", "ln_2"):
                out.update({p + n + ".weight": (w,), p + n + ".bias": (w,)})
        out.update({"ln_f.weight": (w,), "ln_f.bias": (w,)})
        return out
    if d.get("model_type") == "llama":
        w, f = d["hidden_size"], d["intermediate_size"]
        out = {"model.embed_tokens.weight": (VOCAB, w), "model.norm.weight": (w,), "lm_head.weight": (VOCAB, w)}
        for i in range(d["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + f"self_attn.{n}_proj.weight": (w, w) for n in "qkvo"})
            out.update({p + "mlp.gate_proj.weight": (f, w), p + "mlp.up_proj.weight": (f, w), p + "mlp.down_proj.weight": (w, f),
                        p + "input_layernorm.weight": (w,), p + "post_attention_layernorm.weight": (w,)})
        return out
    w, fam = d["width"], d["architecture"]
    out = {"embed": (VOCAB, w), "final.norm": (w,), "head": (VOCAB, w)}
    if fam == "Babotar":
        out["pos"] = (d["max_positions"], w)
    if fam == "Fizelix":
        out["side.embed"] = (VOCAB, len(d["layers"]) * d["token_side"]["dim"])
    if fam == "Nolavik":
        out["loop.step"] = (d["loop"]["times"], w)

    def attention(p, m):
        out.update({p + "q": (m["heads"] * m["dim"], w), p + "k": (m["kv_heads"] * m["dim"], w),
                    p + "v": (m["kv_heads"] * m["vdim"], w), p + "o": (w, m["heads"] * m["vdim"])})

    def delta(p, m):
        for n, c in (("q", m["kv_heads"] * m["dim"]), ("k", m["kv_heads"] * m["dim"]), ("v", m["heads"] * m["vdim"])):
            out.update({p + n: (c, w), p + n + ".conv": (c, m["conv"])})
        out.update({p + "g": (m["heads"] * m["vdim"], w), p + "o": (w, m["heads"] * m["vdim"]), p + "norm": (m["vdim"],)})
        out.update({p + n: (m["heads"], w) for n in "ab"})
        out.update({p + n: (m["heads"],) for n in ("A_log", "dt_bias")})

    def gated(p, ff):
        out.update({p + "gate": (ff, w), p + "up": (ff, w), p + "down": (w, ff)})
    for i, L in enumerate(d["layers"]):
        p, q, m, f = f"l{i}.", f"l{i}.mix.", L["mixer"], L["mlp"]
        out.update({p + "norm1": (w,), p + "norm2": (w,)})
        if fam == "Babotar":
            out[p + "canon1"] = (w, d["canon"]["taps"])
            for k in "12":
                out.update({f"{p}hc{k}.in": (2,), f"{p}hc{k}.out": (2,), f"{p}hc{k}.mix": (2, 2)})
        else:
            out.update({p + "norm1b": (w,), p + "norm2b": (w,)})
        if fam == "Fizelix":
            for k in "12":
                out.update({p + "ls" + k: (w,), p + "rg" + k: (w, w), p + f"rg{k}.b": (w,)})
            s = d["token_side"]["dim"]
            out.update({p + "side.gate": (s, w), p + "side.proj": (w, s), p + "side.norm": (w,)})
        if L["type"] == "lightning":
            out.update({q + n: (m["heads"] * m["dim"], w) for n in "qkvg"})
            out.update({q + "norm": (m["heads"] * m["vdim"],), q + "o": (w, m["heads"] * m["vdim"])})
        elif L["type"] == "delta":
            delta(q, m)
        elif L["type"] == "parallel":
            attention(q + "left.", m["left"])
            if fam == "Babotar":
                a = m["left"]
                out.update({q + "left.q.b": (a["heads"] * a["dim"],), q + "left.k.b": (a["kv_heads"] * a["dim"],),
                            q + "left.v.b": (a["kv_heads"] * a["vdim"],), q + "left.talk": (a["heads"], a["heads"])})
                delta(q + "right.", m["right"])
            else:
                r, g = m["right"], q + "right."
                out.update({g + "in": (2 * r["inner"], w), g + "conv": (r["inner"], r["conv"]), g + "conv.b": (r["inner"],),
                            g + "x": (r["dt_rank"] + 2 * r["state"], r["inner"]), g + "dt": (r["inner"], r["dt_rank"]),
                            g + "dt.b": (r["inner"],), g + "A_log": (r["inner"], r["state"]), g + "D": (r["inner"],),
                            g + "o": (w, r["inner"])})
        elif L["type"] == "attention":
            attention(q, m)
            out[q + "pb"] = (m["heads"],)
        elif L["type"] == "mamba2":
            inner, c = m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
            out.update({q + "in": (inner + c + m["heads"], w), q + "conv": (c, m["conv"]), q + "conv.b": (c,),
                        q + "norm": (inner,), q + "o": (w, inner)})
            out.update({q + n: (m["heads"],) for n in ("dt_bias", "A_log", "D")})
        else:
            out.update({q + "dq": (m["q_rank"], w), q + "dq.norm": (m["q_rank"],),
                        q + "uq": (m["heads"] * (m["dim"] + m["rot_dim"]), m["q_rank"]),
                        q + "dkv": (m["kv_rank"] + m["rot_dim"], w), q + "dkv.norm": (m["kv_rank"],),
                        q + "uk": (m["heads"] * m["dim"], m["kv_rank"]), q + "uv": (m["heads"] * m["vdim"], m["kv_rank"]),
                        q + "o": (w, m["heads"] * m["vdim"])})
        q = p + "mlp."
        if f["kind"] == "dense":
            gated(q, f["ff"])
            continue
        out[q + "router"] = (f["router"]["experts"], w)
        for e in range(f["router"]["experts"]):
            gated(f"{q}e{e}.", f["expert"]["ff"])
        gated(q + "shared.", f["shared"]["ff"])
        if fam == "Nolavik":
            out.update({q + "router.b": (f["router"]["experts"],), q + "shared.sg": (1, w)})
    return out


def checkpoint(d, seed):
    """Random weights: projections ~ N(0, 1 / fan-in), norm weights around one, gates and decays in the ranges trained
    models have them. A token of class c (its id modulo the number of experts) carries a direction of that class, and the
    routers answer it with experts c, c + 1, ..: routing is decided by a clear margin and spread over all experts, as in
    a trained model, so that two correct implementations choose alike."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def rand(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")
    f = next((L["mlp"] for L in d.get("layers", []) if L["mlp"]["kind"] == "moe"), None)
    dirs = None
    if f:
        dirs = rand(f["router"]["experts"], d["width"])
        dirs = dirs / dirs.norm(dim=1, keepdim=True)
        strength = d["width"] ** 0.5 * 0.6
    out = {}
    for name, shp in shapes(d).items():
        t, last = rand(*shp), name.split(".")[-1]
        if len(shp) == 1:
            if last in ("norm1b", "norm2b", "ls1", "ls2") or name.endswith("side.norm"):
                t = 0.5 + 0.1 * t
            elif "norm" in name or "ln_" in name and last == "weight":
                t = 1.0 + 0.1 * t
            elif last == "D":
                t = 1.0 + 0.2 * t
            elif last == "A_log":
                t = 0.5 * t - 0.5
            elif last in ("in", "out"):
                t = (0.5 if last == "in" else 1.0) + 0.1 * t
            elif last == "pb":
                t = 0.5 * t - 2.0  # weights of keys that do not answer: about a tenth
            elif name.endswith("dt.b"):
                t = 0.3 * t - 1.5
            else:
                t = 0.1 * t
        elif last == "A_log":
            t = 0.5 * t
        elif last == "mix" or last == "talk":
            t = torch.eye(shp[0], device="cuda") + 0.1 * t
        elif last == "router":
            t = 0.5 * t * shp[1] ** -0.5
            for j in range(f["router"]["top"]):
                t += (10.0 / strength) * dirs.roll(j, 0)
        elif name in ("embed", "side.embed") or name.endswith(("wte.weight", "embed_tokens.weight")):
            if dirs is not None and name == "embed":
                t += strength * dirs[torch.arange(shp[0], device="cuda") % len(dirs)]
        elif name == "loop.step" or name == "pos" or name == "wpe.weight":
            t = 0.3 * t
        else:
            t = t * (shp[0] if name.startswith("h.") else shp[1]) ** -0.5
        out[name] = t.to(torch.bfloat16)
    return out


class Checkpoint:
    """The tensors with the surface of the framework's checkpoint reader."""

    def __init__(self, tensors):
        self.tensors = tensors

    def keys(self):
        return self.tensors.keys()

    def has(self, name):
        return name in self.tensors

    def get(self, name, dtype=None):
        return self.tensors[name] if dtype is None else self.tensors[name].to(dtype)

    def rows(self, name, lo, hi, dtype=None):
        return self.get(name, dtype)[lo:hi]

    def cols(self, name, lo, hi, dtype=None):
        return self.get(name, dtype)[:, lo:hi]


def tokens_of(case, seed, vocab):
    """Token ids [sequences, longest] (CPU) of everything the sequences hold, and their lengths. A decode step's last
    token is its input; a mixed step's sequences are its single-token rows (context 512 and shorter), then its portions."""
    n = lengths(case)
    if case["do"] == "decode":
        n = [x + 1 for x in n]
    elif case["do"] == "answers":
        n = [x + case["steps"] for x in n]
    elif case["do"] == "mixed":
        n = [513 - 11 * i for i in range(case["decodes"])] + n
    gen = torch.Generator()
    gen.manual_seed(seed + 7)
    return torch.randint(0, vocab, (len(n), max(n)), generator=gen), n


# ------------------------------------------------------------------------------------------------- prepare and run
class Pages:
    """Where the sequences' positions live: scattered pages of the pool, and the step inputs that name them."""

    def __init__(self, tokens, lens, seed):
        self.tokens, self.B = tokens, len(lens)
        self.per = -(-max(lens) // BLOCK)
        self.count = self.B * self.per
        gen = torch.Generator()
        gen.manual_seed(seed + 13)
        self.table = torch.randperm(self.count, generator=gen).view(self.B, self.per)
        self.state = torch.randperm(self.B, generator=gen)

    def step(self, parts, graph=False):
        """StepInput of (sequence, first position, end) parts, single tokens of running sequences first."""
        from llmss_amd.models.decoder import StepInput

        ids = torch.cat([self.tokens[b, a:e] for b, a, e in parts])
        pos = torch.cat([torch.arange(a, e) for _, a, e in parts])
        seq = torch.cat([torch.full((e - a,), b) for b, a, e in parts])
        slots = self.table[seq, pos // BLOCK] * BLOCK + pos % BLOCK
        which = torch.tensor([b for b, _, _ in parts])
        single = 0
        while single < len(parts) and parts[single][1] > 0 and parts[single][2] - parts[single][1] == 1:
            single += 1
        counts = [e - a for _, a, e in parts]
        ends = torch.tensor(counts).cumsum(0)
        last = (ends - 1).cuda()
        common = dict(input_ids=ids.cuda(), positions=pos.cuda(), slots=slots.cuda(), last_idx=last,
                      block_tables=self.table[which].to(torch.int32).cuda(), max_ctx=self.per * BLOCK,
                      ctx_lens=torch.tensor([e for _, _, e in parts], dtype=torch.int32).cuda(),
                      state_slots=self.state[which].to(torch.int32).cuda())
        if single == len(parts):
            return StepInput(kind="decode", **common)
        prefix = any(a > 0 for _, a, _ in parts[single:])
        cu = torch.tensor([0] + counts[single:]).cumsum(0).to(torch.int32)
        return StepInput(kind="extend" if single or prefix else "prefill", cu_seqlens=cu.cuda(),
                         max_seqlen=max(counts[single:]), num_decode=single, has_prefix=prefix, **common)


def prepare(case, seed):
    from llmss_amd.models import weights as loaders
    from llmss_amd.models.config import ModelConfig
    from llmss_amd.models.layered import create_model

    d = describe(case)
    cfg = ModelConfig.from_hf_dict(d)
    reader = Checkpoint(checkpoint(d, seed))
    if "model_type" in d:
        w = loaders.load_hf_weights(cfg, reader, device="cuda", dtype=torch.bfloat16, fp8=bool(case.get("fp8")))
    else:
        load = {"babotar": loaders.load_babotar_weights, "fizelix": loaders.load_fizelix_weights,
                "nolavik": loaders.load_nolavik_weights}[case["family"]]
        w = load(cfg, reader, device="cuda", dtype=torch.bfloat16)
    model = create_model(cfg, w)
    model.kv_fp8 = bool(case.get("fp8"))
    tokens, lens = tokens_of(case, seed, cfg.vocab_size)
    pages = Pages(tokens, lens, seed)
    stateful = bool(getattr(model, "needs_state", False))
    kv = model.allocate_kv_cache(pages.count, BLOCK, num_slots=pages.B) if stateful else \
        model.allocate_kv_cache(pages.count, BLOCK)
    st = dict(model=model, kv=kv, do=case["do"], vocab=cfg.vocab_size,
              states=[c[2]["S"] for c in kv if len(c) > 2 and "S" in c[2]], slots=pages.state.cuda())
    if case["do"] == "prompts":
        st["step"] = pages.step([(b, 0, n) for b, n in enumerate(lens)])
    elif case["do"] == "decode":
        for b, n in enumerate(lens):  # the contexts, as earlier steps left them
            model.hidden_states(pages.step([(b, 0, n - 1)]), kv)
        st["step"] = pages.step([(b, n - 1, n) for b, n in enumerate(lens)])
        st["graph"], st["out"] = capture(model, st["step"], kv)
    elif case["do"] == "mixed":
        nd = case["decodes"]
        parts = [(b, n - 1, n) for b, n in enumerate(lens[:nd])] + [(nd + i, n // 2, n) for i, n in enumerate(lens[nd:])]
        for b, a, _ in parts:
            if a:
                model.hidden_states(pages.step([(b, 0, a)]), kv)
        st["step"] = pages.step(parts)
    else:
        n = lengths(case)
        st["step"] = pages.step([(b, 0, x) for b, x in enumerate(n)])
        steps = [pages.step([(b, x + t, x + t + 1) for b, x in enumerate(n)]) for t in range(case["steps"])]
        # the decode graph reads its inputs from one staging buffer: ids | positions | slots (64 bit) | context lengths
        B, packed = pages.B, [torch.cat([s.input_ids.view(torch.uint8), s.positions.view(torch.uint8),
                                         s.slots.view(torch.uint8), s.ctx_lens.view(torch.uint8)]) for s in steps]
        stage = packed[0].clone()
        wide = stage[:24 * B].view(torch.int64).view(3, B)
        s = steps[0]
        s.input_ids, s.positions, s.slots, s.ctx_lens = wide[0], wide[1], wide[2], stage[24 * B:].view(torch.int32)
        st.update(stage=stage, inputs=packed, decode=s)  # (the graph reads the step's other tensors too: they stay)
        st["graph"], st["out"] = capture(model, s, kv)
    return st


def capture(model, step, kv):
    """A HIP graph of one decode step, and its logits' buffer."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            model(step, kv)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = model(step, kv)
    return graph, out


def run(state):
    model, V = state["model"], state["vocab"]
    if state["do"] == "decode":
        state["graph"].replay()
        return {"logits": state["out"][:, :V]}
    step = state["step"]
    hidden = model.hidden_states(step, state["kv"])
    logits = model.logits(hidden.index_select(0, step.last_idx))[:, :V]
    if state["do"] == "answers":
        logits = [logits]
        for packed in state["inputs"]:
            state["stage"].copy_(packed)
            state["graph"].replay()
            logits.append(state["out"][:, :V].clone())
        logits = torch.stack(logits)
    return {"hidden": hidden, "logits": logits, "states": [s.index_select(0, state["slots"]) for s in state["states"]]}


# -------------------------------------------------------------------------------------------------------------- work
def work(case):
    """Weights once (of the experts those that the tokens reach), cached rows and states read and written once, rows and
    logits written; products of the tokens with the weights they meet, attention over the visible pairs, recurrences."""
    d = describe(case)
    top = experts = 1
    for L in d.get("layers", []):
        if L["mlp"]["kind"] == "moe":
            top, experts = L["mlp"]["router"]["top"], L["mlp"]["router"]["experts"]
    times = {f"l{i}.": runs(d).count(i) for i in range(len(d["layers"]))} if "layers" in d else {}
    fixed = routed = active = head = 0
    for name, s in shapes(d).items():
        if len(s) < 2 or name in ("embed", "pos", "side.embed", "loop.step", "wpe.weight", "model.embed_tokens.weight"):
            continue
        n = s[0] * s[1]
        if name in ("head", "lm_head.weight", "wte.weight"):
            head = n
            continue
        k = times.get(name.split(".")[0] + ".", 1)
        if ".mlp.e" in name:
            routed += n * k
            active += n * k * top / experts
        else:
            fixed += n * k
            active += n * k
    w = case["width"]
    kinds = [d["layers"][i] for i in runs(d)] if "layers" in d else [None] * case["layers"]
    kv = state = 0  # cached numbers per token; state numbers per sequence
    pair = rec = 0  # flops per visible pair; recurrence flops per token
    for L in kinds:
        t = L and L["type"]
        m = L and L["mixer"]
        if t in (None, "attention") or t == "parallel":
            a = {"heads": w // 64 if case["family"] == "gpt2" else w // 128, "kv_heads": w // 64 if case["family"] == "gpt2"
                 else w // 128, "dim": 64 if case["family"] == "gpt2" else 128} if L is None else m.get("left", m)
            kv += 2 * a["kv_heads"] * a["dim"]
            pair += 4 * a["heads"] * a["dim"]
        if t == "latent_attention":
            kv += m["kv_rank"] + m["rot_dim"]
            pair += 2 * m["heads"] * (2 * m["kv_rank"] + m["rot_dim"])
        r = m if t in ("delta", "lightning") else m["right"] if t == "parallel" else None
        if r is not None:
            n = r["inner"] * r["state"] if "inner" in r else r["heads"] * r["dim"] * r["vdim"]
            state, rec = state + n, rec + 6 * n
        if t == "mamba2":
            n = m["heads"] * m["state"] * m["vdim"]
            state, rec = state + n, rec + 5 * n
    wide = 1 if case.get("fp8") else 2

    def cost(parts):  # (cached before, new) per sequence
        T, S = sum(n for _, n in parts), len(parts)
        reach = min(1.0, T * top / experts)
        seen = sum(n * c + n * (n + 1) / 2 for c, n in parts)
        old = sum(c for c, _ in parts)
        if case["family"] == "fizelix":  # a window of 512 and one mean per 16 positions behind it
            seen = sum(sum(min(t, 512) + max(0, t - 512) // 16 for t in range(c + 1, c + n + 1)) for c, n in parts)
            old = sum(min(c, 512) + max(0, c - 512) // 16 for c, _ in parts)
        b = wide * (fixed + routed * reach) + 2 * head + wide * kv * (old + T) + 4 * state * S * (2 if old else 1) \
            + 2 * T * w + 2 * S * VOCAB
        return b, 2 * T * active + 2 * S * head + pair * seen + rec * T
    n = lengths(case)
    if case["do"] == "prompts":
        todo = [[(0, x) for x in n]]
    elif case["do"] == "decode":
        todo = [[(x, 1) for x in n]]
    elif case["do"] == "mixed":
        todo = [[(512 - 11 * i, 1) for i in range(case["decodes"])] + [(x // 2, x - x // 2) for x in n]]
    else:
        todo = [[(0, x) for x in n]] + [[(x + t, 1) for x in n] for t in range(case["steps"])]
    got = [cost(p) for p in todo]
    return {"bytes": float(sum(b for b, _ in got)), "flops": float(sum(f for _, f in got))}


# -------------------------------------------------------------------------------------------------- the same in 64 bits
def rms(x):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + EPS)


def silu(z):
    return z * torch.sigmoid(z)


def softplus(z):
    return torch.clamp(z, min=0.0) + torch.log1p(torch.exp(-z.abs()))


def gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def conv(x, w, b=None):
    """x [B, T, C], w [C, taps]: y_t = sum_j w[:, j] x_(t - taps + 1 + j) (+ b)."""
    taps, T = w.shape[1], x.shape[1]
    full = torch.nn.functional.pad(x, (0, 0, taps - 1, 0))
    y = sum(w[:, j] * full[:, j:j + T] for j in range(taps))
    return y if b is None else y + b


def turn(x, freqs, neighbours, amp=1.0):
    """x [B, T, heads, n]: pairs (i, i + half) - or neighbours (2 i, 2 i + 1) - turned by position * freqs[i]."""
    half = len(freqs)
    ang = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * torch.tensor(freqs, dtype=F64, device=x.device)
    c, s = (amp * torch.cos(ang))[:, None], (amp * torch.sin(ang))[:, None]
    if neighbours:
        u, v = x[..., 0:2 * half:2], x[..., 1:2 * half:2]
        return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), x[..., 2 * half:]], -1)
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], -1)


def blended(r):
    """babotar's frequencies and amplitude: towards f / factor between two numbers of turns."""
    f, sc = [r["base"] ** (-2.0 * i / r["dims"]) for i in range(r["dims"] // 2)], r["scaling"]

    def dim(t):
        return r["dims"] * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(r["base"]))
    lo, hi = max(math.floor(dim(sc["fast"])), 0), min(math.ceil(dim(sc["slow"])), r["dims"] - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(len(f))]
    return [a / sc["factor"] * b + a * (1.0 - b) for a, b in zip(f, ramp)], 0.1 * math.log(sc["factor"]) + 1.0


def stretched(r):
    """nolavik's frequencies: long wavelengths turn ``factor`` times slower, a blend in between."""
    out, sc = [], r["scaling"]
    for i in range(r["dims"] // 2):
        f = r["base"] ** (-2.0 * i / r["dims"])
        wave = 2.0 * math.pi / f
        if wave > sc["original"] / sc["low"]:
            f = f / sc["factor"]
        elif wave >= sc["original"] / sc["high"]:
            s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
            f = (1.0 - s) * f / sc["factor"] + s * f
        out.append(f)
    return out


def attend(q, k, v, scale, unit=0.0, cap=0.0, talk=None):
    """q [B, T, H, n], k / v [B, T, G, ..]: causal softmax attention; ``unit`` more in every denominator, scores through
    cap * tanh(s / cap), the heads' weights mixed by ``talk``."""
    B, T, H, _ = q.shape
    rep = H // k.shape[2]
    later = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    out = q.new_empty(B, T, H, v.shape[3])
    for b in range(B):
        kk, vv = (t[b].repeat_interleave(rep, 1).transpose(0, 1) for t in (k, v))
        step = H if talk is not None else max(1, (1 << 26) // (T * T))
        for h in range(0, H, step):
            s = q[b, :, h:h + step].transpose(0, 1) @ kk[h:h + step].transpose(1, 2) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(later, -math.inf)
            m = s.amax(-1, keepdim=True).clamp(min=0.0)
            e = torch.exp(s - m)
            p = e / (e.sum(-1, keepdim=True) + unit * torch.exp(-m))
            if talk is not None:
                p = (talk @ p.reshape(H, -1)).view_as(p)
            out[b, :, h:h + step] = (p @ vv[h:h + step]).transpose(0, 1)
    return out


def pooled(q, k, v, pb, scale, size, pool):
    """fizelix: weights sigmoid(score + pb[h]) of the last ``size`` positions and of one mean row per ``pool`` positions
    that lie wholly behind them."""
    B, T, H, _ = q.shape
    rep, nb = H // k.shape[2], max(0, T - size) // pool
    i = torch.arange(T, device=q.device)[:, None]
    j = torch.arange(T, device=q.device)[None]
    see = (j <= i) & (j > i - size)
    if nb:
        see = torch.cat([see, torch.arange(nb, device=q.device)[None] * pool + pool - 1 <= i - size], 1)
    out = q.new_empty(B, T, H, v.shape[3])
    for b in range(B):
        kk, vv = k[b], v[b]
        if nb:
            kk, vv = (torch.cat([t, t[:nb * pool].view(nb, pool, *t.shape[1:]).mean(1)]) for t in (kk, vv))
        for h in range(H):
            wgt = torch.sigmoid(q[b, :, h] @ kk[:, h // rep].T * scale + pb[h]) * see
            out[b, :, h] = wgt @ vv[:, h // rep]
    return out


def scan(T, n, S, step):
    """Walk a recurrence: ``step(t, S)`` -> (S, y). A sequence's state stops at its own length. y [B, T, ..], S."""
    out = []
    for t in range(T):
        new, y = step(t, S)
        on = (t < n).view(-1, *[1] * (S.dim() - 1))
        S = torch.where(on, new, S)
        out.append(y)
    return torch.stack(out, 1), S


def decay_scan(q, k, v, decay, n):
    B, T, H, dim = q.shape

    def step(t, S):
        S = decay[:, None, None] * S + k[:, t, :, :, None] * v[:, t, :, None]
        return S, (q[:, t, :, None] @ S)[:, :, 0]
    return scan(T, n, q.new_zeros(B, H, dim, v.shape[3]), step)


def delta_rule(W, p, m, h, n):
    B, T = h.shape[:2]
    H, G, dim, vd = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (silu(conv(h @ W(p + c).T, W(p + c + ".conv"))) for c in "qkv")

    def unit(x):
        x = x.view(B, T, G, dim)
        return (x / torch.sqrt(x.pow(2).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 2)
    q, k, v = unit(q) * dim ** -0.5, unit(k), v.view(B, T, H, vd)
    beta = torch.sigmoid(h @ W(p + "b").T)
    g = torch.exp(-torch.exp(W(p + "A_log")) * softplus(h @ W(p + "a").T + W(p + "dt_bias")))

    def step(t, S):
        S = g[:, t, :, None, None] * S
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
        S = S + k[:, t, :, :, None] * u[:, :, None]
        return S, (q[:, t, :, None] @ S)[:, :, 0]
    o, S = scan(T, n, h.new_zeros(B, H, dim, vd), step)
    o = rms(o) * W(p + "norm") * silu(h @ W(p + "g").T).view(B, T, H, vd)
    return o.reshape(B, T, H * vd) @ W(p + "o").T, S


def state_space(W, p, m, h, n):
    B, T = h.shape[:2]
    H, vd, N = m["heads"], m["vdim"], m["state"]
    inner = H * vd
    proj = h @ W(p + "in").T
    z, dt = proj[..., :inner], softplus(proj[..., 2 * inner + 2 * N:] + W(p + "dt_bias"))
    xbc = silu(conv(proj[..., inner:2 * inner + 2 * N], W(p + "conv"), W(p + "conv.b")))
    x, Bm, C = xbc[..., :inner].view(B, T, H, vd), xbc[..., inner:inner + N], xbc[..., inner + N:]
    fade = torch.exp(-torch.exp(W(p + "A_log")) * dt)

    def step(t, S):
        S = fade[:, t, :, None, None] * S + Bm[:, t, None, :, None] * (dt[:, t, :, None] * x[:, t])[:, :, None]
        return S, (C[:, t, None, None] @ S)[:, :, 0]
    y, S = scan(T, n, h.new_zeros(B, H, N, vd), step)
    y = (y + W(p + "D")[:, None] * x).reshape(B, T, inner) * silu(z)
    return (rms(y) * W(p + "norm")) @ W(p + "o").T, S


def selective(W, p, m, h, n):
    B, T = h.shape[:2]
    inner, N, R = m["inner"], m["state"], m["dt_rank"]
    xz = h @ W(p + "in").T
    x = silu(conv(xz[..., :inner], W(p + "conv"), W(p + "conv.b")))
    dbc = x @ W(p + "x").T
    dt = softplus(dbc[..., :R] @ W(p + "dt").T + W(p + "dt.b"))
    Bm, C, A = dbc[..., R:R + N], dbc[..., R + N:], -torch.exp(W(p + "A_log"))

    def step(t, S):
        S = torch.exp(dt[:, t, :, None] * A) * S + (dt[:, t] * x[:, t])[:, :, None] * Bm[:, t, None]
        return S, (S @ C[:, t, :, None])[..., 0]
    y, S = scan(T, n, h.new_zeros(B, inner, N), step)
    return ((y + W(p + "D") * x) * silu(xz[..., inner:])) @ W(p + "o").T, S


def gated(W, p, h, act=silu):
    return (act(h @ W(p + "gate").T) * (h @ W(p + "up").T)) @ W(p + "down").T


def mixture(W, p, f, h, fizelix):
    flat = h.reshape(-1, h.shape[-1])
    z = flat @ W(p + "router").T
    if not fizelix:
        z = z + W(p + "router.b")
    val, idx = z.topk(f["router"]["top"], -1)
    share = torch.sigmoid(val) if fizelix else torch.softmax(val, -1)
    out = gated(W, p + "shared.", flat)
    if not fizelix:
        out = out * torch.sigmoid(flat @ W(p + "shared.sg").T)
    for e in range(f["router"]["experts"]):
        rows, at = (idx == e).nonzero(as_tuple=True)
        s = share[rows, at][:, None]
        out.index_add_(0, rows, gated(W, f"{p}e{e}.", s * flat[rows]) if fizelix else s * gated(W, f"{p}e{e}.", flat[rows]))
    return out.view_as(h)


def heads_of(W, p, m, h):
    q, k, v = (h @ W(p + n).T + (W(p + n + ".b") if W.has(p + n + ".b") else 0.0) for n in "qkv")
    return q.unflatten(-1, (m["heads"], -1)), k.unflatten(-1, (m["kv_heads"], -1)), v.unflatten(-1, (m["kv_heads"], -1))


def layer_norm(x, w, b=0.0, eps=EPS):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt(d.pow(2).mean(-1, keepdim=True) + eps) * w + b


def dense64(d, W, tok):
    """gpt2 and llama: the normed rows [B, T, width] and the head."""
    if d["model_type"] == "gpt2":
        x, H = W("wte.weight")[tok] + W("wpe.weight")[:tok.shape[1]], d["n_head"]
        for i in range(d["n_layer"]):
            def lin(n, y):
                return y @ W(f"h.{i}.{n}.weight") + W(f"h.{i}.{n}.bias")

            def norm(n, y):
                return layer_norm(y, W(f"h.{i}.{n}.weight"), W(f"h.{i}.{n}.bias"), 1e-5)
            q, k, v = (t.unflatten(-1, (H, -1)) for t in lin("attn.c_attn", norm("ln_1", x)).chunk(3, -1))
            x = x + lin("attn.c_proj", attend(q, k, v, q.shape[-1] ** -0.5).flatten(2))
            x = x + lin("mlp.c_proj", gelu(lin("mlp.c_fc", norm("ln_2", x))))
        return layer_norm(x, W("ln_f.weight"), W("ln_f.bias"), 1e-5), W("wte.weight")
    x, H = W("model.embed_tokens.weight")[tok], d["num_attention_heads"]
    dim = d["hidden_size"] // H
    f = [10000.0 ** (-2.0 * i / dim) for i in range(dim // 2)]
    for i in range(d["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = rms(x) * W(p + "input_layernorm.weight")
        q, k, v = ((h @ W(p + f"self_attn.{n}_proj.weight").T).unflatten(-1, (H, dim)) for n in "qkv")
        o = attend(turn(q, f, False), turn(k, f, False), v, dim ** -0.5).flatten(2)
        x = x + o @ W(p + "self_attn.o_proj.weight").T
        h = rms(x) * W(p + "post_attention_layernorm.weight")
        x = x + (silu(h @ W(p + "mlp.gate_proj.weight").T) * (h @ W(p + "mlp.up_proj.weight").T)) @ W(p + "mlp.down_proj.weight").T
    return rms(x) * W("model.norm.weight"), W("lm_head.weight")


def babotar64(d, W, tok, n):
    x0 = W("embed")[tok] + W("pos")[:tok.shape[1]]
    xs, states = [x0, x0], []
    for i, L in enumerate(d["layers"]):
        p, q, m = f"l{i}.", f"l{i}.mix.", L["mixer"]
        for k in (1, 2):
            hc = f"{p}hc{k}."
            h = layer_norm(W(hc + "in")[0] * xs[0] + W(hc + "in")[1] * xs[1], W(f"{p}norm{k}"))
            if k == 2:
                y = gated(W, p + "mlp.", h, gelu)
            else:
                h = h + conv(h, W(p + "canon1"))
                if L["type"] == "lightning":
                    a, b, c = (silu(h @ W(q + s).T).unflatten(-1, (m["heads"], -1)) for s in "qkv")
                    o, S = decay_scan(a, b, c, torch.tensor(m["decay"], dtype=torch.float32, device=h.device).to(F64), n)
                    y = (rms(o.flatten(2)) * W(q + "norm") * torch.sigmoid(h @ W(q + "g").T)) @ W(q + "o").T
                else:
                    a = m["left"]
                    f, amp = blended(a["rot"])
                    Q, K, V = heads_of(W, q + "left.", a, h)
                    o = attend(turn(Q, f, False, amp), turn(K, f, False, amp), V, a["scale"], 1.0, a["softcap"],
                               W(q + "left.talk"))
                    y, S = delta_rule(W, q + "right.", m["right"], h, n)
                    y = m["left_scale"] * (o.flatten(2) @ W(q + "left.o").T) + m["right_scale"] * y
                states.append(S)
            xs = [W(hc + "mix")[0, t] * xs[0] + W(hc + "mix")[1, t] * xs[1] + W(hc + "out")[t] * y for t in (0, 1)]
    return layer_norm(xs[0] + xs[1], W("final.norm")), W("head"), states


def fizelix64(d, W, tok, n):
    x0 = W("embed")[tok]
    x, states, order = x0.clone(), [], runs(d)
    side = d["token_side"]["dim"]
    for r, i in enumerate(order):
        L, p, q = d["layers"][i], f"l{i}.", f"l{i}.mix."
        m = L["mixer"]
        if i == d["loop"]["start"] and i in order[:r]:  # before every pass but the first
            x = x + x0
        h = rms(x) * W(p + "norm1")
        if L["type"] == "attention":
            f = [m["rot"]["base"] ** (-2.0 * j / m["rot"]["dims"]) for j in range(m["rot"]["dims"] // 2)]
            Q, K, V = heads_of(W, q, m, h)
            o = pooled(turn(Q, f, True), turn(K, f, True), V, W(q + "pb"), m["scale"], m["mask"]["size"], m["mask"]["pool"])
            y = o.flatten(2) @ W(q + "o").T
        else:
            y, S = state_space(W, q, m, h, n)
            states.append(S)
        for k in "12":
            if k == "2":
                h = rms(x) * W(p + "norm2")
                y = gated(W, p + "mlp.", h) if L["mlp"]["kind"] == "dense" else mixture(W, p + "mlp.", L["mlp"], h, True)
            x = x + rms(y * torch.sigmoid(h @ W(p + "rg" + k).T + W(p + f"rg{k}.b"))) * W(p + f"norm{k}b") * W(p + "ls" + k)
        e = W("side.embed")[tok][..., i * side:(i + 1) * side]
        x = x + rms((gelu(x @ W(p + "side.gate").T) * e) @ W(p + "side.proj").T) * W(p + "side.norm")
    return rms(x) * W("final.norm"), W("head"), states


def nolavik64(d, W, tok, n):
    x, states = W("embed")[tok], []
    for i, L in enumerate(d["layers"]):
        p, q, m = f"l{i}.", f"l{i}.mix.", L["mixer"]
        if i == d["loop"]["start"]:
            x = x + W("loop.step")[0]
        h = rms(x) * W(p + "norm1")
        if L["type"] == "delta":
            y, S = delta_rule(W, q, m, h, n)
            states.append(S)
        elif L["type"] == "parallel":
            a, f = m["left"], stretched(m["left"]["rot"])
            Q, K, V = heads_of(W, q + "left.", a, h)
            o = attend(rms(turn(Q, f, False)), rms(turn(K, f, False)), V, a["scale"], 1.0)
            y, S = selective(W, q + "right.", m["right"], h, n)
            states.append(S)
            y = m["left_scale"] * (o.flatten(2) @ W(q + "left.o").T) + m["right_scale"] * y
        else:
            H, dim, R = m["heads"], m["dim"], m["kv_rank"]
            f = [m["rot"]["base"] ** (-2.0 * j / m["rot_dim"]) for j in range(m["rot_dim"] // 2)]
            Q = ((rms(h @ W(q + "dq").T) * W(q + "dq.norm")) @ W(q + "uq").T).unflatten(-1, (H, -1))
            down = h @ W(q + "dkv").T
            c = rms(down[..., :R]) * W(q + "dkv.norm")
            kr = turn(down[..., None, R:], f, False).expand(-1, -1, H, -1)
            K = torch.cat([(c @ W(q + "uk").T).unflatten(-1, (H, dim)), kr], -1)
            Q = torch.cat([Q[..., :dim], turn(Q[..., dim:], f, False)], -1)
            y = attend(Q, K, (c @ W(q + "uv").T).unflatten(-1, (H, -1)), m["scale"]).flatten(2) @ W(q + "o").T
        x = x + rms(y) * W(p + "norm1b")
        x = x + rms(mixture(W, p + "mlp.", L["mlp"], rms(x) * W(p + "norm2"), False)) * W(p + "norm2b")
    return rms(x) * W("final.norm"), W("head"), states


class Weights64:
    """Checkpoint tensors in 64 bits. ``fp8``: the layers' projections as e4m3 rows with one scale each hold them."""

    def __init__(self, tensors, fp8):
        self.tensors, self.fp8 = tensors, fp8

    def has(self, name):
        return name in self.tensors

    def __call__(self, name):
        t = self.tensors[name]
        if self.fp8 and "_proj" in name:
            s = t.float().abs().amax(1, keepdim=True) / 448.0
            return (t.float() * (1.0 / s)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).to(F64) * s.to(F64)
        return t.to(F64)


def exact(case, seed):
    d = describe(case)
    W = Weights64(checkpoint(d, seed), bool(case.get("fp8")))
    tok, lens = tokens_of(case, seed, d.get("vocab_size", VOCAB))
    for b, n in enumerate(lens):
        tok[b, n:] = 0
    tok, n = tok.cuda(), torch.tensor(lens).cuda()
    if "model_type" in d:
        groups = [dense64(d, W, tok[b:b + 8]) for b in range(0, len(lens), 8)]
        x, head, states = torch.cat([g[0] for g in groups]), groups[0][1], []
    else:
        x, head, states = {"babotar": babotar64, "fizelix": fizelix64, "nolavik": nolavik64}[case["family"]](d, W, tok, n)

    def at(where):
        return x[torch.arange(len(lens), device="cuda"), where] @ head.T
    if case["do"] == "decode":
        return {"logits": at(n - 1)}
    if case["do"] == "answers":
        first = n - case["steps"]
        hidden = torch.cat([x[b, :k] for b, k in enumerate(first.tolist())])
        return {"hidden": hidden, "logits": torch.stack([at(first - 1 + t) for t in range(case["steps"] + 1)]),
                "states": states}
    if case["do"] == "mixed":
        hidden = torch.cat([x[b, k - 1 if b < case["decodes"] else k // 2:k] for b, k in enumerate(lens)])
    else:
        hidden = torch.cat([x[b, :k] for b, k in enumerate(lens)])
    return {"hidden": hidden, "logits": at(n - 1), "states": states}
