"""Prompt attention and attention behind prefixes where scores rise and fall from tile to tile of 64 keys: outputs are scaled only where
a row's maximum has grown by more than 8 (in base 2) since the last time, and weights lie between 1 and 2^8 till then. Against 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# scores of a key in base 2, by the number of its tile; rows take them times -1 .. 1
KINDS = {"3": lambda t: 3.0 * t, "9": lambda t: 9.0 * t, "40": lambda t: 40.0 * t, "down": lambda t: -9.0 * t, "steps": lambda t: 7.9 * (t % 4),
         "one": lambda t: 60.0 * (t == 2)}


def rows(kind, T, n, nh, nkv, D, g):
    """Queries [T, nh, D], keys and values [n, nkv, D] of one sequence, its last T rows."""
    u = torch.randn(nkv, D, generator=g)
    s = torch.tensor([KINDS[kind](j // 64) for j in range(n)])
    k = u * (s / (D ** -0.5 * math.log2(math.e)))[:, None, None] / (u * u).sum(-1, keepdim=True) + 0.2 * torch.randn(n, nkv, D, generator=g)
    q = u.repeat_interleave(nh // nkv, 0) * (2 * torch.rand(T, nh, 1, generator=g) - 1) + 0.2 * torch.randn(T, nh, D, generator=g)
    return q.bfloat16().cuda(), k.bfloat16().cuda(), torch.randn(n, nkv, D, generator=g).bfloat16().cuda()


def check(got, q, k, v, window=0):
    """Of rows at the last positions: rounding of weights and of the result to bf16, scores from sums in 32 bits."""
    T, nh, D = q.shape
    n, nkv = k.shape[:2]
    pos, key = torch.arange(n - T, n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
    seen = (key <= pos) & ((key > pos - window) | (window == 0))
    for h in range(nh):
        kd, vd, qd = (t.double().contiguous() for t in (k[:, h * nkv // nh], v[:, h * nkv // nh], q[:, h]))
        s = (qd @ kd.t().contiguous() * D ** -0.5).masked_fill(~seen, -math.inf)
        e = ((D + 8) * 2.0 ** -24 * D ** -0.5 * (qd.abs() @ kd.abs().t().contiguous()) + 2.0 ** -22 * s.abs()).masked_fill(~seen, 0).amax(-1, keepdim=True)
        p = torch.softmax(s, -1)
        want, size = p @ vd, p @ vd.abs()
        lim = (2.0 ** -8 + 2 * e + 2.0 ** -18) * size + 2.0 ** -8 * want.abs() + 1e-30
        assert ((got[:, h].double() - want).abs() <= lim).all(), (h, ((got[:, h].double() - want).abs() / lim).max())


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,nkv,D", [(4, 4, 64), (4, 2, 128), (3, 1, 256)])
def test_prompts(kind, nh, nkv, D):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(D)
    lens = [700, 1, 129, 64, 383]
    seqs = [rows(kind, n, n, nh, nkv, D, g) for n in lens]
    qkv = torch.cat([torch.cat([t.reshape(t.shape[0], -1) for t in s], 1) for s in seqs])
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int().cuda()
    y = hip.attn_prefill(qkv, cu, max(lens), nh, nkv, D, D ** -0.5).view(-1, nh, D)
    for (q, k, v), a in zip(seqs, cu.tolist()):
        check(y[a:a + q.shape[0]], q, k, v)


def paged(seqs, nkv, D, bs, fp8, g):
    """Caches with the sequences' keys and values in blocks out of order, their tables, and what the caches hold."""
    from llmss_amd.ops import reference as ref
    n = [k.shape[0] for _, k, _ in seqs]
    width = max(-(-x // bs) for x in n)
    nb = sum(-(-x // bs) for x in n)
    perm, at = torch.randperm(nb, generator=g), 0
    bt = torch.zeros(len(seqs), width, dtype=torch.int32)
    kc, vc = (torch.zeros(nb, nkv, bs, D + (ref.KV8_TAIL if fp8 else 0), dtype=torch.uint8 if fp8 else torch.bfloat16, device="cuda") for _ in range(2))
    held = []
    for i, (q, k, v) in enumerate(seqs):
        blocks = -(-n[i] // bs)
        ids = perm[at:at + blocks]
        at += blocks
        bt[i, :blocks] = ids.int()
        slot = (ids[:, None] * bs + torch.arange(bs)).flatten()[:n[i]].cuda()
        kv = []
        for cache, t in ((kc, k), (vc, v)):
            r = ref.kv_rows_quant(t) if fp8 else t
            cache[slot // bs, :, slot % bs] = r
            kv.append(ref.kv_rows_dequant(r, D).bfloat16() if fp8 else t)
        held.append((q, *kv))
    return kc, vc, bt.cuda(), held


# one row group a wave, shared keys, and two row groups (64 wide: from 1024 workgroups on; else 420)
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,nkv,D,portions,two", [(4, 4, 64, [(300, 37), (0, 130), (511, 1), (64, 64)], False),
                                                   (8, 2, 128, [(450, 20), (127, 66), (700, 1)], False), (6, 1, 256, [(200, 70), (333, 3)], False),
                                                   (32, 32, 128, [(300, 900), (64, 950)], True), (64, 64, 64, [(200, 1100), (321, 1100)], True)])
@pytest.mark.parametrize("fp8,window", [(False, 0), (False, 150), (True, 0)])
def test_portions_behind_prefixes(kind, nh, nkv, D, portions, two, fp8, window):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(nh + D)
    kc, vc, bt, seqs = paged([rows(kind, t, p + t, nh, nkv, D, g) for p, t in portions], nkv, D, 16, fp8, g)
    lens = [t for _, t in portions]
    assert hip.lib().attn_extend_two(sum(lens), len(lens), max(lens), nh, nkv, D) == two
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int().cuda()
    ctx = torch.tensor([p + t for p, t in portions]).int().cuda()
    q = torch.cat([s[0] for s in seqs]).view(sum(lens), -1)
    y = hip.attn_extend(q, kc, vc, bt, cu, ctx, max(lens), nh, nkv, D, D ** -0.5, window=window).view(-1, nh, D)
    for (q, k, v), a in zip(seqs, cu.tolist()):
        check(y[a:a + q.shape[0]], q, k, v, window)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,nkv,D", [(4, 4, 64), (8, 2, 128), (6, 1, 256)])
@pytest.mark.parametrize("fp8", [False, True])
def test_single_rows_with_split_keys(kind, nh, nkv, D, fp8):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(nh + D)
    ctx = [700, 1, 192, 193, 64, 449]
    kc, vc, bt, seqs = paged([rows(kind, 1, n, nh, nkv, D, g) for n in ctx], nkv, D, 16, fp8, g)
    q = torch.cat([s[0] for s in seqs]).view(len(ctx), -1)
    cu = torch.arange(len(ctx) + 1).int().cuda()
    y = hip.attn_extend(q, kc, vc, bt, cu, torch.tensor(ctx).int().cuda(), 1, nh, nkv, D, D ** -0.5, key_split=(4, 192)).view(-1, nh, D)
    for i, (q, k, v) in enumerate(seqs):
        check(y[i:i + 1], q, k, v)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,D,portions", [(16, 64, [(300, 37), (0, 130)]), (5, 128, [(450, 20), (700, 1)])])
def test_keys_that_are_the_values(kind, nh, D, portions):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(nh + D)
    kc, _, bt, seqs = paged([rows(kind, t, p + t, nh, 1, D, g) for p, t in portions], 1, D, 16, False, g)
    lens = [t for _, t in portions]
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int().cuda()
    ctx = torch.tensor([p + t for p, t in portions]).int().cuda()
    q = torch.cat([s[0] for s in seqs]).view(sum(lens), -1)
    y = hip.attn_extend(q, kc, kc, bt, cu, ctx, max(lens), nh, 1, D, D ** -0.5).view(-1, nh, D)
    for (q, k, _), a in zip(seqs, cu.tolist()):
        check(y[a:a + q.shape[0]], q, k, k)
