"""Rotation and cache writes of four numbers an access (csrc/attention_sink.hip, csrc/attention_pool.hip) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows on both sides of the spread over workgroups; a row of one access, rows with remainders of 1024; offsets that are no multiple of
# four and rotated parts that are no multiple take the kernels of single numbers
@pytest.mark.parametrize("T,H,G,dim,vdim,rot,off", [(1, 1, 1, 4, 4, 0, 0), (5, 3, 1, 24, 20, 8, 4), (256, 4, 2, 128, 64, 128, 8),
                                                   (300, 8, 4, 64, 136, 32, 0), (7, 2, 2, 16, 8, 4, 4), (7, 2, 2, 16, 8, 16, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["halves", "halves+bias", "pairs"])
def test_rope_rows(T, H, G, dim, vdim, rot, off, dtype, form):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(T + dim)
    nq, nk, nv = H * dim, G * dim, G * vdim
    pad = (-(off + nq + nk + nv)) % 4 + 4
    proj = torch.randn(T, off + nq + nk + nv + pad, generator=g).to(dtype).cuda()
    kc, vc = torch.full((T + 3, 1, nk), 7.0, dtype=dtype, device="cuda"), torch.full((T + 3, 1, nv), 7.0, dtype=dtype, device="cuda")
    slots = (torch.randperm(T + 3, generator=g)[:T]).cuda()
    if T > 1:
        slots[1] = -1
    ang = torch.rand(T, rot // 2, generator=g) * 6
    cs = torch.stack([ang.cos(), ang.sin()], -1).contiguous().cuda()
    x = proj.double()
    if form == "pairs":
        q = hip.rope_pairs_cache(proj, off, off + nq, off + nq + nk, cs if rot else None, kc, vc, slots, H, G, dim, vdim)
    else:
        bias = torch.randn(nq + nk + nv, generator=g).to(dtype).cuda() if "bias" in form else None
        pos = torch.arange(T).flip(0).contiguous().cuda()
        q = hip.rope_bias_cache(proj, off, off + nq, off + nq + nk, bias, pos, cs.flip(0).contiguous(), rot, kc, vc, slots, H, G, dim, vdim)
        if bias is not None:
            x = torch.cat([x[:, :off], x[:, off:off + nq + nk + nv] + bias.double(), x[:, off + nq + nk + nv:]], 1)
    a = x[:, off:off + nq + nk].reshape(T, H + G, dim)
    c, s = cs.double()[:, None, :, 0], cs.double()[:, None, :, 1]
    want, mag = a.clone(), a.abs().clone()
    if rot:
        i, j = (slice(0, rot, 2), slice(1, rot, 2)) if form == "pairs" else (slice(0, rot // 2), slice(rot // 2, rot))
        want[..., i], want[..., j] = a[..., i] * c - a[..., j] * s, a[..., j] * c + a[..., i] * s
        mag[..., i] = mag[..., j] = a[..., i].abs() + a[..., j].abs()
    lim = 4 * 2.0 ** -24 * mag  # the sums with the bias, two products, their sum
    assert ((q.double().view(T, H, dim) - want[:, :H]).abs() <= lim[:, :H]).all()
    rnd = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    for cache, w, lm in ((kc, want[:, H:].reshape(T, nk), lim[:, H:].reshape(T, nk)),
                         (vc, x[:, off + nq + nk:off + nq + nk + nv], 2.0 ** -23 * x[:, off + nq + nk:off + nq + nk + nv].abs())):
        full = torch.full_like(cache, 7.0)[:, 0].double()
        flim = torch.zeros_like(full)
        live = slots >= 0
        full[slots[live]], flim[slots[live]] = w[live], lm[live] + rnd * w[live].abs()
        assert ((cache[:, 0].double() - full).abs() <= flim).all()


# latent rows of more numbers than a wave asks for at once, of one and of a few; heads and pairs past whole rounds of three waves, or turned by the
# row's own wave (4096 rows on); rows that are not cached
@pytest.mark.gpu
@pytest.mark.parametrize("T,H,R,rot,rdims", [(3, 1, 1, 2, 2), (5, 7, 511, 64, 62), (70, 16, 513, 64, 64), (2, 130, 700, 34, 34), (4, 3, 192, 6, 0), (9, 1, 96, 0, 0),
                                            (4096, 4, 64, 64, 64), (4097, 43, 130, 8, 6), (4095, 9, 257, 30, 28), (6, 4, 128, 66, 66), (4100, 5, 65, 20, 0), (4, 8, 64, 128, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_latent_rows_and_their_queries(T, H, R, rot, rdims, dtype):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(T + R)
    qdim, n = 5, R + rot
    src = torch.randn(T, n + H * (qdim + rot), generator=g).to(dtype)
    w = torch.randn(R, generator=g).to(dtype)
    cs = torch.randn(T, rdims // 2, 2, generator=g)
    slots = torch.randperm(T + 3, generator=g)[:T]
    slots[0] = -1
    cache, qa = torch.full((T + 3, 1, n), 7.0, dtype=dtype).cuda(), torch.full((T, H, n), 7.0).cuda()
    hip.latent_norm_cache(src.cuda(), 0, R, w.cuda(), 1e-6, cache, slots.cuda(), rot, cs.cuda() if rot else None, qa if rot else None, n, qdim)

    def turn(x):  # [..., rot] of row t
        x = x.double().clone()
        c, s = (cs[:, :, k].double().view(T, *[1] * (x.dim() - 2), rdims // 2) for k in range(2))
        a, b = x[..., 0:rdims:2].clone(), x[..., 1:rdims:2].clone()
        x[..., 0:rdims:2], x[..., 1:rdims:2] = a * c - b * s, b * c + a * s
        return x
    x = src.double()
    row = x[:, :R] / (x[:, :R].pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * w.double()
    want = torch.full((T + 3, n), 7.0, dtype=torch.float64)
    for t in range(1, T):
        want[slots[t], :R] = row[t]
        want[slots[t], R:] = turn(x[:, R:n])[t]
    # fp32: a few units, the mean over R of them; a rotation's two products of up to 4 x 4; bf16 results 2^-9 of theirs
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((cache.cpu().double()[:, 0] - want).abs() <= want.abs() * (eps + 64 * 2.0 ** -24) + 32 * 2.0 ** -24).all()
    if rot:
        q = turn(x[:, n:].view(T, H, qdim + rot)[..., qdim:])
        assert ((qa.cpu().double()[..., R:] - q).abs() <= 64 * 2.0 ** -24 + q.abs() * 2.0 ** -20).all()
        assert (qa[..., :R] == 7.0).all()
