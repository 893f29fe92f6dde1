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
