"""Single rows that complete a block of the pooled caches behind their rotation (csrc/attention_pool.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# blocks of one position, of less and more than the rows in flight, over the ends of pages; rows of one access and of several workgroups,
# shapes of single numbers (the means in a launch of their own)
@pytest.mark.parametrize("pool,bs", [(1, 4), (3, 2), (8, 16), (9, 16), (16, 16), (17, 5)])
@pytest.mark.parametrize("T,H,G,dim,vdim,rot,off", [(1, 1, 1, 4, 4, 0, 0), (33, 4, 2, 128, 64, 128, 8), (300, 3, 1, 24, 20, 8, 4), (7, 2, 2, 16, 8, 16, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_means_of_completed_blocks(T, H, G, dim, vdim, rot, off, pool, bs, dtype):
    from llmss_amd.ops import hip
    g = torch.Generator().manual_seed(T + pool)
    nq, nk, nv = H * dim, G * dim, G * vdim
    proj = torch.randn(T, off + nq + nk + nv + (-(off + nq + nk + nv)) % 4 + 4, generator=g).to(dtype).cuda()
    ctx = torch.randint(0, 4 * pool + 1, (T,), generator=g)
    ctx[::2] = ctx[::2] // pool * pool  # half of them complete a block (or are empty)
    if T > 2:
        ctx[:2] = 0
    pages = -(-4 * pool // bs)
    tables = torch.randperm(T * pages, generator=g).view(T, pages).int()
    slots = torch.where(ctx > 0, tables[torch.arange(T), (ctx - 1).clamp_min(0) // bs].long() * bs + (ctx - 1).clamp_min(0) % bs, -1).cuda()
    tables, ctx = tables.cuda(), ctx.int().cuda()
    cu = torch.arange(T + 1, dtype=torch.int32, device="cuda")
    ang = torch.rand(T, rot // 2, generator=g) * 6
    cs = torch.stack([ang.cos(), ang.sin()], -1).contiguous().cuda() if rot else None
    per = -(-bs // pool)
    init = [torch.randn(T * pages, b, n, generator=g).to(dtype).cuda() for b, n in ((bs, nk), (bs, nv), (per, nk), (per, nv))]
    res = []
    for fused in (False, True):
        kc, vc, kp, vp = (t.clone() for t in init)
        q = hip.rope_pairs_cache(proj, off, off + nq, off + nq + nk, cs, kc, vc, slots, H, G, dim, vdim,
                                 pooled=(kp, vp, tables, cu, ctx, pool) if fused else None)
        if not fused:
            hip.pool_update(kc, vc, kp, vp, tables, cu, ctx, pool, max_qlen=1)
        res.append((q, kc, vc, kp, vp))
    for a, b in zip(*res):  # the same sums in the same order
        assert torch.equal(a, b)
    assert T == 1 or not torch.equal(res[1][3], init[2])
