"""The causal convolution of a decode step - rows and tails in one launch - with the input itself added, with and without bias and
activation, against float64 and against the form of portions: registers (C % 4 == 0, up to 9 taps) and the general kernel."""
import pytest
import torch

from llmss_amd import ops

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                             (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("residual,bias,silu", [(True, False, False), (True, True, False), (True, False, True), (False, True, True)])
@pytest.mark.parametrize("C,taps", [(40, 4), (70, 3), (1032, 9), (8, 1), (12, 2), (16, 12), (72, 5), (40, 6), (16, 8)])
def test_single_rows(device, dtype, out_dtype, residual, bias, silu, C, taps):
    gen = torch.Generator().manual_seed(C + taps)
    B, steps, R = 5, 14, taps - 1
    xs = torch.randn(steps, B, C, generator=gen).to(dtype)
    w, b = (torch.randn(C, taps, generator=gen) * taps ** -0.5).to(dtype), torch.randn(C, generator=gen).to(dtype)
    slots = torch.tensor([4, 0, -1, 2, 5], dtype=torch.int32)
    first = torch.tensor([0, 3, 0, 1, 20])  # a sequence's rows before this step: none, fewer than the tail, more
    state = torch.randn(6, max(R, 1), C, generator=gen)[:, :R].contiguous()
    past = torch.zeros(B, R, C, dtype=torch.float64)  # the inputs before, zeros before position 0
    for s in range(B):
        if slots[s] >= 0 and first[s]:
            n = min(R, int(first[s]))
            past[s, R - n:] = state[slots[s], R - n:].double()
    y, z = [state.clone().to(device) for _ in range(2)]
    cu = torch.arange(B + 1, dtype=torch.int32).to(device)
    for t in range(steps):
        ctx = torch.where(slots >= 0, first + t + 1, 0).int().to(device)  # (the third row is a padded one)
        args = (cu, ctx, slots.to(device), residual, silu, out_dtype)
        got, other = (ops.causal_conv(xs[t].to(device), w.to(device), s if R else None, *args, bias=b.to(device) if bias else None,
                                      single=one) for s, one in ((y, True), (z, False)))
        full = torch.cat([past, xs[t].double()[:, None]], 1)
        want = (full * w.double().t()).sum(1) + (xs[t].double() if residual else 0) + (b.double() if bias else 0)
        want = want * torch.sigmoid(want) if silu else want
        past = full[:, 1:]
        live = slots >= 0
        # fp32 sums of at most 14 terms, v_rcp / v_exp in the sigmoid of bf16 results; one rounding to the result's type
        tol = 2.0 ** -8 if out_dtype == torch.bfloat16 else 2e-6
        for r in (got, other):
            r = r.double().cpu()[live]
            assert ((r - want[live]).abs() <= tol * (want[live].abs() + (full.abs() * w.double().t().abs()).sum(1)[live])
                    + 1e-6).all(), t
    if R:
        for s in range(B):
            if slots[s] >= 0:
                assert torch.equal(y[slots[s]].cpu().double(), past[s])
        assert torch.equal(y.cpu(), z.cpu()) and torch.equal(y[[1, 3]].cpu(), state[[1, 3]])


# portions over strips of sixteen rows: strips within one, over its first rows, over a border, past the last row and with a padded sequence
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("residual,bias,silu", [(True, False, False), (False, True, True)])
@pytest.mark.parametrize("C,taps", [(40, 4), (1032, 9), (12, 2), (70, 3), (12, 5), (40, 7), (70, 4)])
# strips from 256 rows on; that for strips within one portion in bf16, of 2, 4, 5 and 9 taps
@pytest.mark.parametrize("lens", [[19, 100, 1, 16, 40, 35], [59, 100, 1, 26, 40, 35], [119, 300, 1, 16, 40, 35], [32, 200, 1, 16, 96, 39]])
def test_strips_of_portions(dtype, out_dtype, residual, bias, silu, C, taps, lens):
    gen = torch.Generator().manual_seed(C + taps)
    first, slots = [0, 7, 2, 0, 3, 0], [4, 0, 1, 2, -1, 5]
    T, R = sum(lens), taps - 1
    x = torch.randn(T, C, generator=gen).to(dtype)
    w, b = (torch.randn(C, taps, generator=gen) * taps ** -0.5).to(dtype), torch.randn(C, generator=gen).to(dtype)
    state = torch.randn(6, R, C, generator=gen)
    want, size, t = torch.zeros(T, C, dtype=torch.float64), torch.zeros(T, C, dtype=torch.float64), 0
    for n, p0, s in zip(lens, first, slots):
        if s >= 0:
            past = torch.zeros(R, C, dtype=torch.float64)
            if p0:
                past[max(R - p0, 0):] = state[s, max(R - p0, 0):].double()
            full = torch.cat([past, x[t:t + n].double()])
            for k in range(taps):
                want[t:t + n] += full[k:k + n] * w[:, k].double()
                size[t:t + n] += (full[k:k + n] * w[:, k].double()).abs()
            want[t:t + n] += (x[t:t + n].double() if residual else 0) + (b.double() if bias else 0)
        t += n
    size += want.abs() + x.double().abs() + 1
    want = want * torch.sigmoid(want) if silu else want
    ctx = torch.tensor([n + p if s >= 0 else 0 for n, p, s in zip(lens, first, slots)], dtype=torch.int32)
    got = ops.causal_conv(x.cuda(), w.cuda(), state.clone().cuda(), torch.tensor([0] + lens).cumsum(0).int().cuda(), ctx.cuda(),
                          torch.tensor(slots, dtype=torch.int32).cuda(), residual, silu, out_dtype, bias=b.cuda() if bias else None)
    # sums of up to 11 terms in fp32, 2^-24 of their absolute sum each; the activation's slope is under 1.1, its own error 8 units; bf16 results 2^-8
    lim = size * 24 * 2.0 ** -24 + (want.abs() * 2.0 ** -8 if out_dtype == torch.bfloat16 else 0)
    live = torch.cat([torch.full((n,), s >= 0) for n, s in zip(lens, slots)])
    assert ((got.cpu().double() - want).abs() <= lim)[live].all()
    assert (got.cpu()[~live] == 0).all()
