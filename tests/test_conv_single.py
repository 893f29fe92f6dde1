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
