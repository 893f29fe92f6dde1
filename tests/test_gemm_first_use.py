"""The counters that products with split sums combined in the launch share are made by the first such product of a process (csrc/gemm.hip
sk_counters): that one under graph capture, and beside another thread's capture, each in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEAD = """
import sys
sys.path[:0] = [%r, %r]
import torch
from llmss_amd.ops import hip as H

def rand(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()

def combines(M, N, K, glu=False):
    return H.lib().gemm_plan(M, N, K, False, glu, False)[0] >> 8 & (2048 | 256) == 2048 | 256

def near(y, z, x, w, slope=1.0):  # sums in 32 bits in any order, a rounding to bf16
    lim = slope * (x.shape[1] + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    return ((y.double() - z).abs() <= lim + 2.0 ** -8 * (z.abs() + lim) + 2.0 ** -18).all()

H._GEMM_WS.get(64 << 20, torch.device("cuda", 0))
""" % (ROOT, os.path.join(ROOT, "tests"))


def child(body):
    r = subprocess.run([sys.executable, "-c", HEAD + body], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1:] == ["done"], r.stdout[-2000:] + r.stderr[-4000:]


def test_first_combining_products_under_capture():
    """No counters can be made there: a plain product leaves slabs and sums them in a launch of its own, with bias and activation, or its gate,
    and one with the rotation and the cache write runs unsplit. Replays among eager launches, which combine."""
    child("""
M, N, K = 40, 384, 1920
assert combines(M, N, K) and combines(M, N, K, True)
x, w, b = rand(1, M, K), rand(2, N, K) * K ** -0.5, rand(3, N)
z = x.double() @ w.double().t()
want = torch.nn.functional.gelu(z + b.double())
gate, up = (t.reshape(M, -1) for t in z.view(M, N // 32, 2, 16).unbind(2))
gated = torch.nn.functional.silu(gate) * up
from test_qkv_untuned import check
nh, nkv, D, rot = 4, 1, 64, 64
pos, slots = torch.arange(M).cuda() * 2, torch.randperm(48, generator=torch.Generator().manual_seed(4))[:M].cuda()
ang = torch.rand(90, rot // 2, generator=torch.Generator().manual_seed(5)).cuda() * 6
cos, sin = ang.cos(), ang.sin()
kc, vc = (torch.zeros(3, nkv, 16, D, dtype=torch.bfloat16, device="cuda") for _ in range(2))
qkv = lambda: H.linear_qkv(x, w, b, pos, cos, sin, kc, vc, slots, nh, nkv, D, rot, "gptj", True, *H.lib().gemm_plan(M, N, K, False, False, False))
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    y = H.linear(x, w, b, act="gelu")
    g = H.linear(x, w, glu=True)
    q = qkv()
lim = 1.2 * gate.abs().max() + 1.2 * up.abs().max()
for _ in range(3):
    for t in (y, g, q):
        t.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert near(y, want, x, w, 1.13)
    assert ((g.double() - gated).abs() <= 2.0 ** -8 * gated.abs() + lim * 1928 * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()).max() + 1e-6).all()
    check(q, kc, vc, x, w, b, pos, slots, cos, sin, nh, nkv, D, rot, "gptj")
    assert near(H.linear(x, w, b, act="gelu"), want, x, w, 1.13)
    check(qkv(), kc, vc, x, w, b, pos, slots, cos, sin, nh, nkv, D, rot, "gptj")
print("done")
""")


def test_first_combining_product_beside_a_capture():
    """Another thread's capture neither refuses the product nor is ended by it. (Into rows that are there: an allocation by torch would end it.)"""
    child("""
import threading
M, N, K = 40, 384, 1920
assert combines(M, N, K)
x, w = rand(1, M, K), rand(2, N, K) * K ** -0.5
a, got, side = torch.arange(5.0, device="cuda"), [], torch.cuda.Stream()
out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")

def work():
    try:
        with torch.cuda.stream(side):
            got.append(H.linear(x, w, out=out))
    except Exception as e:
        got.append(e)

torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    y = a * 2
    t = threading.Thread(target=work)
    t.start()
    t.join()
    y = y + 1
side.synchronize()
assert torch.is_tensor(got[0]), got
assert near(got[0], x.double() @ w.double().t(), x, w)
for _ in range(2):
    y.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, a * 2 + 1)
print("done")
""")
