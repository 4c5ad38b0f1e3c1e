"""The specialized GEMM's plans whose last, partial round of tiles runs as K pieces: against the float64 product of the
oracle's weights at the remainders of tiles (M, N) and K ranges, in float32 and bfloat16, bit for bit across calls and between
mbq_matmul and mbq_matmul_noalloc, on a layer of a stack and on none, and recorded first thing into a graph (where there is
no workspace yet and the tiles run whole)."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import mashbox_amd.int8 as I8
import mashbox_amd.kernels as KQ
from mashbox_amd import _lib as LIB
from oracle import gen as G
from oracle import ref as R
from tests._check import assert_product_dev

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CASES = [(R.Q4_K, 512, 5120, 6144), (R.Q4_K, 257, 5003, 6144), (R.Q6_K, 511, 5120, 17408), (R.Q8_0, 500, 4999, 10272),
         (R.Q4_0, 512, 5120, 6176), (R.Q5_K, 256, 5120, 6144), ("int8", 384, 34816, 1024), ("int8", 300, 5120, 10288)]


def _x(m, k, cuda, seed=0):
    return torch.from_numpy(G.acts(np.random.default_rng(seed), m, k).astype(np.int16)).view(torch.bfloat16).to(cuda)


def _weight(t, n, k, cuda, seed=3):
    rng = np.random.default_rng(seed)
    if t == "int8":
        q, s = G.int8_weights(rng, n, k)
        return LIB.I8T, I8.repack(torch.from_numpy(q).to(cuda), torch.from_numpy(s).to(cuda)).buf, torch.from_numpy(q).to(cuda).double() * torch.from_numpy(s).to(cuda).double()[:, None]
    raw = G.RAW[t](rng, n, k)
    p = KQ.repack_host(t, raw, (n, k), tiled=True).to(cuda)
    return p.t, p.buf, KQ.dequant(p).double()


def _call(fn, t, buf, x, m, n, k, y, layer=None, nl=1):
    LIB.check(fn(t, buf.data_ptr(), 0, layer, nl, x.data_ptr(), m, n, k, y.data_ptr(), int(y.dtype == torch.bfloat16),
                 LIB.current_stream()), "matmul")
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("t,m,n,k", CASES)
def test_pieces_against_the_exact_product(t, m, n, k, cuda):
    tt, buf, w = _weight(t, n, k, cuda)
    plan = LIB.gemm_plan(tt, m, n, k)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        SEEN.append(plan[1:3] == (256, 192) and plan[3] > 1)
    x = _x(m, k, cuda)
    ref = x.double() @ w.T
    L = LIB.lib()
    y = _call(L.mbq_matmul, tt, buf, x, m, n, k, torch.full((m, n), 9.0, device=cuda))
    assert_product_dev(y, ref, f"{t} {m}x{n}x{k} {LIB.plan_str(tt, m, n, k)}")
    z = _call(L.mbq_matmul_noalloc, tt, buf, x, m, n, k, torch.full((m, n), 9.0, device=cuda))
    assert torch.equal(z.view(torch.int32), y.view(torch.int32))
    b = _call(L.mbq_matmul, tt, buf, x, m, n, k, torch.empty((m, n), dtype=torch.bfloat16, device=cuda))
    assert torch.equal(b.view(torch.int16), y.to(torch.bfloat16).view(torch.int16))


SEEN = []


@pytest.mark.gpu
def test_the_cases_above_run_pieces():
    if not SEEN:
        pytest.skip("runs after test_pieces_against_the_exact_product, on 256 CUs")
    assert sum(SEEN) >= 5, SEEN


@pytest.mark.gpu
def test_layers_of_a_stack(cuda):
    m, n, k = 512, 5120, 6144
    tt, buf, w = _weight(R.Q4_K, n, k, cuda)
    stack = torch.cat([torch.zeros_like(buf), buf])
    x = _x(m, k, cuda)
    layer = torch.tensor(1, dtype=torch.int32, device=cuda)
    y = _call(LIB.lib().mbq_matmul, tt, stack, x, m, n, k, torch.empty((m, n), device=cuda), layer.data_ptr(), 2)
    assert_product_dev(y, x.double() @ w.T, "layer 1 of 2")
    layer.fill_(2)
    y = _call(LIB.lib().mbq_matmul, tt, stack, x, m, n, k, torch.zeros((m, n), device=cuda), layer.data_ptr(), 2)
    assert bool(torch.isnan(y).all())


SCRIPT = r"""
import sys
sys.path.insert(0, sys.argv[1])
import torch
import tests.test_gpu_gemm_pieces as P
from mashbox_amd import _lib as LIB
dev = torch.device("cuda", 0)
m, n, k = 512, 5120, 6144
tt, buf, w = P._weight(12, n, k, dev)
x, y = P._x(m, k, dev), torch.empty((m, n), dtype=torch.bfloat16, device=dev)
torch.cuda.synchronize()
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g):
    P._call(LIB.lib().mbq_matmul, tt, buf, x, m, n, k, y)
whole = None
for _ in range(3):
    y.zero_()
    g.replay()
    torch.cuda.synchronize()
    P.assert_product_dev(y, x.double() @ w.T, "recorded before any eager call")
    whole = y.clone() if whole is None else whole
    assert torch.equal(y, whole)
eager = P._call(LIB.lib().mbq_matmul, tt, buf, x, m, n, k, torch.empty_like(y))
torch.cuda.synchronize()
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g):
    P._call(LIB.lib().mbq_matmul, tt, buf, x, m, n, k, y)
for _ in range(3):
    y.zero_()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, eager), "a recorded call differs from the eager call"
    P._call(LIB.lib().mbq_matmul, tt, buf, x, m, n, k, torch.empty_like(y))
print("pieces capture ok", flush=True)
"""


@pytest.mark.gpu
def test_recorded_before_and_after_an_eager_call():
    r = subprocess.run([sys.executable, "-c", SCRIPT, ROOT], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr[-4000:])
    assert r.returncode == 0 and "pieces capture ok" in r.stdout


SPARE_SCRIPT = r"""
import sys
sys.path.insert(0, sys.argv[1])
import torch
import tests.test_gpu_gemm_pieces as P
from mashbox_amd import _lib as LIB
dev = torch.device("cuda", 0)
L = LIB.lib()
a, b = (512, 5120, 6144), (16, 1024, 5120)                  # pieces; a K split that has no other form
ta, bufa, wa = P._weight(12, *a[1:], dev)
pb = P.KQ.repack_host(12, P.G.RAW[12](P.np.random.default_rng(4), *b[1:]), b[1:]).to(dev)
tb, bufb = pb.t, pb.buf
assert LIB.gemm_plan(tb, *b)[3] > 1, "the case must split K"
xa, xb = P._x(a[0], a[2], dev), P._x(b[0], b[2], dev)
ya, yb = torch.empty(a[:2], device=dev), torch.empty(b[:2], device=dev)
eager = P._call(L.mbq_matmul, tb, bufb, xb, *b, torch.empty_like(yb))
torch.cuda.synchronize()
ga, gb = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
with torch.cuda.graph(ga, stream=torch.cuda.Stream()):
    P._call(L.mbq_matmul, ta, bufa, xa, *a, ya)
with torch.cuda.graph(gb, stream=torch.cuda.Stream()):
    P._call(L.mbq_matmul, tb, bufb, xb, *b, yb)
for _ in range(3):
    ya.zero_(), yb.zero_()
    ga.replay()
    gb.replay()
    torch.cuda.synchronize()
    P.assert_product_dev(ya, xa.double() @ wa.T, "pieces' product")
    assert torch.equal(yb, eager)
    P._call(L.mbq_matmul, tb, bufb, xb, *b, torch.empty_like(yb))
print("spare ok", flush=True)
"""


@pytest.mark.gpu
def test_pieces_leave_the_spare_workspace_to_split_k():
    """after one eager split-K call, a pieces product recorded on one new stream and a split-K product on another: the first
    can do without a workspace, the second is refused without one"""
    r = subprocess.run([sys.executable, "-c", SPARE_SCRIPT, ROOT], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr[-4000:])
    assert r.returncode == 0 and "spare ok" in r.stdout
