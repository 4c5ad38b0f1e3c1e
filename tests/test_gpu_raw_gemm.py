"""mbq_gemm_raw: the exact path's product of more than 8 bfloat16 rows on the file's blocks (types without kernel planes).

Decode: x = the unit rows, so that output (k, n) is weight value (n, k) itself: the bits of the rebuild (its bfloat16 terms
add back to it exactly; a zero may lose its sign in the sum).
Product: against the float64 product of the rebuilt weights, at the edges of its tiles (32, 64, 128 and 256 rows by 256
weight rows, K steps of 64 with half a step left over) and of its K pieces. Every product is exact and K of them are
added in float32: relative 2-norm below sqrt(K) 2^-24 for random signs, 1e-6 at K <= 5120, and measured 3e-7.
"""
import ctypes

import numpy as np
import pytest
import torch

from mashbox_amd import _lib as LIB
import mashbox_amd.ops as OPS
from oracle import ref as R
from tests.test_gpu_raw_types import NAME, _weights

TOL = 1e-6


def _bound(x, w, ref):
    """TOL of the result's norm, or of the norm that random signs would give it (a few outputs may cancel by chance)"""
    typical = 1.25 * float((x.double().abs() @ w.double().abs().T).norm()) / w.shape[1] ** 0.5
    return TOL * max(float(ref.norm()), typical)


def _gemm_raw(t, raw, x, n, k, dtype=torch.float32):
    m = x.shape[0]
    y = torch.full((m, n), 7.0, dtype=dtype, device=x.device)
    nb = LIB.check(LIB.lib().mbq_gemm_raw_work(m, n, k), "work")
    work = torch.empty(nb, dtype=torch.uint8, device=x.device)
    p = ctypes.c_void_p
    LIB.check(LIB.lib().mbq_gemm_raw(t, p(raw.data_ptr()), p(x.data_ptr()), m, n, k, p(y.data_ptr()),
                                     int(dtype == torch.bfloat16), p(work.data_ptr()), nb,
                                     p(torch.cuda.current_stream().cuda_stream)), "gemm_raw")
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("t", R.EXACT_ONLY, ids=NAME.get)
def test_unit_rows_give_back_the_weights(t, cuda):
    k, n = 512, 75
    raw = torch.from_numpy(_weights(t, n, k, 77 + t)).to(cuda)
    w = OPS._raw_dequant(raw, t, n, k)
    for x in (torch.eye(k, device=cuda), torch.eye(k, device=cuda)[100:130]):
        y = _gemm_raw(t, raw, x.to(torch.bfloat16), n, k)
        want = x @ w.T
        assert torch.equal(y, want)                                   # by value: -0 and +0 are equal


@pytest.mark.gpu
@pytest.mark.parametrize("t", R.EXACT_ONLY, ids=NAME.get)
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (9, 255, 320), (70, 90, 96), (32, 257, 64), (33, 513, 1280), (64, 70, 4096), (65, 300, 2304),
                                   (129, 256, 5120), (257, 1025, 768), (513, 40, 544)])
def test_gemm_raw_against_the_exact_product(t, m, n, k, cuda):
    k = -(-k // max(32, R.TYPES[t][1])) * max(32, R.TYPES[t][1])
    raw = torch.from_numpy(_weights(t, n, k, 31 * t + m)).to(cuda)
    x = torch.from_numpy(np.random.default_rng(m + n).standard_normal((m, k)).astype(np.float32)).to(cuda).to(torch.bfloat16)
    w = OPS._raw_dequant(raw, t, n, k)
    ref = x.double() @ w.double().T
    y = _gemm_raw(t, raw, x, n, k)
    assert bool(torch.isfinite(y).all())
    assert float((y.double() - ref).norm()) <= _bound(x, w, ref)
    assert torch.equal(_gemm_raw(t, raw, x, n, k).view(torch.int32), y.view(torch.int32))
    yb = _gemm_raw(t, raw, x, n, k, torch.bfloat16)
    assert torch.equal(yb.view(torch.int16), y.to(torch.bfloat16).view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("t", [R.F32, R.F16, R.BF16, R.Q5_1, R.Q3_K, R.IQ4_XS], ids=NAME.get)
@pytest.mark.parametrize("m,n,k", [(16, 300, 2304), (300, 40, 512), (512, 65800, 256)])
def test_non_finite_values_come_out_as_the_float32_product_has_them(t, m, n, k, cuda):
    """infinite and NaN block scales (or values) and activations: the cut terms meet inf - inf and 0 * inf, so those
    outputs are computed again value by value; every output is inf, -inf, NaN or finite as the float64 product is"""
    raw = _weights(t, n, k, 5 * t + m).copy()
    rng = np.random.default_rng(m)
    ts = R.TYPES[t][2]
    at = {R.F32: 0, R.F16: 0, R.BF16: 0, R.Q5_1: 0, R.Q3_K: 108, R.IQ4_XS: 0}[t]
    blocks = raw.reshape(n, -1, ts)
    special = {R.F32: np.array([np.inf, np.nan], np.float32).view(np.uint8).reshape(2, 4),
               R.BF16: np.array([0x7F80, 0x7FC0], np.uint16).view(np.uint8).reshape(2, 2)}.get(
        t, np.array([np.inf, np.nan], np.float16).view(np.uint8).reshape(2, 2))
    for i, row in enumerate(rng.choice(n, 6, replace=False)):
        blocks[row, rng.integers(blocks.shape[1]), at:at + special.shape[1]] = special[i % 2]
    raw_d = torch.from_numpy(raw).to(cuda)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(cuda).to(torch.bfloat16)
    x[1, 3], x[2, 7], x[3, 9] = float("inf"), float("-inf"), float("nan")
    w = OPS._raw_dequant(raw_d, t, n, k)
    keep = torch.cat([torch.arange(min(n, 4000), device=cuda), torch.nonzero(~torch.isfinite(w).all(1)).flatten()])
    ref = x.cpu().double() @ w[keep].cpu().double().T                 # on the host: no library's own shortcuts for zeros
    y = _gemm_raw(t, raw_d, x, n, k)[:, keep].cpu().double()
    assert not torch.isfinite(ref).all()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    assert torch.equal(torch.isinf(y) * y.sign().nan_to_num(), torch.isinf(ref) * ref.sign().nan_to_num())
    f = torch.isfinite(ref)
    assert float((y[f] - ref[f]).norm()) <= TOL * float(ref[f].norm())


@pytest.mark.gpu
def test_qmatmul_takes_it_and_leaves_gradients_and_transforms_to_torch(cuda):
    n, k, t = 96, 1024, R.IQ4_XS
    raw = _weights(t, n, k, 3)
    h = OPS.prepare(raw, t, (n, k))
    x = torch.randn((40, k), device=cuda).to(torch.bfloat16)
    y = OPS.qmatmul(x, h)
    assert torch.equal(y.view(torch.int16), _gemm_raw(t, h.raw, x, n, k, torch.bfloat16).view(torch.int16))
    odd = torch.empty(40 * k + 1, dtype=torch.bfloat16, device=cuda)[1:].view(40, k).copy_(x)   # 2-byte aligned
    assert torch.equal(OPS.qmatmul(odd, h), y)
    xg = x.clone().requires_grad_()
    OPS.qmatmul(xg, h).float().sum().backward()
    w = OPS.dequant(h)
    assert torch.allclose(xg.grad.float(), w.sum(0).expand(40, k), rtol=2e-2, atol=2e-2 * float(w.sum(0).abs().max()))
    yv = torch.func.vmap(lambda r: OPS.qmatmul(r, h))(x.reshape(4, 10, k))
    assert float((yv.reshape(40, n).double() - y.double()).norm()) <= 4e-3 * float(y.double().norm())


def test_argument_checks():
    lib = LIB.lib()
    assert lib.mbq_gemm_raw(R.Q4_K, None, None, 16, 8, 256, None, 0, None, 0, None) < 0        # has planes
    assert lib.mbq_gemm_raw(16, None, None, 16, 8, 256, None, 0, None, 0, None) < 0            # code book type
    assert lib.mbq_gemm_raw(R.F16, None, None, 16, 8, 48, None, 0, None, 0, None) < 0          # K % 32
    assert lib.mbq_gemm_raw(R.Q2_K, None, None, 16, 8, 128, None, 0, None, 0, None) < 0        # K % 256
    assert lib.mbq_gemm_raw(R.Q2_K, None, None, 16, 8, 256, None, 5, None, 0, None) < 0        # out dtype
    assert lib.mbq_gemm_raw(R.Q2_K, None, None, 16, 8, 256, None, 0, None, 0, None) < 0        # NULL pointers
    assert lib.mbq_gemm_raw(R.Q2_K, None, None, 1 << 20, 1 << 20, 256, None, 0, None, 0, None) < 0   # 2^40 outputs
    assert lib.mbq_gemm_raw(R.Q2_K, None, None, 0, 8, 256, None, 0, None, 0, None) == 0
    assert lib.mbq_gemm_raw_work(-1, 8, 256) < 0 and lib.mbq_gemm_raw_work(0, 8, 256) == 0


# --------------------------------------------------------------------------------------------- 1-8 rows (mbq_matmul_raw)
@pytest.mark.gpu
@pytest.mark.parametrize("t", R.EXACT_ONLY, ids=NAME.get)
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (1, 8200, 256), (2, 63, 544), (4, 9, 17408), (5, 130, 8448), (8, 8195, 512)])
def test_decode_rows_against_the_exact_product(t, m, n, k, cuda):
    """1 to 8 waves per row, rows past a block, a K of half a super-block, x in one or several LDS stages; float32 sums as
    above: relative 2-norm 1e-6"""
    from tests.test_gpu_raw_types import _matmul_raw
    k = -(-k // max(32, R.TYPES[t][1])) * max(32, R.TYPES[t][1])
    raw = torch.from_numpy(_weights(t, n, k, 13 * t + m)).to(cuda)
    x = torch.from_numpy(np.random.default_rng(k + n).standard_normal((m, k)).astype(np.float32)).to(cuda).to(torch.bfloat16)
    w = OPS._raw_dequant(raw, t, n, k)
    ref = x.double() @ w.double().T
    y = _matmul_raw(t, raw, x, n, k, False)
    assert float((y.double() - ref).norm()) <= _bound(x, w, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("t", R.EXACT_ONLY, ids=NAME.get)
def test_decode_rows_on_any_bytes(t, cuda):
    """blocks of random bytes, non-finite and overflowing scales (values) among them, and non-finite activations: inf, -inf
    and NaN where the float64 product of the rebuilt values has them, wherever no float32 sum can overflow on the way"""
    from tests.test_gpu_raw_types import _matmul_raw
    k, n = 512, 700
    rng = np.random.default_rng(40 + t)
    raw = _weights(t, n, k, 5).copy()
    blocks = raw.reshape(n, -1, R.TYPES[t][2])
    for row in range(0, n, 2):
        if t == R.MXFP4:
            blocks[row, rng.integers(blocks.shape[1]), 0] = rng.integers(246, 256)
        else:
            blocks[row, rng.integers(blocks.shape[1])] = rng.integers(0, 256, blocks.shape[2], dtype=np.uint8)
    raw_d = torch.from_numpy(raw).to(cuda)
    w = OPS._raw_dequant(raw_d, t, n, k).cpu().double()
    x = torch.from_numpy((rng.standard_normal((3, k)) * 2.0 ** -10).astype(np.float32)).to(torch.bfloat16)
    x[1, 5], x[2, 7] = float("inf"), float("nan")
    ref = x.double() @ w.T
    y = _matmul_raw(t, raw_d, x.to(cuda), n, k, False).cpu().double()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(y[inf], ref[inf])
    f = torch.isfinite(ref)
    assert f.any() and bool(((y[f] - ref[f]).abs() <= 1e-5 * (x[0].double().abs() @ w.nan_to_num(0, 0, 0).abs().T).expand(3, n)[f] + 1e-30).all())
