"""ops.take_rows on kernel planes takes int32 and int64 ids to the kernel as they are (mbq_lookup_rows): row by row what the
ids mean, also past either end (below zero counts from the end, once more where the 32-bit sum is still below zero, then
clamped), bit for bit the rows of the whole dequantization."""
import numpy as np
import pytest
import torch

from mashbox_amd import _lib as LIB
import mashbox_amd.kernels as KQ
import mashbox_amd.ops as OPS
from oracle import gen as G
from oracle import ref as R


def _row(i, n):
    i = i + n if i < 0 else i
    i = (i + 2 ** 31) % 2 ** 32 - 2 ** 31                             # as an int32
    i = i + n if i < 0 else i
    return min(max(i, 0), n - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("t", [R.Q4_0, R.Q8_0, R.Q4_K, R.Q5_K, R.Q6_K])
@pytest.mark.parametrize("layout", ["tiles", "rowmajor"])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_rows_by_any_id(t, layout, dtype, cuda):
    n, k = 37, 512
    raw = G.RAW[t](np.random.default_rng(t), n, k)
    p = KQ.repack_host(t, raw, (n, k), layout=layout).to(cuda)
    ids = [0, 36, -1, -37, -38, -74, -75, -200, 37, 5000, 2 ** 31 - 1, -2 ** 31]
    if dtype == torch.int64:
        ids += [2 ** 32 + 5, -2 ** 32 - 3, 2 ** 40, 2 ** 31]
    h = OPS.Packed(p, t, (n, k))
    OPS.load_kernels()
    try:
        got = OPS.take_rows(h, torch.tensor(ids + ids, dtype=dtype, device=cuda).reshape(2, -1)[:, ::1])
        empty = OPS.take_rows(h, torch.zeros((0, 3), dtype=dtype, device=cuda))
        one = OPS.take_rows(h, torch.tensor(-2, dtype=dtype))
    finally:
        OPS.load_kernels(module="off")
    want = KQ.dequant(p)[[_row(i, n) for i in ids]]
    assert got.shape == (2, len(ids), k) and torch.equal(got.view(torch.int32), torch.stack([want, want]).view(torch.int32))
    assert empty.shape == (0, 3, k) and torch.equal(one, KQ.dequant(p)[n - 2])


def test_refusals():
    lib = LIB.lib()
    assert lib.mbq_lookup_rows(12, 16, 0, None, 1, 8, 256, 16, 2, 1, 16, None) < 0              # 2-byte ids
    assert lib.mbq_lookup_rows(12, 16, 0, None, 1, 8, 256, 4, 8, 1, 16, None) < 0               # ids at 4 mod 8
    assert lib.mbq_lookup_rows(-9, 16, 0, None, 1, 8, 256, 16, 8, 1, 16, None) < 0              # int8 planes
    assert lib.mbq_lookup_rows(12, 16, 0, None, 1, 8, 256, None, 8, 0, None, None) == 0         # no ids
