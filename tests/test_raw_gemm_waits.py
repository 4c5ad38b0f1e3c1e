"""raw_gemm_kernel's hand-counted vector-memory wait, in the gfx950 code of the built library, by the walk of
tests/test_vmcnt.py: step i issues the DMA of the x stage read after barrier i + 2, so at no barrier may a DMA issued a
whole step earlier still be in flight, and none may be at the end of the kernel (its block's LDS is another's next)."""
from concurrent.futures import ProcessPoolExecutor

from tests.test_vmcnt import _library_functions, check


def test_raw_gemm_dma_lands_before_the_barrier_that_publishes_it():
    kernels = [(f, ins, 1) for f, ins in _library_functions() if "15raw_gemm_kernel" in f]
    assert len(kernels) == 14 * 4, len(kernels)
    with ProcessPoolExecutor(max_workers=8) as ex:
        problems = [p for r in ex.map(check, kernels, chunksize=2) for p in r]
    assert not problems, problems[:4]
