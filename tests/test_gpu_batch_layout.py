"""The layout ACC_BATCH_AUTO picks on an untuned handle, told by its kernels: a
batch on the matrix cores is four, any other three.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def kernels(acc, g, nq, ck, k):
    x = acc.DeviceBuffer.from_numpy(acc.generate_queries(nq, g.info.cols, seed=1))
    out = acc.DeviceBuffer((nq, k, 2), np.int32)
    g.set_profiling(True)
    g.topk_lowbit_batch(x, np.full(nq, k, np.int32), ck, out, k)
    acc.synchronize()
    n = len(g.stage_times())
    g.set_profiling(False)
    return n


# (rows, cols, entries per row, split, CK): batches on the matrix cores (us packets / matrix cores)
CASES = [
    ((20000, 500, (40, 100), 32, 512), {1: False, 8: True, 15: True, 16: True, 100: True}),   # 66 / 38
    ((20000, 500, (40, 100), 16, 1024), {2: False, 8: False, 16: False, 64: False}),          # 84 / 147: full lists
    ((3000, 120, (5, 20), 16, 256), {2: False, 8: False}),                                    # 30 / 38: lists of fewer than M
    ((2000000, 64, (2, 5), 32, 512), {1: False, 8: True, 16: True, 17: True}),                # 127 / 75
    ((20000, 1500, (20, 60), 16, 128), {2: False, 40: False}),                                # too wide for them
]


@pytest.mark.parametrize("shape,want", CASES)
def test_layout(acc, gpu, shape, want):
    rows, cols, deg, split, ck = shape
    csr = acc.CSRMatrix.generate(rows, cols, deg=deg, seed=rows)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split))
    assert {nq: kernels(acc, g, nq, ck, 50) == 4 for nq in want} == want


def test_crossover_of_the_caller(acc, gpu):
    csr = acc.CSRMatrix.generate(20000, 500, deg=(40, 100), seed=3)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=16))
    g.set_batch_mode(acc.BATCH_AUTO, 5)
    assert [kernels(acc, g, nq, ck, 20) for nq in (4, 5, 40) for ck in (64, 1024)] == [3, 3, 4, 4, 4, 4]
    g.set_batch_mode(acc.BATCH_AUTO)  # 0 keeps it
    assert [kernels(acc, g, nq, 64, 20) for nq in (4, 5)] == [3, 4]
    for mode, n in ((acc.BATCH_SPARSE, 3), (acc.BATCH_DENSE, 4), (acc.BATCH_SINGLE, 3)):
        g.set_batch_mode(mode)
        assert kernels(acc, g, 9, 1024, 20) == n
