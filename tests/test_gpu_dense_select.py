"""dense_select_regs / dense_select where one hands over to the other and at
the edges of their lists: partitions of one slice up to past the 1,024 slices
held in registers, up to and past 32 rows kept, partial slices, slices that
hold more of the best rows than a list, more candidates than lanes, every
lanes-per-row group of the rescoring.  Results are compared with the oracle
exactly.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def check(acc, csr, split, ck, nq, k, bits=8, signed=False, X=None):
    ptr, idx, val = csr.arrays()
    q, _ = O.quantize(val, bits, signed)
    g = acc.GpuMatrix(csr, csr.pack(bits=bits, split=split, is_signed=signed))
    g.set_batch_mode(acc.BATCH_DENSE)
    if X is None:
        X = acc.generate_queries(nq, csr.cols, seed=ck)
    out = acc.DeviceBuffer((nq, k, 2), np.int32)
    g.topk_lowbit_batch(acc.DeviceBuffer.from_numpy(X), np.full(nq, k, np.int32), ck, out, k)
    acc.synchronize()
    got = out.numpy()
    for i in range(nq):
        _, rows, vals = O.two_stage(ptr, idx, val, q, X[i], csr.cols, g.info.group, split, ck, k)
        np.testing.assert_array_equal(got[i, :, 1], rows)
        np.testing.assert_array_equal(got[i, :, 0].view(np.float32), vals)


@pytest.mark.parametrize("slices,split,M", [(1, 8, 4), (2, 8, 16), (63, 2, 16), (64, 2, 32), (65, 2, 33), (256, 2, 16),
                                            (257, 2, 32), (512, 1, 24), (513, 1, 16), (1024, 1, 32), (1025, 1, 16)])
def test_partition_slices(acc, gpu, slices, split, M):
    rows = slices * 64 * split - 5  # a partial last slice
    csr = acc.CSRMatrix.generate(rows, 90, deg=(4, 9), seed=slices)
    check(acc, csr, split, split * M, 6, min(split * M, 50))


# mean rows of 3, 10, 20, 50 and 90 entries: 2, 4, 8, 16 and 32 lanes per row
@pytest.mark.parametrize("deg", [(1, 5), (5, 15), (10, 30), (30, 70), (60, 120)])
@pytest.mark.parametrize("M", [1, 16, 31])
def test_rescoring_groups(acc, gpu, deg, M):
    csr = acc.CSRMatrix.generate(6000, 400, deg=deg, seed=deg[1])
    check(acc, csr, 8, 8 * M, 5, min(8 * M, 40))


# rows of one length stay in order, so these lie in neighbouring slots: lists that drop rows, and tied candidates past 64
@pytest.mark.parametrize("count,tied", [(6, False), (40, False), (40, True), (300, True)])
def test_best_rows_share_slices(acc, gpu, count, tied):
    rng = np.random.default_rng(count)
    rows, cols = 16000, 100
    ptr = np.arange(rows + 1, dtype=np.int64) * 10
    idx = np.tile(np.arange(10, dtype=np.int32) * 10, rows)
    val = (0.1 + 0.05 * rng.random(rows * 10)).astype(np.float32)
    for first in (0, 3990, 9000):
        part = slice(first * 10, (first + count) * 10)
        val[part] = 1.0 if tied else 0.9 + 0.1 * rng.random(count * 10)
    csr = acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)
    X = np.abs(acc.generate_queries(4, cols, seed=count)) + 0.5
    check(acc, csr, 4, 64, 4, 60, X=X.astype(np.float32))
