"""Queries of zeros (padding of a batch, warm-up calls): every row ties at 0, so
each partition keeps its first rows.  One query and a batch that is answered one
query at a time agree with the packet layout over rows in order and shuffled over
the partitions, and take no multiple of the time of any other query.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# partitions of fewer rows than M, of one slice, of few and of many; -0.0 is a zero as well
@pytest.mark.parametrize("rows,split,M", [(300, 20, 17), (700, 8, 64), (8330, 2, 64), (70000, 1, 20), (140000, 2, 48), (40000, 64, 1)])
@pytest.mark.parametrize("seed", [0, 7])
@pytest.mark.parametrize("zero", [0.0, -0.0])
def test_rows_of_a_zero_query(acc, gpu, rows, split, M, seed, zero):
    cols, ck = 90, split * M
    k = min(ck, rows, 960)
    csr = acc.CSRMatrix.generate(rows, cols, deg=(1, 12), val_kind=acc.VAL_ABSNORMAL, seed=rows)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split, shuffle_seed=seed))
    x = np.full((3, cols), zero, np.float32)
    x[1] = np.random.default_rng(rows).standard_normal(cols)
    X = acc.DeviceBuffer.from_numpy(x)
    got = {}
    for mode in (acc.BATCH_SPARSE, acc.BATCH_SINGLE):
        g.set_batch_mode(mode)
        out = acc.DeviceBuffer.from_numpy(np.full((3, k, 2), 9, np.int32))
        g.topk_lowbit_batch(X, np.full(3, k, np.int32), ck, out, k)
        acc.synchronize()
        got[mode] = out.numpy()
    np.testing.assert_array_equal(got[acc.BATCH_SINGLE], got[acc.BATCH_SPARSE])
    if seed == 0:  # the first M rows of each partition, all of a score of 0
        size = rows // split
        ends = [rows if p == split - 1 else (p + 1) * size for p in range(split)]
        best = [r for p in range(split) for r in range(p * size, min(ends[p], p * size + M))][:k]
        np.testing.assert_array_equal(got[acc.BATCH_SINGLE][0, :len(best), 1], best)


@pytest.mark.parametrize("split", [1, 16])
def test_time_of_zero_queries(acc, gpu, split):
    csr = acc.CSRMatrix.generate(200000, 120, deg=(5, 30), val_kind=acc.VAL_ABSNORMAL, seed=5)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split))
    g.set_batch_mode(acc.BATCH_SINGLE)
    out, us = acc.DeviceBuffer((2, 16, 2), np.int32), {}
    for kind in ("usual", "zeros"):
        x = np.zeros((2, 120), np.float32) if kind == "zeros" else np.random.default_rng(1).random((2, 120), dtype=np.float32)
        X, ks, best = acc.DeviceBuffer.from_numpy(x), np.full(2, 16, np.int32), np.inf
        for _ in range(4):  # the first run warms up
            a, b = acc.Event(), acc.Event()
            a.record()
            for _ in range(10):
                g.topk_lowbit_batch(X, ks, 16 * split, out, 16)
            b.record()
            best = min(best, a.elapsed_ms(b) * 100)
        us[kind] = best
    assert us["zeros"] < 3 * us["usual"], us  # row after row rescanned: 4 to 30 times
