"""lowbit_slicemax / lowbit_select at the edges of their slice lists: rows that
share a slice with more of the best than the list holds, partitions of fewer
slices than rows kept, of one partial slice, and past the slices a thread
keeps in registers.  Candidates are compared with the oracle exactly.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def check(acc, rows, cols, ptr, idx, val, split, ck, bits=8, signed=False):
    csr = acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)
    g = acc.GpuMatrix(csr, csr.pack(bits=bits, split=split, is_signed=signed))
    q, _ = O.quantize(val, bits, signed)
    M = ck // split
    for seed in range(2):
        x = acc.generate_queries(1, cols, seed=seed)[0]
        rd, sd = acc.DeviceBuffer((split * M,), np.int32), acc.DeviceBuffer((split * M,), np.int32)
        n = g.candidates_lowbit(acc.DeviceBuffer.from_numpy(x), ck, rd, sd)
        ro, so = candidates(ptr, idx, q, x, cols, split, M)
        got_r, got_s = rd.numpy().reshape(split, M), sd.numpy().reshape(split, M)
        assert n == sum(len(r) for r in ro)
        for p in range(split):
            np.testing.assert_array_equal(got_r[p, :len(ro[p])], ro[p])
            np.testing.assert_array_equal(got_s[p, :len(ro[p])], so[p])
            assert (got_r[p, len(ro[p]):] == -1).all()


def candidates(ptr, idx, q, x, cols, split, M):
    """Per partition the M best rows by (score, lower row)."""
    xq, _ = O.quantize(x, 8, True)
    score = O.spmv_i32(ptr, idx, q, xq)
    n, size = len(ptr) - 1, (len(ptr) - 1) // split
    rows, scores = [], []
    for p in range(split):
        r = np.arange(p * size, n if p == split - 1 else (p + 1) * size)
        best = r[np.lexsort((r, -score[r].astype(np.int64)))][:M]
        rows.append(best)
        scores.append(score[best])
    return rows, scores


def matrix(rng, rows, cols, lo, hi):
    lengths = rng.integers(lo, hi + 1, rows)
    ptr = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    idx = np.concatenate([np.sort(rng.permutation(cols)[:n]) for n in lengths] or [[]]).astype(np.int32)
    return ptr, idx, np.abs(rng.standard_normal(len(idx))).astype(np.float32)


# rows per partition: one partial slice, one full slice, a few slices, 64 and 65 slices, past 1,024 slices
@pytest.mark.parametrize("per_part,split,M", [(40, 4, 16), (64, 4, 16), (65, 3, 64), (640, 4, 16), (640, 2, 1),
                                              (4096, 2, 16), (4160, 2, 64), (70000, 1, 16)])
def test_partition_sizes(acc, gpu, per_part, split, M):
    rng = np.random.default_rng(per_part + M)
    rows = per_part * split + 7
    ptr, idx, val = matrix(rng, rows, 60, 3, 9)
    check(acc, rows, 60, ptr, idx, val, split, split * M)


# the best rows of a partition all in one slice (equal rows of one length sort together), tied or not
@pytest.mark.parametrize("bits,signed", [(8, False), (4, False), (6, True)])
@pytest.mark.parametrize("jitter", [False, True])
def test_best_rows_share_slices(acc, gpu, bits, signed, jitter):
    rng = np.random.default_rng(5)
    rows, cols, split = 20000, 80, 4
    ptr = np.arange(rows + 1, dtype=np.int64) * 8
    idx = np.tile(np.arange(8, dtype=np.int32) * 10, rows)
    val = np.full(rows * 8, 0.1, np.float32)
    for first in (100, 5200, 5264, 15000):
        block = slice(first * 8, (first + 20) * 8)
        val[block] = 1.0 - (rng.random(160).astype(np.float32) * 0.05 if jitter else 0.0)
    if signed:
        val *= rng.choice([-1.0, 1.0], len(val)).astype(np.float32)
    check(acc, rows, cols, ptr, idx, val.astype(np.float32), split, split * 16, bits, signed)
