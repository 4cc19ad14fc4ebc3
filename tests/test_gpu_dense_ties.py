"""Batches on the matrix cores where many rows tie: queries of zeros (as in a
padded batch), matrices of ones and queries of a few terms, the best rows side
by side; partitions of few slices and at the edges of the kernels' sizes, with
a partial last slice.  All candidates are compared with the packet layout, and
such a batch takes no multiple of the time of any other.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def queries(kind, nq, cols, rng):
    x = rng.standard_normal((nq, cols)).astype(np.float32)
    if kind == "zeros":
        x[:] = 0
        x[0, 0] = 1  # one column
    elif kind == "few":
        for q in range(nq):
            x[q] = np.isin(np.arange(cols), rng.permutation(cols)[:8])
    elif kind == "same_sign":
        x = np.abs(x)
    return x


def matrix(acc, kind, rows, cols, deg, signed, rng):
    csr = acc.CSRMatrix.generate(rows, cols, deg=deg, val_kind=acc.VAL_NORMAL if signed else acc.VAL_ABSNORMAL, seed=rows)
    ptr, idx, val = csr.arrays()
    if kind == "few":
        val = np.ones_like(val)
    elif kind == "same_sign":  # a run of good rows
        val = val.copy()
        val[ptr[rows // 3]:ptr[rows // 3 + min(rows // 8, 3000)]] *= 3
    else:
        return csr
    return acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)


# slices per partition: 2 (the last one partial), 64, 65, 256, 257, 512, 513, 1024
@pytest.mark.parametrize("rows,split", [(700, 8), (8200, 2), (8330, 2), (65536, 4), (65800, 4), (65500, 2), (65700, 2), (65536, 1)])
@pytest.mark.parametrize("kind", ["zeros", "few", "same_sign", "usual"])
@pytest.mark.parametrize("M,bits,signed", [(1, 8, False), (16, 4, True), (32, 8, False)])
def test_candidates_of_ties(acc, gpu, rows, split, kind, M, bits, signed):
    rng = np.random.default_rng(rows + M)
    cols, nq, ck = 120, 9, split * M
    csr = matrix(acc, kind, rows, cols, (5, 30), signed, rng)
    g = acc.GpuMatrix(csr, csr.pack(bits=bits, split=split, is_signed=signed))
    X = acc.DeviceBuffer.from_numpy(queries(kind, nq, cols, rng))
    got = {}
    for mode in (acc.BATCH_SPARSE, acc.BATCH_DENSE):
        g.set_batch_mode(mode)
        out = acc.DeviceBuffer.from_numpy(np.full((nq, ck, 2), 9, np.int32))
        g.topk_lowbit_batch(X, np.full(nq, ck, np.int32), ck, out, ck)
        acc.synchronize()
        got[mode] = out.numpy()
    np.testing.assert_array_equal(got[acc.BATCH_DENSE], got[acc.BATCH_SPARSE])


def call_us(acc, g, x, ck, k):
    nq = len(x)
    xd, out = acc.DeviceBuffer.from_numpy(x), acc.DeviceBuffer((nq, k, 2), np.int32)
    ks, best = np.full(nq, k, np.int32), np.inf
    for _ in range(4):  # the first run warms up
        a, b = acc.Event(), acc.Event()
        a.record()
        for _ in range(10):
            g.topk_lowbit_batch(xd, ks, ck, out, k)
        b.record()
        best = min(best, a.elapsed_ms(b) * 100)
    return best


@pytest.mark.parametrize("kind", ["zeros", "few"])
def test_time_of_ties(acc, gpu, kind):
    rng = np.random.default_rng(6)
    csr = matrix(acc, kind, 400000, 500, (40, 100), False, rng)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=16))
    g.set_batch_mode(acc.BATCH_DENSE)
    usual = call_us(acc, g, queries("usual", 8, 500, rng), 512, 100)
    ties = call_us(acc, g, queries(kind, 8, 500, rng), 512, 100)
    assert ties < 4 * usual, (ties, usual)  # slice after slice rescanned: 10 to 30 times


# up to 64 rows a partition, of 1 to 1,094 slices (each way to hold their lists; past 1,024 they are streamed), fewer rows or
# listed rows than M, rows shuffled over the partitions or not: the three layouts agree on ties, and a query of zeros ranks
# the rows in their order
@pytest.mark.parametrize("rows,split,M", [(700, 8, 64), (8330, 2, 64), (20000, 16, 64), (30000, 2, 64), (65800, 4, 33), (70000, 2, 64),
                                          (70000, 1, 64), (70000, 1, 20), (140000, 2, 48), (300, 20, 17)])
@pytest.mark.parametrize("seed", [0, 7])
@pytest.mark.parametrize("kind", ["zeros", "few", "usual"])
def test_every_layout_of_ties(acc, gpu, rows, split, M, seed, kind):
    rng = np.random.default_rng(rows + M)
    cols, nq, ck = 90, 5, split * M
    k = min(ck, rows, 960)
    csr = matrix(acc, kind, rows, cols, (4, 12), False, rng)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split, shuffle_seed=seed))
    x = queries(kind, nq, cols, rng)
    x[nq - 1] = -0.0
    X = acc.DeviceBuffer.from_numpy(x)
    got = {}
    for mode in (acc.BATCH_SPARSE, acc.BATCH_DENSE, acc.BATCH_SINGLE):
        g.set_batch_mode(mode)
        out = acc.DeviceBuffer.from_numpy(np.full((nq, k, 2), 9, np.int32))
        g.topk_lowbit_batch(X, np.full(nq, k, np.int32), ck, out, k)
        acc.synchronize()
        got[mode] = out.numpy()
    np.testing.assert_array_equal(got[acc.BATCH_DENSE], got[acc.BATCH_SPARSE])
    np.testing.assert_array_equal(got[acc.BATCH_SINGLE], got[acc.BATCH_SPARSE])


# more than 32 rows a partition; more than 1,024 slices
@pytest.mark.parametrize("split,M", [(16, 64), (1, 20)])
@pytest.mark.parametrize("kind", ["zeros", "few"])
def test_time_of_ties_in_every_layout(acc, gpu, kind, split, M):
    rng = np.random.default_rng(8)
    csr = matrix(acc, kind, 200000, 300, (5, 30), False, rng)
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split))
    g.set_batch_mode(acc.BATCH_DENSE)
    usual = call_us(acc, g, queries("usual", 8, 300, rng), split * M, 20)
    ties = call_us(acc, g, queries(kind, 8, 300, rng), split * M, 20)
    assert ties < 4 * usual, (ties, usual)  # slice after slice rescanned: 10 to 200 times
