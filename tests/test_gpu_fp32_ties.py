"""FP32 Top-K where many scores reach the threshold of the groups' best keys:
equal scores (a query of zeros, a few levels), the best rows in few groups,
scores that rise in the order in which such groups are read.  Results are
compared exactly (higher score first, the lower row on ties), and such a query
takes about as long as any other of the matrix.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def one_entry_rows(acc, val):
    rows = len(val)
    idx = (np.arange(rows) % 8).astype(np.int32)
    return acc.CSRMatrix.from_arrays(rows, 8, np.arange(rows + 1, dtype=np.int64), idx, val)


def check(acc, val, ks):
    g = acc.GpuMatrix(one_entry_rows(acc, val))
    order = np.lexsort((np.arange(len(val)), -val))[:max(ks)]
    for k in ks:
        got = g.topk_fp32_host(np.ones(8, np.float32), k)
        np.testing.assert_array_equal(got["index"], order[:k])
        np.testing.assert_array_equal(got["value"], val[order[:k]])


# rows of one entry: 512 per workgroup's step; workgroup counts that the launch may take
@pytest.mark.parametrize("groups", [1024, 1280, 2048])
@pytest.mark.parametrize("kind", ["rising", "falling", "levels", "copies"])
def test_best_rows_in_few_groups(acc, gpu, groups, kind):
    rows = groups * 512 * 4 + 77
    rng = np.random.default_rng(groups)
    val = rng.random(rows).astype(np.float32)
    high = np.nonzero(np.arange(rows) // 512 % groups < 20)[0]
    rise = (10 + np.arange(len(high)) / len(high)).astype(np.float32)
    val[high] = {"rising": rise, "falling": rise[::-1], "levels": rng.integers(10, 14, len(high)),
                 "copies": np.float32(10)}[kind]
    check(acc, val, (1, 20, 100, 500, 960))


# every row of one score but a few: the rows to take are the first of that score
@pytest.mark.parametrize("rows", [300, 5000, 100003, 2000003])
@pytest.mark.parametrize("above", [0, 1, 99, 2000])
def test_equal_scores(acc, gpu, rows, above):
    rng = np.random.default_rng(rows + above)
    val = np.zeros(rows, np.float32)
    val[rng.integers(0, rows, above)] = 1 + rng.integers(0, 9, above)
    val[rng.integers(0, rows, rows // 3)] = -1
    check(acc, val, (1, 100, 256))
    if rows > 960:
        check(acc, val, (257, 960))


def call_us(acc, g, x, k):
    xd, out = acc.DeviceBuffer.from_numpy(x), acc.DeviceBuffer((k, 2), np.int32)
    best = np.inf
    for _ in range(4):  # the first run warms up
        a, b = acc.Event(), acc.Event()
        a.record()
        for _ in range(20):
            g.topk_fp32(xd, k, out)
        b.record()
        best = min(best, a.elapsed_ms(b) * 50)
    return best


@pytest.mark.parametrize("k", [100, 700])
def test_time_of_equal_scores(acc, gpu, k):
    csr = acc.CSRMatrix.generate(2000000, 500, deg=(20, 40), val_kind=acc.VAL_NORMAL, seed=4)
    g = acc.GpuMatrix(csr)
    usual = call_us(acc, g, acc.generate_queries(1, 500, seed=1)[0], k)
    equal = call_us(acc, g, np.zeros(500, np.float32), k)
    assert equal < 1.6 * usual, (equal, usual)  # a selection that reads all rows several times: 4 to 5 times
