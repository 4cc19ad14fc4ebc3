"""fp32_spmv at the edges of its staging: steps and rows that fill, just exceed
and far exceed the area, every lanes-per-row group, the last column of the
widest matrix.  The oracle restates the declared summation order, so scores
are compared bit by bit.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def csr_of(acc, lengths, cols, seed):
    rng = np.random.default_rng(seed)
    ptr = np.concatenate(([0], np.cumsum(lengths))).astype(np.int64)
    idx = np.concatenate([np.sort(rng.permutation(cols)[:n]) for n in lengths] or [[]]).astype(np.int32)
    val = rng.standard_normal(len(idx)).astype(np.float32)
    return acc.CSRMatrix.from_arrays(len(lengths), cols, ptr, idx, val), ptr, idx, val


LENGTHS = {
    "one_row": lambda r: [5],
    "short_rows": lambda r: r.integers(0, 7, 3001),                              # two lanes per row
    "eight_to_sixteen": lambda r: r.integers(6, 20, 2003),
    "twenty": lambda r: r.integers(10, 31, 1999),
    "fifty": lambda r: r.integers(30, 91, 1501),
    "seventy": lambda r: r.integers(50, 91, 1777),
    "full_steps": lambda r: np.full(97, 75),                                     # B * 2 * 75 entries per step
    "area_exactly": lambda r: np.full(33, 448),                                  # two rows fill the area
    "area_plus_one": lambda r: np.tile([448, 449], 20),                          # a block of two rows exceeds it
    "wide_rows": lambda r: r.integers(900, 3000, 41),                            # every row exceeds it
    "long_among_short": lambda r: np.where(r.random(4001) < 0.01, 700, r.integers(0, 30, 4001)),
    "longer_among_short": lambda r: np.where(r.random(2001) < 0.01, 2900, r.integers(5, 20, 2001)),
    "empty_tail": lambda r: np.concatenate((r.integers(10, 31, 200), np.zeros(77, int))),
    "all_empty": lambda r: np.zeros(130, int),
}


@pytest.mark.parametrize("cols", [3000, 8192])
@pytest.mark.parametrize("kind", LENGTHS)
def test_spmv_bitexact(acc, gpu, kind, cols):
    lengths = np.asarray(LENGTHS[kind](np.random.default_rng(7)))
    csr, ptr, idx, val = csr_of(acc, lengths, cols, seed=cols)
    g = acc.GpuMatrix(csr)
    x = acc.generate_queries(1, cols, seed=3)[0]
    y = acc.DeviceBuffer.from_numpy(np.full(len(lengths), 7, np.float32))
    g.spmv_fp32(acc.DeviceBuffer.from_numpy(x), y)
    acc.synchronize()
    np.testing.assert_array_equal(y.numpy(), O.spmv_f32(ptr, idx, val, x, g.info.group))


def topk_both(acc, csr, ptr, idx, val, x, k):
    g = acc.GpuMatrix(csr)
    got = g.topk_fp32_host(x, k)
    rows, vals = O.topk(O.spmv_f32(ptr, idx, val, x, g.info.group), k)
    m = min(k, csr.rows)
    np.testing.assert_array_equal(got["index"][:m], rows[:m])
    np.testing.assert_array_equal(got["value"][:m], np.asarray(vals[:m], np.float32))
    assert (got["index"][m:] == -1).all() and np.isneginf(got["value"][m:]).all()


# one row per step and group, groups of a few rows, of several steps; K below, at and above the ranking by counting
@pytest.mark.parametrize("rows,deg", [(977, (50, 90)), (20011, (50, 90)), (130001, (10, 30)), (700001, (1, 6))])
@pytest.mark.parametrize("k", [1, 100, 256, 257, 960])
def test_topk_from_groups(acc, gpu, rows, deg, k):
    csr = acc.CSRMatrix.generate(rows, 300, deg=deg, val_kind=acc.VAL_NORMAL, seed=rows + k)
    topk_both(acc, csr, *csr.arrays(), acc.generate_queries(1, 300, seed=k)[0], k)


# "zeros": every score ties; "same_group": the best rows lie in the same groups (more than the LDS list holds);
# "levels": a handful of score levels
@pytest.mark.parametrize("kind", ["zeros", "levels", "same_group", "infinite"])
@pytest.mark.parametrize("k", [3, 100, 700])
def test_topk_ties_and_clusters(acc, gpu, kind, k):
    rows, cols = 400000, 64
    rng = np.random.default_rng(k)
    ptr = np.arange(rows + 1, dtype=np.int64)
    idx = rng.integers(0, cols, rows).astype(np.int32)
    val = np.ones(rows, np.float32)
    x = np.ones(cols, np.float32)
    if kind == "zeros":
        x[:] = 0.0
    elif kind == "levels":
        val = rng.integers(-3, 3, rows).astype(np.float32)
    elif kind == "same_group":
        # steps of 128 rows (two lanes per row, four blocks): every 16th step scores high
        val = np.where(np.arange(rows) // 128 % 16 == 5, rng.random(rows) + 10, rng.random(rows)).astype(np.float32)
    else:
        val[rng.integers(0, rows, 50)] = np.inf
        val[rng.integers(0, rows, 50)] = -np.inf
    csr = acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)
    topk_both(acc, csr, ptr, idx, val, x, k)
