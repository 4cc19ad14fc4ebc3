"""The FP32 Top-K from each workgroup's three best rows at the edges of its
rule (K up to the count of workgroups to the power 2/3): odd and even counts of
groups, K on both sides, the best rows side by side in one workgroup, in one
wavefront of each, and alone.  Results are compared with the oracle exactly.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


# rows of 50 .. 90 entries: eight per step, 32 per workgroup: 1, 31, 32 and 626 workgroups, and two steps per wavefront
@pytest.mark.parametrize("rows,ks", [(29, (1, 2)), (977, (1, 9, 10)), (1019, (10, 11)), (20011, (1, 73, 74)), (90001, (64, 100))])
@pytest.mark.parametrize("best", ["anywhere", "neighbours", "every_32nd"])
def test_workgroup_groups(acc, gpu, rows, ks, best):
    rng = np.random.default_rng(rows)
    lens = rng.integers(50, 91, rows)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([np.sort(rng.permutation(300)[:n]) for n in lens]).astype(np.int32)
    val = np.abs(rng.standard_normal(len(idx))).astype(np.float32)
    x = np.abs(rng.standard_normal(300)).astype(np.float32)
    high = {"anywhere": [], "neighbours": range(rows // 2, min(rows // 2 + 90, rows)), "every_32nd": range(5, rows, 32)}[best]
    for r in high:
        val[ptr[r]:ptr[r + 1]] *= 8
    csr = acc.CSRMatrix.from_arrays(rows, 300, ptr, idx, val)
    g = acc.GpuMatrix(csr)
    y = O.spmv_f32(ptr, idx, val, x, g.info.group)
    for k in ks:
        got = g.topk_fp32_host(x, k)
        r, v = O.topk(y, k)
        np.testing.assert_array_equal(got["index"], r)
        np.testing.assert_array_equal(got["value"], np.asarray(v, np.float32))


# steps of three or four blocks that become one less: rows of 20, 35 and 60 entries on average, a few of many
@pytest.mark.parametrize("mean,long", [(20, 0), (20, 100), (35, 0), (35, 300), (60, 0), (60, 280)])
def test_step_blocks_by_spread(acc, gpu, mean, long):
    rng = np.random.default_rng(mean + long)
    lens = rng.integers(mean - 3, mean + 4, 6007)
    lens = np.where(rng.random(6007) < 0.1, long, lens) if long else lens
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    idx = np.concatenate([np.sort(rng.permutation(310)[:n]) for n in lens]).astype(np.int32)
    val = rng.standard_normal(len(idx)).astype(np.float32)
    x = rng.standard_normal(310).astype(np.float32)
    x[0] = np.inf  # read by slots past a row's end: no row has column 0, so none may sum it
    keep = idx != 0
    ptr = np.concatenate([[0], np.cumsum(np.add.reduceat(keep, ptr[:-1]))]).astype(np.int64)
    idx, val = idx[keep], val[keep]
    csr = acc.CSRMatrix.from_arrays(6007, 310, ptr, idx, val)
    g = acc.GpuMatrix(csr)
    y = acc.DeviceBuffer.from_numpy(np.full(6007, 7, np.float32))
    g.spmv_fp32(acc.DeviceBuffer.from_numpy(x), y)
    acc.synchronize()
    np.testing.assert_array_equal(y.numpy(), O.spmv_f32(ptr, idx, val, x, g.info.group))


# the best rows in one workgroup's group of several thousand rows, which all wavefronts read together
@pytest.mark.parametrize("rows,first,count,k", [(2000003, 1000, 300, 100), (2000003, 1999900, 103, 100), (3000001, 77, 5000, 90)])
def test_long_groups(acc, gpu, rows, first, count, k):
    rng = np.random.default_rng(rows + first)
    ptr = np.arange(rows + 1, dtype=np.int64)
    idx = rng.integers(0, 8, rows).astype(np.int32)
    val = rng.random(rows).astype(np.float32)
    val[first:first + count] += 10
    x = np.ones(8, np.float32)
    got = acc.GpuMatrix(acc.CSRMatrix.from_arrays(rows, 8, ptr, idx, val)).topk_fp32_host(x, k)
    order = np.lexsort((np.arange(rows), -val))[:k]
    np.testing.assert_array_equal(got["index"], order)
    np.testing.assert_array_equal(got["value"], val[order])
