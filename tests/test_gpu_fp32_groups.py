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
