"""Matrix-core scores of one and two query tiles, whose two row tiles go to two
wavefronts that merge their lists a round later: every count of column blocks
held, workgroups of one, two and more slices (the merge's first, second and
steady rounds; even and odd last slices), batches at the edges of a tile, the
best rows in one row tile.  Compared with the packet layout exactly.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [200, 500, 700, 900, 1024])
@pytest.mark.parametrize("rows", [40, 5000, 33000, 70000, 101000])
def test_row_tiles(acc, gpu, cols, rows):
    csr = acc.CSRMatrix.generate(rows, cols, deg=(2, 9), seed=rows + cols)
    ptr, idx, val = csr.arrays()
    val = np.array(val)
    low = np.repeat(np.arange(rows) % 3 == 0, np.diff(ptr))  # score levels: lists with ties across row tiles
    val[low] = 0.5
    csr = acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)
    split = 2 if rows < 1000 else 16
    g = acc.GpuMatrix(csr, csr.pack(bits=8, split=split))
    X = acc.generate_queries(65, cols, seed=cols)
    for nq in (1, 31, 32, 33, 64, 65):
        k = 16 if rows < 1000 else 60
        got = []
        for mode in (acc.BATCH_DENSE, acc.BATCH_SPARSE):
            g.set_batch_mode(mode)
            out = acc.DeviceBuffer((nq, k, 2), np.int32)
            g.topk_lowbit_batch(acc.DeviceBuffer.from_numpy(X[:nq]), np.full(nq, k, np.int32), split * 8, out, k)
            acc.synchronize()
            got.append(out.numpy())
        np.testing.assert_array_equal(got[0], got[1])
