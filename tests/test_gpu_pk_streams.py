"""Image packets at the edges of their streams: decode wavefronts with no
entries, one group of four per lane, exactly and one past the eight groups
loaded ahead and the second chunk, the most groups a stream can hold (rows
without an absent column), offsets up to 16 rows of 1024 columns; and the
whole range of the image's bytes.  The batched scores' results are compared
with the packet layout's, which reads other packets, and exactly.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (columns, entries of a row): 16 rows of n entries are n / 16 groups of 256
@pytest.mark.parametrize("cols,nnz", [(3, 1), (3, 3), (40, 16), (40, 17), (200, 128), (200, 129), (600, 256), (600, 257),
                                      (512, 512), (1024, 1), (1024, 385), (1024, 1024)])
@pytest.mark.parametrize("bits,signed", [(8, False), (8, True), (4, False), (5, True)])
def test_streams(acc, gpu, cols, nnz, bits, signed):
    rng = np.random.default_rng(cols + nnz)
    rows = 64 * 7 + 9
    # some rows empty, a whole wavefront's rows among them: the packer sorts by length
    lens = np.where(np.arange(rows) % 5 == 0, 0, nnz)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    idx = np.concatenate([np.sort(rng.permutation(cols)[:n]) for n in lens]) if ptr[-1] else np.empty(0)
    val = rng.uniform(-1 if signed else 0, 1, int(ptr[-1])).astype(np.float32)
    csr = acc.CSRMatrix.from_arrays(rows, cols, ptr, idx, val)
    g = acc.GpuMatrix(csr, csr.pack(bits=bits, split=2, is_signed=signed))
    X = acc.generate_queries(9, cols, seed=nnz)
    got = []
    for mode in (acc.BATCH_DENSE, acc.BATCH_SPARSE):
        g.set_batch_mode(mode)
        out = acc.DeviceBuffer((9, 30, 2), np.int32)
        g.topk_lowbit_batch(acc.DeviceBuffer.from_numpy(X), np.full(9, 30, np.int32), 40, out, 30)
        acc.synchronize()
        got.append(out.numpy())
    np.testing.assert_array_equal(got[0], got[1])
