"""ACC_BATCH_AUTO on an untuned handle: whatever layout it picks for a batch
size, the results are those of the packet and matrix-core layouts, and a
crossover set by the caller holds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(acc, g, X, ks, ck):
    out = acc.DeviceBuffer.from_numpy(np.full((len(ks), 64, 2), 9, np.int32))
    g.topk_lowbit_batch(acc.DeviceBuffer.from_numpy(X[:len(ks)]), ks, ck, out, 64)
    acc.synchronize()
    return out.numpy()


@pytest.mark.parametrize("rows,cols,deg,bits,signed", [(3000, 120, (5, 20), 8, False), (60000, 500, (20, 60), 4, False),
                                                       (20000, 1500, (20, 60), 8, False), (300000, 900, (5, 15), 6, True)])
def test_auto_matches_fixed_layouts(acc, gpu, rows, cols, deg, bits, signed):
    csr = acc.CSRMatrix.generate(rows, cols, deg=deg, val_kind=acc.VAL_NORMAL if signed else acc.VAL_ABSNORMAL, seed=rows)
    g = acc.GpuMatrix(csr, csr.pack(bits=bits, split=16, is_signed=signed))
    X = acc.generate_queries(40, cols, seed=3)
    modes = [acc.BATCH_SPARSE] + ([acc.BATCH_DENSE] if g.info.dense_ok else [])
    for nq in (1, 2, 3, 7, 16, 17, 40):
        ks = (np.arange(nq, dtype=np.int32) * 7) % 64 + 1
        g.set_batch_mode(acc.BATCH_AUTO)
        auto = run(acc, g, X, ks, 128)
        for mode in modes:
            g.set_batch_mode(mode)
            np.testing.assert_array_equal(auto, run(acc, g, X, ks, 128))
    g.set_batch_mode(acc.BATCH_AUTO, 5)  # a crossover
    np.testing.assert_array_equal(run(acc, g, X, ks, 128), auto)
    np.testing.assert_array_equal(run(acc, g, X, ks[:4], 128), auto[:4])
