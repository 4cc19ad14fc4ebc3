"""Device memory of the single-query state: 16 bytes per slice up to 65,536
slices, where each slice's three largest scores are kept, 4 above; results on
both sides against the packet batch.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,split,slices,each", [
    (4194304, 1, 65536, 16), (4194305, 1, 65537, 4), (4192320, 32, 65536, 16), (4194305, 32, 65537, 4),
    (4172800, 400, 65200, 16), (4198400, 400, 65600, 4)])
def test_slice_state(acc, gpu, rows, split, slices, each):
    csr = acc.CSRMatrix.generate(rows, 40, deg=(1, 3), seed=split)
    pk = csr.pack(bits=8, split=split)
    assert pk.info.nslices == slices
    packets = acc.GpuMatrix(None, pk)
    # packets and slot map, image packets, row counts, 64 candidates per partition
    known = pk.info.stream_bytes + pk.info.perm_bytes + packets.info.dense_bytes + slices + split * 64 * 16
    assert 0 <= packets.info.device_bytes - known - each * slices < 400000
    del packets
    g = acc.GpuMatrix(csr, pk)
    x, ck = acc.generate_queries(1, 40, seed=slices), split * max(1, 64 // split)
    xd, k = acc.DeviceBuffer.from_numpy(x), min(ck, 100)
    one, batch = (acc.DeviceBuffer.from_numpy(np.full((1, k, 2), 9, np.int32)) for _ in range(2))
    g.topk_lowbit(xd, k, ck, one)
    g.set_batch_mode(acc.BATCH_SPARSE)
    g.topk_lowbit_batch(xd, np.full(1, k, np.int32), ck, batch, k)
    acc.synchronize()
    np.testing.assert_array_equal(one.numpy(), batch.numpy())
