"""A matrix is admitted to a server whose budget it just fits, and not to one
a byte smaller: what is reserved before the upload never exceeds what the
upload and the workspaces take.
"""
import pytest

pytestmark = pytest.mark.gpu


# with and without image packets, repeated columns, short rows, one slot and several
@pytest.mark.parametrize("rows,cols,deg,split", [(20000, 1500, (100, 200), 32), (20000, 500, (40, 100), 16), (700, 2048, (1, 900), 1),
                                                 (50, 30, (1, 3), 8), (200000, 700, (0, 4), 64)])
@pytest.mark.parametrize("slots,max_batch", [(1, 1), (2, 16)])
def test_exact_budget(acc, gpu, rows, cols, deg, split, slots, max_batch):
    csr = acc.CSRMatrix.generate(rows, cols, deg=deg, seed=rows)
    pk = csr.pack(bits=8, split=split)
    ck = split * 4
    probe = acc.Server(max_batch=max_batch, slots=slots, ck=ck)
    probe.add_matrix(csr, pk)
    need = probe.stats()["device_bytes"]
    probe.close()
    srv = acc.Server(memory_budget=need, max_batch=max_batch, slots=slots, ck=ck)
    srv.add_matrix(csr, pk)
    assert srv.stats()["device_bytes"] == need
    srv.close()
    srv = acc.Server(memory_budget=need - 1, max_batch=max_batch, slots=slots, ck=ck)
    with pytest.raises(acc.AccelesError, match="budget"):
        srv.add_matrix(csr, pk)
    srv.close()
