"""Set-up calls from several threads at once: the device scratch kept between
calls serves one of them at a time, the others take memory of their own; and
host arrays around the sizes where uploads go from direct copies to the
pinned buffers (64 MiB, pieces of 16 MiB)."""
import threading

import numpy as np
import pytest

import mlem_amd as M
from matrices import make

pytestmark = pytest.mark.gpu


def test_concurrent_set_up():
    kinds = ["ragged", "heavy", "row_gaps", "dups"]
    mats = [make(k, seed=3) for k in kinds]
    ATs = [M.transpose(A) for A in mats]
    errors = []

    def work(i):
        try:
            A, AT = mats[i], ATs[i]
            g, f0 = np.full(A.rows, 3, np.int32), np.ones(A.cols, np.float32)
            imgs = []
            for _ in range(6):
                with M.ResidentMatrix(A) as m:
                    m.build_transpose()
                    T = m.download_transpose()
                    assert np.array_equal(T.rowptr, AT.rowptr) and np.array_equal(T.col, AT.col)
                    assert np.array_equal(T.val.view(np.uint32), AT.val.view(np.uint32))
                    imgs.append(M.mlem_run(m, g, f0, 3, options=M.opts(tile_width=1024)))
            assert all(np.array_equal(x.view(np.uint32), imgs[0].view(np.uint32)) for x in imgs)
        except Exception as e:  # noqa: BLE001 (reported below, in the test's own thread)
            errors.append((kinds[i], repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(mats))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors


@pytest.mark.parametrize("mib", [63, 64, 65, 80, 81])
def test_uploads_around_the_piece_sizes(mib):
    """col and val of mib MiB, plus one entry."""
    nnz = mib * (1 << 18) + 1
    rows = 1000
    rowptr = np.linspace(0, nnz, rows + 1).astype(np.uint64)
    col = (np.arange(nnz, dtype=np.uint64) * 2654435761 % 4999).astype(np.uint32)
    val = np.arange(nnz, dtype=np.uint32).view(np.float32)
    A = M.Csr(rows, 5000, rowptr, col, val)
    with M.ResidentMatrix(A) as m:
        B = m.download()
    assert np.array_equal(B.rowptr, rowptr) and np.array_equal(B.col, col)
    assert np.array_equal(B.val.view(np.uint32), val.view(np.uint32))
