"""The device tile builder at the edges of its walk (a wave takes a row 64
entries at a time, the columns of four such steps loaded together): rows
that end just before, at and after those steps, runs of one column segment
that cross them, and a pair of swapped columns at each step's edge.

Bars: the FP64 oracle within 1e-5 rel-L2 with f32 values (the bar of every
FP32 path), FP64 MLEM on the oracle's quantized matrix within 2e-6 with
16-bit values (as for the other matrices)."""
import numpy as np
import pytest

import mlem_amd as M
import oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 511, 512, 513, 1000, 1025]


def rel_l2(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def matrix(first_cols, cols=4500, seed=5):
    """Rows of LENGTHS consecutive columns (runs of one segment as long as the row) from each of first_cols on."""
    rng = np.random.default_rng(seed)
    starts = [(c, n) for c in first_cols for n in LENGTHS]
    rowptr = np.concatenate([[0], np.cumsum([n for _, n in starts])]).astype(np.uint64)
    col = np.concatenate([np.arange(c, c + n, dtype=np.uint32) for c, n in starts])
    val = (rng.random(col.size) + 0.05).astype(np.float32)
    return M.Csr(len(starts), cols, rowptr, col, val)


@pytest.mark.parametrize("first_cols", [(0, 1000, 1023), (960, 961, 1024 - 65, 2048 - 64, 3000)])
@pytest.mark.parametrize("values,per_pass", [(0, 1), (0, 4), (3, 1), (2, 4), (1, 8)])
def test_rows_at_the_edges_of_the_walk(first_cols, values, per_pass):
    A = matrix(first_cols)
    g = np.random.default_rng(1).integers(0, 50, A.rows).astype(np.int32)
    f0 = np.ones(A.cols, np.float32)
    val = O.quantize_values(A.rowptr, A.val, A.rows, values).astype(np.float32) if values else A.val
    sens = O.colsum_f64(A.rowptr, A.col, val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    ref = O.mlem_f64(A.rowptr, A.col, val, A.rows, A.cols, g, sens, f0, 6)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        if per_pass == 1:
            img = M.mlem_run(m, g, f0, 6, options=M.opts(tile_width=1024, values=values))
        else:
            with M.Batch(m, 1, values=values, per_pass=per_pass) as b:
                b.set(0, g, f0)
                b.iterate(6)
                img = b.image(0)
    assert rel_l2(img, ref) <= (2e-6 if values else 1e-5)


@pytest.mark.parametrize("at", [0, 1, 62, 63, 64, 127, 254, 255, 256, 510])
def test_unsorted_row_is_refused(at):
    A = matrix((0, 1000))
    r = LENGTHS.index(513)  # swap two neighbours of the 513-entry row
    k = int(A.rowptr[r]) + at
    A.col[[k, k + 1]] = A.col[[k + 1, k]]
    g, f0 = np.ones(A.rows, np.int32), np.ones(A.cols, np.float32)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        with pytest.raises(M.MlemError):
            M.Recon(m, g, f0, options=M.opts(tile_width=1024))
        with M.Recon(m, g, f0) as r:  # automatic: the plain merge path
            r.iterate(1)
