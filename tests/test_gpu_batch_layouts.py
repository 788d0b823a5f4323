"""The shapes that batches take by themselves, by the layout the matrix leads to: row slices have rows per block and
runs of their own, and a matrix that they do not suit keeps those of the block streams."""
import numpy as np
import pytest

import mlem_amd as M
import oracle as O

pytestmark = pytest.mark.gpu

def rel_l2(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def matrix(rows, cols, per_row, dense, seed=5):
    """Rows of about per_row spread columns; a dense block of `dense` rows and columns at the origin, whose rows and
    columns have more entries in a tile than a row slice holds (1020)."""
    rng = np.random.default_rng(seed)
    parts = []
    for r in range(rows):
        c = np.unique(rng.integers(dense if r < dense else 0, cols, per_row))
        parts.append(np.concatenate([np.arange(dense), c]) if r < dense else c)
    rowptr = np.concatenate([[0], np.cumsum([p.size for p in parts])]).astype(np.uint64)
    col = np.concatenate(parts).astype(np.uint32)
    return M.Csr(rows, cols, rowptr, col, (rng.random(col.size) + 0.05).astype(np.float32))


@pytest.fixture(scope="module")
def mats():
    return {dense: matrix(4000, 20000, 300, dense) for dense in (0, 1100)}


def reconstruct(m, A, values, **kw):
    g = np.random.default_rng(2).integers(0, 50, A.rows).astype(np.int32)
    f0 = np.ones(A.cols, np.float32)
    with M.Batch(m, 5, values=values, per_pass=kw.pop("per_pass", 4), **kw) as b:
        b.set(0, 0 * g + 1, f0)
        b.set(4, g, f0)
        b.iterate(5)
        img = b.image(4)
        layouts = [b.layout(s) for s in (0, 1)]
    val = O.quantize_values(A.rowptr, A.val, A.rows, values).astype(np.float32) if values else A.val
    sens = O.colsum_f64(A.rowptr, A.col, val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    ref = O.mlem_f64(A.rowptr, A.col, val, A.rows, A.cols, g, sens, f0, 5)
    assert rel_l2(img, ref) <= (2e-6 if values else 1e-5)
    return layouts


@pytest.mark.parametrize("values", [0, 3])
def test_block_streams_keep_their_shape(mats, values):
    A = mats[1100]
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        for _ in range(2):  # found unsuited, then remembered
            for side in reconstruct(m, A, values):
                assert side["kind"] == "block streams" and side["tile_width"] == 1024
                # 2.4e6 nonzeros: under two units of 2048 for each of 8 runs per CU
                assert side["tile_rows"] == 512
        for side in reconstruct(m, A, values, tile_rows=1024):  # a shape asked for is the shape taken
            assert side["kind"] == "block streams" and side["tile_rows"] == 1024
    with M.ResidentMatrix.tiles_only(A, values=values, per_pass=4) as m:
        for side in reconstruct(m, A, values):
            assert side["kind"] == "block streams" and side["tile_rows"] == 512


@pytest.mark.parametrize("values", [0, 3])
def test_row_slices_keep_theirs(mats, values):
    A = mats[0]
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        for side in reconstruct(m, A, values):
            assert side["kind"] == "row slices" and side["tile_rows"] == 1024 and side["max_steps"] > 0
