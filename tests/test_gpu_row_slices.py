"""Batches over row slices (16 rows of a tile share their steps, a row takes
four entries a step) at their edges: rows of 1 ... 1020 entries in a tile
(255 steps, the most a slice holds; 1024 takes the other layout), 1, 15, 16,
17 and 129 rows in a tile, row blocks that end in the last slice, tiles
without entries, and runs that would cover more than 64 tiles.

Bars: a row's f32 sum of n <= 1020 positive products, in four interleaved
parts, is off by about eps * sqrt(n / 12) = 5e-7 at most (rms), so FP64 MLEM
on the values the tiles hold within 1e-5 rel-L2 with f32 values and 2e-6 with
16-bit values, as for every other matrix."""
import numpy as np
import pytest

import mlem_amd as M
import oracle as O

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def csr(lens, starts, cols, stride=1, seed=7):
    """Row i: lens[i] columns from starts[i] on, `stride` apart."""
    rng = np.random.default_rng(seed)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    col = np.concatenate([c + stride * np.arange(n) for c, n in zip(starts, lens)]).astype(np.uint32)
    return M.Csr(len(lens), cols, rowptr, col, (rng.random(col.size) + 0.05).astype(np.float32))


def shapes():
    rng = np.random.default_rng(3)
    for n in (1, 15, 16, 17, 129):  # rows in the one tile that has any
        lens = [1 + (5 * i) % 37 for i in range(n)]
        yield f"rows{n}", csr(lens, rng.integers(0, 900, n), 2500)
    yield "long", csr([1020, 1016, 5, 4, 3, 1020, 1] * 9, [1024, 0, 3, 2047, 0, 4, 2900] * 9, 4096)
    yield "too_long", csr([1024, 7, 1024, 2] * 9, [1024, 0, 0, 9] * 9, 2048)
    for n in (511, 513, 2047, 2049):  # row blocks' ends; every third row empty
        lens = np.where(np.arange(n) % 3 == 1, 0, rng.integers(1, 12, n))
        yield f"block{n}", csr(lens, rng.integers(0, 1800, n), 2000)
    # 130 column segments of 1024 for one row block, two entries of a row in each
    yield "wide", csr([260] * 300, rng.integers(0, 500, 300), 130 * 1024 + 77, stride=512)


SHAPES = dict(shapes())


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("values,per_pass,width,rows,groups", [(0, 4, 1024, 2048, 0), (3, 4, 1024, 512, 1),
                                                               (2, 4, 512, 1024, 3), (0, 8, 512, 512, 1),
                                                               (1, 8, 512, 1024, 0), (3, 8, 512, 2048, 0)])
def test_edges_of_slices_and_runs(name, values, per_pass, width, rows, groups):
    A = SHAPES[name]
    rng = np.random.default_rng(2)
    sinos = [rng.integers(0, 50, A.rows).astype(np.int32) for _ in range(2)]
    f0 = np.ones(A.cols, np.float32)
    val = O.quantize_values(A.rowptr, A.val, A.rows, values).astype(np.float32) if values else A.val
    sens = O.colsum_f64(A.rowptr, A.col, val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    slots = per_pass + 1  # two passes
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        with M.Batch(m, slots, values=values, per_pass=per_pass, tile_width=width, tile_rows=rows,
                     tile_groups=groups) as b:
            for k in range(slots):
                b.set(k, sinos[k % 2], f0)
            b.iterate(5)
            images = [b.image(k) for k in range(slots)]
    for k, img in enumerate(images):
        if k < 2:
            ref = O.mlem_f64(A.rowptr, A.col, val, A.rows, A.cols, sinos[k], sens, f0, 5)
            assert rel_l2(img, ref) <= (2e-6 if values else 1e-5)
        else:
            assert np.array_equal(img, images[k % 2])  # the slot does not matter


@pytest.mark.parametrize("per_pass,values", [(4, 0), (4, 3), (8, 1)])
@pytest.mark.parametrize("rows,cols,gap", [(1, 40, 0), (511, 1025, 0), (512, 16 * 512, 0), (513, 16 * 512 + 1, 0),
                                           (1537, 16 * 1024, 0), (1537, 16 * 1024 + 1, 0), (2000, 300, 600)])
def test_row_blocks_as_one_run(rows, cols, gap, per_pass, values):
    """Default tiles of small matrices, whose row blocks are one run each (no partial sums): a last block of one
    row or one short of a block, as many column segments as such a run takes and one more, and a block without any
    entries (rows 512 .. 512 + gap empty), whose run has no tiles."""
    rng = np.random.default_rng(rows + cols)
    lens = rng.integers(0, 1 + min(cols, 24), rows)
    lens[0] = 3
    if gap:
        lens[512:512 + gap] = 0
    A = csr(lens, rng.integers(0, max(1, cols // 2), rows), cols, stride=1)
    g = rng.integers(0, 50, A.rows).astype(np.int32)
    f0 = np.ones(A.cols, np.float32)
    val = O.quantize_values(A.rowptr, A.val, A.rows, values).astype(np.float32) if values else A.val
    sens = O.colsum_f64(A.rowptr, A.col, val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    ref = O.mlem_f64(A.rowptr, A.col, val, A.rows, A.cols, g, sens, f0, 5)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        with M.Batch(m, 3 * per_pass, values=values, per_pass=per_pass, use_graph=1) as b:
            for k in range(3 * per_pass):
                b.set(k, g, f0)
            for n in (2, 1, 2):
                b.iterate(n)
                b.sync()
            for k in (0, per_pass - 1, 2 * per_pass, 3 * per_pass - 1):
                assert rel_l2(b.image(k), ref) <= (2e-6 if values else 1e-5)
