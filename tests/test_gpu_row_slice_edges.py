"""Row slices at the edges of their layout, each case checked to be kept as row slices (matrices whose few long rows
would be padded go to the block streams instead): rows of 1020 entries in a tile (255 steps, the most a row may
have), tiles of 1, 15, 16, 17 and 129 rows beside full ones, tiles without entries, and row blocks that are one run
over 16 column segments with entries in each, the most such a run takes (17: runs with partial sums).

Bars: those of the other row-slice tests, FP64 MLEM within 1e-5 rel-L2 with f32 values and 2e-6 with 16-bit values on
the values that the tiles hold."""
import numpy as np
import pytest

import mlem_amd as M
import oracle as O

pytestmark = pytest.mark.gpu


def csr(rows, cols, seed=7):
    """rows: one array of columns per row."""
    rng = np.random.default_rng(seed)
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint64)
    col = np.concatenate(rows).astype(np.uint32)
    return M.Csr(len(rows), cols, rowptr, col, (rng.random(col.size) + 0.05).astype(np.float32))


def long_rows():
    """64 rows of 1020 and 1016 entries in the tile of columns 0 ... 1023 (4 slices of 255 and 254 steps), 400 of 60
    in the next; their columns hold 64 entries each."""
    rows = [np.arange(1020)] * 32 + [np.arange(4, 1020)] * 32
    rows += [1024 + 16 * np.arange(60) + i % 16 for i in range(400)]
    return csr(rows, 2048)


def ragged_tiles():
    """1024 full rows over two segments; segments of 1, 15, 16, 17 and 129 rows with entries, one with none, one of
    rows of 1 ... 37 entries."""
    rng = np.random.default_rng(5)
    rows = [[np.sort(rng.choice(1024, 48, replace=False)) + 1024 * s for s in (0, 1)] for _ in range(1024)]
    for s, n in ((2, 1), (3, 15), (4, 16), (5, 17), (6, 129)):
        for i in rng.choice(1024, n, replace=False):
            rows[i].append(1024 * s + 8 * np.arange(1 + i % 5))
    for i in range(300):
        rows[i].append(1024 * 8 + 20 * np.arange(1 + i // 8))
    return csr([np.concatenate(r) for r in rows], 9 * 1024 + 5)


def check(m, A, values, per_pass, **kw):
    rng = np.random.default_rng(2)
    sinos = [rng.integers(0, 50, A.rows).astype(np.int32) for _ in range(2)]
    f0 = np.ones(A.cols, np.float32)
    val = O.quantize_values(A.rowptr, A.val, A.rows, values).astype(np.float32) if values else A.val
    sens = O.colsum_f64(A.rowptr, A.col, val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    slots = 2 * per_pass + 1
    with M.Batch(m, slots, values=values, per_pass=per_pass, **kw) as b:
        for k in range(slots):
            b.set(k, sinos[k % 2], f0)
        b.iterate(5)
        images, layouts = [b.image(k) for k in range(slots)], [b.layout(s) for s in (0, 1)]
    for k, img in enumerate(images):
        if k < 2:
            ref = O.mlem_f64(A.rowptr, A.col, val, A.rows, A.cols, sinos[k], sens, f0, 5)
            assert np.linalg.norm(img - ref) <= (2e-6 if values else 1e-5) * np.linalg.norm(ref)
        else:
            assert np.array_equal(img, images[k % 2])
    print(layouts, flush=True)
    return layouts


@pytest.mark.parametrize("values", [0, 1, 2, 3])
@pytest.mark.parametrize("rows,groups", [(2048, 0), (1024, 2), (512, 4096)])
def test_rows_of_255_steps(values, rows, groups):
    A = long_rows()
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        a, t = check(m, A, values, 4, tile_width=1024, tile_rows=rows, tile_groups=groups)
    assert a["kind"].startswith("row slices") and a["max_steps"] >= 255
    assert t["kind"].startswith("row slices") and t["max_steps"] >= 16


@pytest.mark.parametrize("values,per_pass,width,rows,groups", [(0, 4, 1024, 2048, 0), (3, 4, 1024, 512, 1),
                                                               (2, 4, 512, 1024, 3), (0, 8, 512, 512, 1),
                                                               (1, 8, 512, 1024, 0), (3, 8, 512, 1024, 4096)])
def test_ragged_tiles(values, per_pass, width, rows, groups):
    A = ragged_tiles()
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        a, t = check(m, A, values, per_pass, tile_width=width, tile_rows=rows, tile_groups=groups)
    assert a["kind"].startswith("row slices") and t["kind"].startswith("row slices")


@pytest.mark.parametrize("values,per_pass", [(0, 4), (3, 4), (1, 8)])
@pytest.mark.parametrize("segs", [16, 17])
def test_one_run_over_16_segments(segs, values, per_pass):
    """2 entries a row in every segment (8 per pass: 1), a last row block of 476 or 500 rows."""
    w, n = (512, 1) if per_pass == 8 else (1024, 2)
    rng = np.random.default_rng(segs)
    rows = [np.concatenate([np.sort(rng.choice(w, n, replace=False)) + w * s for s in range(segs)])
            for _ in range(1500 if per_pass == 4 else 500)]
    A = csr(rows, segs * w)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        a, _ = check(m, A, values, per_pass)
    assert a["kind"] == ("row slices, one run per row block" if segs == 16 else "row slices")
    assert a["tile_rows"] == 512 if segs == 16 else a["runs"] >= 1
