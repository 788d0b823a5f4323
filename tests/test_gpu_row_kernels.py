"""The CSR-vector kernel for long rows (a mean of 384 entries per row or
more) and the scatter through column windows in LDS, at the sizes where they
turn: rows of 0, 1, 63, 64, 65 entries and around a chunk of 1024, rows that
start off a multiple of four, windows of 32,768 columns with entries on both
sides of their edges, one row up to several per wave, unsorted rows and
repeated columns.

Bars: a row of n FP32 products added in any order differs from the FP64 sum
by at most (n + 1) 2^-24 sum |v x| (the products' rounding included); the
scatter adds its sums once more per workgroup and window, so its column sums
get n + 64 terms."""
import numpy as np
import pytest

import mlem_amd as M

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def matrix(lens, cols, seed, kind):
    rng = np.random.default_rng(seed)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    col = rng.integers(0, cols, int(rowptr[-1])).astype(np.uint32)
    if kind != "unsorted":
        for r in range(len(lens)):
            b, e = int(rowptr[r]), int(rowptr[r + 1])
            if kind == "edges" and e - b <= cols:  # consecutive columns around a window's edge
                start = max(0, min(cols - (e - b), 32768 - (e - b) // 2 - r % 7))
                col[b:e] = np.arange(start, start + e - b, dtype=np.uint32)
            else:
                col[b:e].sort()
    return M.Csr(len(lens), cols, rowptr, col, (rng.random(col.size) + 0.01).astype(np.float32))


LENS = {
    "around_chunks": [1024, 1023, 1025, 1, 2048, 2047, 2049, 63, 64, 65, 0, 4096, 255, 256, 257, 3000],
    "short_tail": [900] * 41 + [0] * 3,
    "one_row": [70001],
    "many": list(range(0, 800)) * 2 + [384] * 500,
}


def exact(A, x):
    """A x and the sums of |a x| per row in FP64."""
    m = A.to_scipy().astype(np.float64)
    return m @ x.astype(np.float64), abs(m) @ np.abs(x.astype(np.float64))


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("cols,kind", [(50000, "sorted"), (70000, "edges"), (33000, "unsorted"), (40, "sorted")])
def test_long_rows(lens, cols, kind):
    A = matrix(LENS[lens], cols, 1, kind)
    x = np.random.default_rng(2).random(cols).astype(np.float32)
    y, mag = exact(A, x)
    g = np.arange(1, A.rows + 1, dtype=np.int32)
    n = np.diff(A.rowptr.astype(np.int64))
    bar = (n + 1) * EPS * mag
    with M.ResidentMatrix(A) as m:
        rp, ci, va = m.device_arrays()[:3]
        dx, dg, out = M.DeviceArray.from_numpy(x), M.DeviceArray.from_numpy(g), M.DeviceArray(A.rows, np.float32)
        M.fp_csr_vector(rp, ci, va, dx, out, A.rows, A.nnz)
        got = out.numpy()
        assert np.all(np.abs(got - y) <= bar)
        M.fp_csr_vector(rp, ci, va, dx, out, A.rows, A.nnz)
        assert np.array_equal(out.numpy().view(np.uint32), got.view(np.uint32))
        M.fp_ratio_csr_vector(rp, ci, va, dx, dg, out, A.rows, A.nnz)
        assert np.array_equal(out.numpy(), np.divide(g.astype(np.float32), got, where=got != 0, out=got.copy()))
        norm = (np.arange(A.rows) % 3).astype(np.float32)
        f = np.random.default_rng(3).random(A.rows).astype(np.float32)
        df, dn = M.DeviceArray.from_numpy(f), M.DeviceArray.from_numpy(norm)
        M.bp_update_csr_vector(rp, ci, va, dx, dn, df, A.rows, A.nnz)
        v = f * got
        assert np.array_equal(df.numpy(), np.divide(v, norm, where=norm != 0, out=v.copy()))
    # infinities of x stay where their columns are
    x2 = x.copy()
    x2[0] = np.inf
    y2 = A.to_scipy().astype(np.float64) @ x2.astype(np.float64)
    with M.ResidentMatrix(A) as m:
        rp, ci, va = m.device_arrays()[:3]
        dx, out = M.DeviceArray.from_numpy(x2), M.DeviceArray(A.rows, np.float32)
        M.fp_csr_vector(rp, ci, va, dx, out, A.rows, A.nnz)
        assert np.array_equal(np.isfinite(out.numpy()), np.isfinite(y2))


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("cols,kind", [(50000, "sorted"), (70000, "edges"), (32768, "sorted"), (33000, "unsorted"),
                                       (40, "sorted")])
def test_scatter_windows(lens, cols, kind):
    lengths = LENS[lens]
    A = matrix(lengths, cols, 4, kind)
    rows_per_wg = -(-A.rows // 256)
    windows = 16 * A.nnz >= -(-A.rows // rows_per_wg) * cols  # else one atomic per entry
    r = np.random.default_rng(5).random(A.rows).astype(np.float32)
    r[::5] = 0.0
    m = A.to_scipy().astype(np.float64).T
    y, mag = m @ r.astype(np.float64), m @ r.astype(np.float64)
    n = np.bincount(A.col, minlength=cols)
    with M.ResidentMatrix(A) as mm:
        rp, ci, va = mm.device_arrays()[:3]
        dr, out = M.DeviceArray.from_numpy(r), M.DeviceArray.from_numpy(np.full(cols, 7.0, np.float32))
        for lanes in (0, 64):  # the automatic choice, one atomic per entry
            M.bp_scatter(rp, ci, va, dr, out, A.rows, cols, A.nnz, lanes)
            err = np.abs(out.numpy() - y)
            assert np.all(err <= (n + 64) * EPS * mag), (lanes, windows)


def test_scatter_windows_over_several_rounds_of_rows():
    """More rows than one workgroup per CU holds (262,144)."""
    lens = np.random.default_rng(6).integers(0, 12, 300001)
    A = matrix(list(lens), 1500, 7, "unsorted")
    r = np.random.default_rng(8).random(A.rows).astype(np.float32)
    y = A.to_scipy().astype(np.float64).T @ r.astype(np.float64)
    n = np.bincount(A.col, minlength=A.cols)
    with M.ResidentMatrix(A) as mm:
        rp, ci, va = mm.device_arrays()[:3]
        dr, out = M.DeviceArray.from_numpy(r), M.DeviceArray(A.cols, np.float32)
        M.bp_scatter(rp, ci, va, dr, out, A.rows, A.cols, A.nnz)
        assert np.all(np.abs(out.numpy() - y) <= (n + 64) * EPS * y)


@pytest.mark.parametrize("lens,edge", [([127, 128, 129, 255, 256, 257, 383, 384] * 200, 20224), ([40, 64, 65, 90] * 1500, 20224),
                                       ([20000, 4096, 1000] * 3, 20224), ([20000, 4096, 1000] * 3, 40448),
                                       ([3, 9, 24, 1] * 15000, 32768)])
def test_scatter_windows_of_each_kind(lens, edge):
    """Rows of consecutive columns across a window's edge, with few, some and many entries per row and window (FP32
    sums, FP64 sums 64 and 128 entries at a time), and rows that end with a piece."""
    cols = edge + max(lens)
    assert 16 * sum(lens) >= min(len(lens), 256) * cols  # windows
    rng = np.random.default_rng(11)
    start = [max(0, min(cols - n, edge - rng.integers(0, n + 1))) for n in lens]
    start[0], start[1] = 0, edge  # from the first column; from the edge on
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    col = np.concatenate([np.arange(s, s + n) for s, n in zip(start, lens)]).astype(np.uint32)
    A = M.Csr(len(lens), cols, rowptr, col, (rng.random(col.size) + 0.01).astype(np.float32))
    r = rng.random(A.rows).astype(np.float32) + 0.1
    y = A.to_scipy().astype(np.float64).T @ r.astype(np.float64)
    n = np.bincount(A.col, minlength=cols)
    with M.ResidentMatrix(A) as mm:
        rp, ci, va = mm.device_arrays()[:3]
        dr, out = M.DeviceArray.from_numpy(r), M.DeviceArray.from_numpy(np.full(cols, 7.0, np.float32))
        M.bp_scatter(rp, ci, va, dr, out, A.rows, cols, A.nnz)
        assert np.all(np.abs(out.numpy() - y) <= (n + 64) * EPS * y)
