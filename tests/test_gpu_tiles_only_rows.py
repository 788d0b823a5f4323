"""Tiles-only matrices whose default rows per block differ between the sides, or do not fit the scratch allowed:
the taller blocks of row slices give way to those of the block streams, as small as they were before the slices."""
import numpy as np
import pytest

import mlem_amd as M
from test_gpu_batch_layouts import matrix

pytestmark = pytest.mark.gpu


def images(m, A, values):
    rng = np.random.default_rng(3)
    sinos = [rng.integers(0, 40, A.rows).astype(np.int32) for _ in range(6)]
    f0 = np.ones(A.cols, np.float32)
    with M.Batch(m, 6, values=values, per_pass=4) as b:
        for k, g in enumerate(sinos):
            b.set(k, g, f0)
        b.iterate(5)
        return [b.layout(s) for s in (0, 1)], [b.image(k) for k in range(6)]


@pytest.mark.parametrize("values", [0, 3])
def test_scratch_for_512_rows_only(values):
    """64 MiB of scratch hold 512 rows of A^T of this matrix, not the 1024 of row slices."""
    A = matrix(4000, 20000, 300, 1100)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        _, ref = images(m, A, values)
    with M.ResidentMatrix.tiles_only(A, values=values, per_pass=4, chunk_bytes=64 << 20) as m:
        layouts, got = images(m, A, values)
    assert [s["tile_rows"] for s in layouts] == [512, 512]
    for a, b in zip(got, ref):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("values", [0, 3])
def test_sides_of_different_rows(c1, values):
    """The 2D ring: A's row blocks of 512 rows are one run each, A^T's blocks have 1024.  Images bitwise those of the
    resident batch.  512 stands for the automatic rows of a matrix of this size; other rows are refused, those of
    one side too."""
    A = c1["A"]
    with M.ResidentMatrix(A, c1["AT"]) as m:
        want, ref = images(m, A, values)
    with M.ResidentMatrix.tiles_only(A, values=values, per_pass=4) as m:
        layouts, got = images(m, A, values)
        with M.Batch(m, 4, values=values, per_pass=4, tile_rows=512) as b:
            assert [b.layout(s) for s in (0, 1)] == want
        for rows in (1024, 2048):
            with pytest.raises(M.MlemError) as e:
                M.Batch(m, 4, values=values, per_pass=4, tile_rows=rows)
            assert "512 (A) and 1024 (A^T) rows" in str(e.value)
    assert layouts == want and [s["tile_rows"] for s in layouts] == [512, 1024]
    assert layouts[0]["kind"] == "row slices, one run per row block"
    for a, b in zip(got, ref):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    with M.ResidentMatrix.tiles_only(A, values=values, per_pass=4, tile_rows=2048) as m:
        for rows in (512, 1024):
            with pytest.raises(M.MlemError):
                M.Batch(m, 4, values=values, per_pass=4, tile_rows=rows)


def test_reconstructions_by_the_name_of_the_automatic_rows():
    """2.6e7 nonzeros: automatic tiles of 1024 rows; 2048 stands for them."""
    n, per = 52_000, 500
    rowptr = (np.arange(n + 1, dtype=np.uint64) * per)
    col = (np.arange(n * per, dtype=np.uint64) % per * 20 + np.arange(n * per, dtype=np.uint64) // per % 20)
    A = M.Csr(n, 10_000, rowptr, col.astype(np.uint32), np.ones(n * per, np.float32))
    g, f0 = np.full(n, 7, np.int32), np.ones(A.cols, np.float32)
    imgs = []
    with M.ResidentMatrix.tiles_only(A) as m:
        for rows in (0, 1024, 2048):
            with M.Recon(m, g, f0, options=M.opts(tile_rows=rows)) as r:
                r.iterate(2)
                imgs.append(r.image())
        with pytest.raises(M.MlemError):
            M.Recon(m, g, f0, options=M.opts(tile_rows=512))
    for img in imgs[1:]:
        assert np.array_equal(img.view(np.uint32), imgs[0].view(np.uint32))
