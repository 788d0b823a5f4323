"""The partial sums that runs leave for a row are added in FP64: with one entry per run and row, 60 or 200 runs, the
forward projection rounds like its products, not like a chain of as many FP32 sums.

Bar: one iteration on a matrix with one entry per column and row block makes five roundings per pixel (the row sum,
the ratio, its product with a, with f, the division by a), each 2.6e-8 rms (2^-24 / sqrt(3) over mantissas spread
over an octave): 5.8e-8, and 1.23e-7 with a chain of 60 FP32 sums (both also by direct calculation in numpy).  The bar
lies between: 8e-8."""
import numpy as np
import pytest

import mlem_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("segs", [60, 200])
@pytest.mark.parametrize("per_pass", [1, 4, 8])
def test_rows_over_many_runs(segs, per_pass):
    rng = np.random.default_rng(segs + per_pass)
    rows, w = 512, 512 if per_pass == 8 else 1024
    # row i: column 2 i (i where tiles are 512 wide) of every segment, so no two rows share a column
    col = (np.arange(segs)[None, :] * w + (w // 512) * np.arange(rows)[:, None]).astype(np.uint32)
    val = (rng.random((rows, segs)) + 0.05).astype(np.float32)
    A = M.Csr(rows, segs * w, np.arange(rows + 1, dtype=np.uint64) * segs, col.ravel(), val.ravel())
    f0 = (0.5 + rng.random(A.cols)).astype(np.float32)
    g = rng.integers(1, 50, rows).astype(np.int32)
    x = f0[col].astype(np.float64)
    ref = x * (g / (val.astype(np.float64) * x).sum(1))[:, None]
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        if per_pass == 1:
            with M.Recon(m, g, f0, options=M.opts(tile_rows=512, tile_width=1024, tile_groups=6144)) as r:
                r.iterate(1)
                img = r.image()
        else:
            with M.Batch(m, 1, per_pass=per_pass, tile_rows=512, tile_groups=6144) as b:
                assert b.layout(0)["runs"] >= segs
                b.set(0, g, f0)
                b.iterate(1)
                img = b.image(0)
    assert np.linalg.norm(img[col] - ref) <= 8e-8 * np.linalg.norm(ref)
