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
