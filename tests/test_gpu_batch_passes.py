"""Batches whose passes share launches: one pass, a full launch (8 passes),
one more than that, ragged last passes, and passes without an active slot
in between.  Every slot's image is bitwise the image of its sinogram alone
(the passes of a launch have their own vectors and partial sums; nothing is
summed across them)."""
import numpy as np
import pytest

import mlem_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_pass,slots,graph", [(4, 1, 0), (4, 32, 1), (4, 36, 1), (4, 41, 0), (8, 13, 1),
                                                  (8, 72, 0), (1, 11, 0)])
def test_slots_equal_their_sinograms_alone(c1, per_pass, slots, graph):
    A = c1["A"]
    rng = np.random.default_rng(slots)
    sinos = [rng.poisson(3.0 + k, A.rows).astype(np.int32) for k in range(3)]
    f0 = np.ones(A.cols, np.float32)
    idle = set(range(per_pass, 2 * per_pass)) if slots > 2 * per_pass else set()  # the second pass
    with M.ResidentMatrix(A, c1["AT"]) as m:
        alone = []
        for g in sinos:
            with M.Batch(m, 1, per_pass=per_pass) as b:
                b.set(0, g, f0)
                b.iterate(4)
                alone.append(b.image(0))
        with M.Batch(m, slots, per_pass=per_pass, use_graph=graph) as b:
            for k in range(slots):
                b.set(k, sinos[k % 3], f0)
            for k in idle:
                b.deactivate(k)
            for n in (1, 2, 1):
                b.iterate(n)
                b.sync()
            for k in range(slots):
                img = b.image(k)
                assert np.array_equal(img, f0 if k in idle else alone[k % 3]), k
