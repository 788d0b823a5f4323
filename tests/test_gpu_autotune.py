"""The autotuner's candidates cover what batches do by themselves: one run per row block on small matrices, the
shapes of the block streams on matrices that row slices do not suit; and it does with one pass's memory where that of
four is not free."""
import ctypes as C

import numpy as np
import pytest
import torch

import mlem_amd as M
from test_gpu_batch_layouts import matrix

pytestmark = pytest.mark.gpu


def layouts(m, t, **kw):
    with M.Batch(m, 4, tile_width=t["tile_width"], tile_rows=t["tile_rows"], tile_groups=t["tile_groups"],
                 tile_threads=t["tile_threads"], **kw) as b:
        return [b.layout(s) for s in (0, 1)]


def test_one_run_per_row_block_is_a_candidate(c1):
    with M.ResidentMatrix(c1["A"], c1["AT"]) as m:
        t = m.autotune(per_pass=4, values=3)
        print(t, flush=True)
        # row slices: 3 shapes at 4 and 8 runs per CU, and 512 rows with the automatic runs
        assert t["candidates"] >= 7
        a = layouts(m, t, values=3, per_pass=4)
        assert [x["tile_rows"] for x in a] == [t["tile_rows"]] * 2
        if t["tile_groups"] == 0:
            assert "one run per row block" in a[0]["kind"] + a[1]["kind"]


def test_block_stream_candidates():
    A = matrix(4000, 20000, 300, 1100)
    with M.ResidentMatrix(A, M.transpose(A)) as m:
        t = m.autotune(per_pass=4)
        print(t, flush=True)
        # 4 shapes x 4, 8 and 16 runs per CU x two workgroup sizes
        assert t["candidates"] >= 24
        assert all(x["kind"] == "block streams" for x in layouts(m, t, per_pass=4))


def test_memory_for_one_pass_only():
    """8e6 rows of one entry: vectors and partial sums of four passes need 1.15 GB beside 0.3 of tiles and their scratch,
    those of one 0.3; 1.3 GiB are free."""
    rows = 8_000_000
    rowptr = np.arange(rows + 1, dtype=np.uint64)
    col = (np.arange(rows, dtype=np.uint64) * 2654435761 % 1000).astype(np.uint32)
    A = M.Csr(rows, 1000, rowptr, col, np.ones(rows, np.float32))
    p = C.c_void_p()
    with M.ResidentMatrix(A) as m:
        m.build_transpose()
        M.release_scratch()
        before = m.info()["device_bytes"]
        assert M.hip_lib().mlem_device_alloc(C.byref(p), torch.cuda.mem_get_info(0)[0] - (1300 << 20)) == 0
        try:
            t = m.autotune(per_pass=4)
        finally:
            M.hip_lib().mlem_device_free(p)
        print(t, flush=True)
        assert t["candidates"] >= 12  # four passes at a time left 4
        assert m.info()["device_bytes"] < before + 2 * 6 * 4 * rows + (256 << 20)  # the chosen tiles at most
