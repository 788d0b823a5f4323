"""Row slices may store up to a quarter more than the quad tiles of the block streams.  Where that would cost the room
for what a batch, a server's budget or the device holds with the quads, the quads are built instead: the same images
within rounding, and never a refusal that the quads would have spared."""
import ctypes as C

import numpy as np
import pytest
import torch

import mlem_amd as M
import oracle as O

pytestmark = pytest.mark.gpu

OPTS = dict(values=0, per_pass=8)  # 512 columns: the 2D ring's slices take more than its quads


def images(b, A, f0):
    gs = [np.random.default_rng(s).integers(0, 50, A.rows).astype(np.int32) for s in (1, 2)]
    for k, g in enumerate(gs):
        b.set(k, g, f0)
    b.iterate(5)
    return gs, [b.image(k) for k in range(2)]


@pytest.fixture(scope="module")
def sizes(c1):
    """Bytes of a fresh matrix and of the batch's fixed part and one pass, with slices and with quads."""
    A, out = c1["A"], {}
    f0 = np.ones(A.cols, np.float32)
    sens = O.colsum_f64(A.rowptr, A.col, A.val, A.rows, A.cols).astype(np.float32).astype(np.float64)
    free = torch.cuda.mem_get_info(0)[0]
    for kind, slots in (("row slices", 8), ("block streams", 8 * (1 + free // (8 * 4 * 2 * A.rows)))):
        with M.ResidentMatrix(A, c1["AT"]) as m:
            with M.Batch(m, slots, **OPTS) as b:
                assert [b.layout(s)["kind"].split(",")[0] for s in (0, 1)] == [kind] * 2
                before = b.info()["device_bytes"]  # partial sums of one pass: there is one, or the device is full
                fixed = before - 32 * (b.info()["passes"] - 1)  # the flags of one pass
                gs, imgs = images(b, A, f0)
                for g, img in zip(gs, imgs):
                    ref = O.mlem_f64(A.rowptr, A.col, A.val, A.rows, A.cols, g, sens, f0, 5)
                    assert np.linalg.norm(img - ref) <= 1e-5 * np.linalg.norm(ref)
                out[kind] = m.info()["device_bytes"], fixed, b.info()["device_bytes"] - before
    assert out["row slices"][0] > out["block streams"][0]
    return out


def test_a_batch_whose_passes_fill_the_device_takes_the_quads(sizes):
    """(the fixture: as many slots as the device's free memory holds, and a few; images within the bar)"""
    assert sizes["block streams"][2] == sizes["row slices"][2] > 0


def test_a_budget_that_holds_the_quads_holds_the_matrix(c1, sizes):
    A = c1["A"]
    for kept in (sizes["block streams"], sizes["row slices"]):
        budget = sum(kept) + 4096
        with M.ResidentMatrix(A, c1["AT"]) as m:
            with M.Server(hbm_budget_bytes=budget, **OPTS) as srv:
                mid = srv.add_matrix(m, slots=8)
                assert m.info()["device_bytes"] == kept[0]
                rid = srv.submit(mid, np.full(A.rows, 3, np.int32), np.ones(A.cols, np.float32), 2)
                for _ in range(20):
                    srv.step()
                    if srv.poll(rid, mid) is not None:
                        break
                else:
                    pytest.fail("the budget admits no request")


@pytest.mark.parametrize("values", [0, 3])
def test_tiles_only_on_a_device_three_quarters_full(c1, values):
    A = c1["A"]
    f0 = np.ones(A.cols, np.float32)
    p = C.c_void_p()
    kinds, imgs = [], []
    for fill in (0, 1):
        if fill:
            assert M.hip_lib().mlem_device_alloc(C.byref(p), torch.cuda.mem_get_info(0)[1] // 100 * 78) == 0
        with M.ResidentMatrix.tiles_only(A, values=values, per_pass=8) as m, M.Batch(m, 2, values=values, per_pass=8) as b:
            kinds.append([b.layout(s)["kind"].split(",")[0] for s in (0, 1)])
            imgs.append(images(b, A, f0)[1])
    M.hip_lib().mlem_device_free(p)
    assert kinds == [["row slices"] * 2, ["block streams"] * 2]
    for a, b in zip(*imgs):
        assert np.linalg.norm(a - b) <= 2e-6 * np.linalg.norm(b)


def test_a_pass_takes_the_memory_of_spare_partial_sums(c1):
    """The partial sums of several passes per launch are optional: a pass that finds the device full gets theirs, and
    the images stay the same.  33 MB per pass, filled up to 16 MB."""
    rng = np.random.default_rng(4)
    rows, per = 1_000_000, 4
    rowptr = np.arange(rows + 1, dtype=np.uint64) * per
    col = (np.sort(rng.integers(0, 1000, (rows, per)), axis=1) + 1000 * np.arange(per)).astype(np.uint32).ravel()
    A = M.Csr(rows, 4000, rowptr, col, (0.5 + rng.random(col.size)).astype(np.float32))
    gs = [rng.integers(0, 50, rows).astype(np.int32) for _ in range(3)]
    f0 = np.ones(A.cols, np.float32)
    lib, held, imgs = M.hip_lib(), [], []
    with M.ResidentMatrix(A) as m:
        m.build_transpose()
        for full in (False, True):
            with M.Batch(m, 24, per_pass=4, use_graph=1) as b:
                for k in (0, 1):
                    b.set(4 * k, gs[k], f0)
                b.iterate(2)
                b.sync()
                fixed = b.info()["device_bytes"]
                for size in ([torch.cuda.mem_get_info(0)[0] - (1 << 30)] + [16 << 20] * 256) if full else []:
                    p = C.c_void_p()
                    if lib.mlem_device_alloc(C.byref(p), size) != 0:
                        break
                    held.append(p)
                try:
                    b.set(8, gs[2], f0)
                    b.iterate(2)
                    imgs.append([b.image(4 * k) for k in range(3)])
                    one_pass = 16 * (2 * rows + A.cols)
                    if full:  # five of the six passes' partial sums given up
                        assert b.info()["device_bytes"] < fixed
                    else:
                        assert b.info()["device_bytes"] >= fixed + one_pass
                finally:
                    for p in held:
                        lib.mlem_device_free(p)
    for x, y in zip(*imgs):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
