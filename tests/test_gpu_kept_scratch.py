"""The device scratch that set-up calls keep for the next matrix (from the
third matrix of a process on): every way in which it is given back, and that a
small call's tiles are not refused memory because it holds a large buffer."""
import ctypes as C

import numpy as np
import pytest
import torch

import mlem_amd as M

pytestmark = pytest.mark.gpu

NNZ = 24_000_000  # 24 bytes of transposition scratch each: 576 MB
SLACK = 64 << 20  # what the runtime itself may take in between


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(0)[0]


@pytest.fixture(scope="module")
def big():
    rows, cols = 60_000, 20_000
    rowptr = (np.arange(rows + 1, dtype=np.uint64) * (NNZ // rows)).astype(np.uint64)
    step = cols // (NNZ // rows)
    col = (np.arange(NNZ, dtype=np.uint64) % (NNZ // rows) * step
           + np.arange(NNZ, dtype=np.uint64) // (NNZ // rows) % step).astype(np.uint32)
    val = (0.5 + np.random.default_rng(1).random(NNZ)).astype(np.float32)
    return M.Csr(rows, cols, rowptr, col, val)


def transpose_once(A):
    with M.ResidentMatrix(A) as m:
        m.build_transpose()


def keep(A):
    """Scratch is kept afterwards (no matrix alive); the free memory without it."""
    for _ in range(4):
        transpose_once(A)
    M.release_scratch()
    base = free_bytes()
    transpose_once(A)
    assert base - free_bytes() > 24 * NNZ - SLACK
    return base


def test_release_gives_it_back(big):
    base = keep(big)
    M.release_scratch()
    M.release_scratch()  # nothing kept: nothing done
    assert abs(base - free_bytes()) <= SLACK


def test_batches_and_the_autotuner_give_it_back(big):
    base = keep(big)
    with M.ResidentMatrix(big) as m:
        m.build_transpose()
        with M.Batch(m, 4, values=3, per_pass=4) as b:
            held = m.info()["device_bytes"] + b.info()["device_bytes"]
            assert base - free_bytes() <= held + SLACK
        m.build_transpose()  # keeps it again
        m.autotune(per_pass=4)
        assert base - free_bytes() <= m.info()["device_bytes"] + SLACK


def test_allocations_of_the_library_get_it_back(big):
    """All of the device in pieces: the one that finds no memory gets the scratch's."""
    base = keep(big)
    lib, held = M.hip_lib(), []
    try:
        for size in [base - (4 << 30)] + [64 << 20] * 128:
            p = C.c_void_p()
            if lib.mlem_device_alloc(C.byref(p), size) != 0:
                break
            held.append(p)
        else:
            pytest.fail("the device did not fill up")
    finally:
        for p in held:
            lib.mlem_device_free(p)
    assert abs(base - free_bytes()) <= SLACK
    transpose_once(big)  # the refused allocation is not reported again by what follows


def test_a_device_more_than_half_full_keeps_none(big):
    M.release_scratch()
    p = C.c_void_p()
    assert M.hip_lib().mlem_device_alloc(C.byref(p), torch.cuda.mem_get_info(0)[1] * 6 // 10) == 0
    before = free_bytes()
    for _ in range(4):
        transpose_once(big)
    assert abs(before - free_bytes()) <= SLACK
    M.hip_lib().mlem_device_free(p)
