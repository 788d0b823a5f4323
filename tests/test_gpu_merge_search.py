"""Merge-path products of small matrices, whose tiles find their own split
points (up to 8192 tiles; above, a partition kernel does): tiles that end
with the last row end or the last nonzero, 1 ... 8193 tiles, empty rows in
front, between and behind, a row over many tiles, and nonzero counts of every
remainder by 4.

Bar: a row of n positive products summed in f32 in any order is within
(n + 2) * 2^-24 of its sum."""
import numpy as np
import pytest
import torch

import mlem_amd as M

pytestmark = pytest.mark.gpu


def lens_of(name):
    rng = np.random.default_rng(11)
    if name.startswith("items"):  # rows + nonzeros = the number, about 7 a row
        total = int(name[5:])
        n = max(1, total // 8)
        lens = np.full(n, (total - n) // n)
        lens[: (total - n) % n] += 1
        return lens
    if name == "empty_rows":
        return np.zeros(5000, int)
    if name == "empty_ends":
        return np.concatenate([np.zeros(3000, int), rng.integers(1, 9, 40), np.zeros(3000, int)])
    if name == "one_row":
        return np.array([50001])
    if name == "long_between":
        return np.concatenate([rng.integers(0, 4, 700), [30003], rng.integers(0, 4, 700)])
    raise ValueError(name)


@pytest.mark.parametrize("name,secsize", [(f"items{n}", 8) for n in (1, 2, 5, 2047, 2048, 2049, 4095, 4096, 40961)] +
                         [(n, s) for n in ("empty_rows", "empty_ends", "one_row", "long_between") for s in (1, 8)] +
                         [(f"items{8192 * 256}", 1), (f"items{8192 * 256 + 1}", 1), ("items30003", 32)])
def test_product_at_the_edges_of_tiles(name, secsize):
    lens = lens_of(name)
    rng = np.random.default_rng(5)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rows, nnz, cols = len(lens), int(rowptr[-1]), 977
    col = rng.integers(0, cols, max(nnz, 1)).astype(np.int32)[:nnz]
    val = (rng.random(nnz) + 0.05).astype(np.float32)
    x = (rng.random(cols) + 0.05).astype(np.float32)
    dev = [torch.from_numpy(a).cuda() for a in (rowptr, col, val, x)]
    out = torch.full((rows,), -1.0, device="cuda")
    ws = torch.zeros(M.merge_workspace_bytes(rows, nnz, secsize), dtype=torch.uint8, device="cuda")
    M.fp_merge(*(t.data_ptr() for t in dev[:3]), dev[3].data_ptr(), out.data_ptr(), secsize, rows, nnz, ws.data_ptr(),
               ws.numel(), stream=torch.cuda.current_stream().cuda_stream)
    prod = val.astype(np.float64) * x.astype(np.float64)[col]
    ref = np.add.reduceat(np.append(prod, 0.0), np.minimum(rowptr[:-1], nnz))
    ref[lens == 0] = 0.0
    assert np.all(np.abs(out.cpu().numpy().astype(np.float64) - ref) <= (lens + 2) * 2.0**-24 * ref)
