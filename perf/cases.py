"""The work a user of the MLEM engine has it do, as cases that can be timed and checked.

A case names a scanner (crystal rings, crystals per ring, image grid, sub-rays per line of response) and one of
four uses of the public entry points:

  project   one MLEM iteration out of the kernel-level calls on device pointers (forward projection, ratio, back
            projection, update), as a program does that brings its own loop: merge-path, CSR-vector, or the
            back projection by scatter over A (no transpose)
  run       one whole reconstruction over a resident matrix (mlem_run): blocked or CSR-vector kernels, eager or
            captured iterations, f32 or 16-bit matrix values
  batch     many sinograms iterated together over one resident matrix (Batch): counts in, images out
  oneshot   a new system matrix from host arrays to an image: upload, transpose, sensitivity, tiles, iterations

The scanners run from the 2D ring (2.0e6 nonzeros, where launches and latency count) over the mid-sized 3D
scanner (1.8e8) to the 12 GB one (1.5e9).  Inputs come from the package's seeded generator: Siddon-traced
intersection lengths with jittered sub-rays, ellipsoid phantoms, Poisson counts.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "bachelorarbeit-mlem_amd")
if _PKG not in sys.path:
    sys.path.append(_PKG)

import mlem_amd as M  # noqa: E402

VALUES = {"f32": 0, "bf16": 1, "fp16": 2, "uf16": 3}

RING = dict(rings=1, per_ring=288, nx=64, ny=64, nz=1, sub=0)         # the 2D ring workload
MID = dict(rings=2, per_ring=288, nx=96, ny=96, nz=24, sub=16)        # the mid-sized 3D scanner
ODD = dict(rings=2, per_ring=277, nx=95, ny=93, nz=23, sub=13)        # the same class, odd and ragged sizes
HALF = dict(rings=2, per_ring=383, nx=139, ny=141, nz=39, sub=22)     # the 12 GB scanner at under half its rows, odd
FULL = dict(rings=2, per_ring=576, nx=140, ny=140, nz=40, sub=22)     # the 12 GB scanner


def listed():
    return [
        # A program with its own loop around the kernels on the smallest scanner: four short launches an
        # iteration, each a chain of memory latencies.
        dict(name="project_ring_merge", use="project", algo="merge", **RING),
        # The CSR-vector pair in such a loop on a 3D scanner of odd sizes.
        dict(name="project_odd_csr_vector", use="project", algo="csr_vector", **ODD),
        # The back projection without a transpose (half the memory): what a program with one copy of A runs.
        dict(name="project_mid_scatter", use="project", algo="scatter", **MID),
        # 2D reconstruction in the pairing that workload names (merge-based FP, CSR-vector BP), captured
        # iterations: launch-bound.
        dict(name="run_ring_graph", use="run", algo="pair", values="f32", graph=True, iters=100, **RING),
        # The default reconstruction of a mid-sized 3D scanner.
        dict(name="run_mid", use="run", algo="merge", values="f32", graph=False, iters=30, **MID),
        # The other choice of the command line (CSR-vector kernels both ways).
        dict(name="run_mid_csr_vector", use="run", algo="csr_vector", values="f32", graph=False, iters=10, **MID),
        # 16-bit matrix values on odd sizes (the matrix that has to share the card).
        dict(name="run_odd_uf16", use="run", algo="merge", values="uf16", graph=False, iters=30, **ODD),
        # The headline: the 12 GB scanner, one reconstruction, default options.
        dict(name="run_full", use="run", algo="merge", values="f32", graph=False, iters=10, **FULL),
        # Many small 2D sinograms (slices) over one matrix, captured iterations.
        dict(name="batch_ring", use="batch", values="uf16", per_pass=4, slots=16, graph=True, iters=50, **RING),
        # A batch with unrounded values and 8 slots to a pass, the last pass ragged.
        dict(name="batch_odd_8", use="batch", values="f32", per_pass=8, slots=13, graph=False, iters=10, **ODD),
        # A large batch over a large matrix: how a scanner's queue of frames is reconstructed.
        dict(name="batch_half", use="batch", values="uf16", per_pass=4, slots=16, graph=True, iters=10, **HALF),
        # A new system matrix, once through: what one command-line run pays besides its iterations.
        dict(name="oneshot_mid", use="oneshot", values="f32", iters=10, **MID),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if rng.random() < 0.25:  # 2D rings
        nx = log_int(32, 200)
        case = dict(rings=1, per_ring=log_int(64, 500), nx=nx, ny=max(32, nx + rng.randint(-3, 3)), nz=1, sub=0)
    else:  # two rings, 3D
        nx = log_int(40, 130)
        case = dict(rings=2, per_ring=log_int(96, 330), nx=nx, ny=nx + rng.randint(-3, 3), nz=log_int(8, 38),
                    sub=log_int(4, 20))
    use = rng.choice(["project", "run", "run", "batch", "batch", "oneshot"])
    case["use"] = use
    if use == "project":
        case["algo"] = rng.choice(["merge", "csr_vector", "scatter"])
    elif use == "run":
        case["algo"] = rng.choice(["merge", "merge", "pair", "csr_vector"])
        case["values"] = rng.choice(["f32", "f32", "bf16", "fp16", "uf16"]) if case["algo"] == "merge" else "f32"
        case["graph"] = rng.random() < 0.5
        case["iters"] = rng.randint(5, 40)
    elif use == "batch":
        case["values"] = rng.choice(["f32", "bf16", "fp16", "uf16", "uf16"])
        case["per_pass"] = rng.choice([4, 4, 4, 8])
        case["slots"] = rng.randint(2, 24)
        case["graph"] = rng.random() < 0.5
        case["iters"] = rng.randint(3, 10)
    else:
        case["values"] = rng.choice(["f32", "f32", "uf16"])
        case["iters"] = rng.randint(5, 20)
    return case


def _geometry(case):
    """The scanner: a 40 mm ring of point crystals with 1 mm voxels scaled to the grid (2D), or rings of 1 mm-class
    crystals on a 35.5 mm radius around a 70 x 70 x 20 mm field of view (3D)."""
    if case["nz"] == 1:
        voxel = 64.0 / case["nx"]
        return M.geometry(case["rings"], case["per_ring"], 40.0, (0.0, 0.0, 0.0), 0.0,
                          (case["nx"], case["ny"], 1), (voxel, voxel, 1.0), case["sub"])
    return M.geometry(case["rings"], case["per_ring"], 35.5, (576.0 / case["per_ring"], 10.0, 10.0), 10.0,
                      (case["nx"], case["ny"], case["nz"]),
                      (70.0 / case["nx"], 70.0 / case["nx"], 20.0 / case["nz"]), case["sub"])


def _matrix(case, seed):
    return M.gen_system_matrix(_geometry(case), seed=seed)


def _counts(case, A, seed, n):
    """n sinograms: Poisson counts of mixtures of two phantoms' projections, totals between about 20 and 2000 per
    LOR (log-uniform)."""
    geo = _geometry(case)
    lam = []
    for k in range(2 if n > 1 else 1):
        x = M.gen_phantom(geo, seed=97 * seed + k, n_shapes=4 + k)
        g, e = M.gen_sinogram(A, x, 100.0 * A.rows, seed=97 * seed + k, return_expected=True)
        lam.append(e)
    if n == 1:
        return [g]
    rng = np.random.default_rng(seed)
    out = []
    for k in range(n):
        a, s = rng.random(), float(20.0 * 100.0 ** rng.random()) / 100.0
        out.append(rng.poisson(s * (a * lam[0] + (1.0 - a) * lam[1])).astype(np.int32))
    return out


def _slots(case):
    return case["slots"] if case["use"] == "batch" else 1


def prepare(case, seed):
    A = _matrix(case, seed)
    sinos = _counts(case, A, seed, _slots(case))
    f0 = np.ones(A.cols, np.float32)
    st = dict(case=case, f0=f0, sinos=sinos)
    if case["use"] == "oneshot":
        st["A"] = A
        st["options"] = M.opts(values=VALUES[case["values"]])
        return st
    m = M.ResidentMatrix(A)
    scatter = case.get("algo") == "scatter"
    if not scatter:
        m.build_transpose()
    st["m"] = m
    if case["use"] == "batch":
        if case["nz"] > 1:  # the row order that batches take on a 3D scanner
            m.set_row_order(M.lor_order(A, (case["nx"], case["ny"], case["nz"])))
        st["batch"] = M.Batch(m, case["slots"], values=VALUES[case["values"]], per_pass=case["per_pass"],
                              use_graph=int(case["graph"]))
        return st
    s32, _ = m.sensitivity()
    st["s32"] = s32
    if case["use"] == "run":
        algo = case["algo"]
        st["options"] = M.opts(spmv=int(algo == "csr_vector"), bp_spmv=2 if algo == "pair" else 0,
                               use_graph=int(case["graph"]), values=VALUES[case["values"]])
        return st
    # project: vectors on the device, the workspace of the merge-path kernels
    st["arrays"] = m.device_arrays()
    st["f"] = torch.from_numpy(0.5 + np.random.default_rng(seed).random(A.cols)).float().cuda()
    st["g"] = torch.from_numpy(sinos[0]).cuda()
    st["sens"] = torch.from_numpy(s32).cuda()
    st["ratio"] = torch.empty(A.rows, dtype=torch.float32, device="cuda")
    st["image"] = torch.empty(A.cols, dtype=torch.float32, device="cuda")
    if case["algo"] == "merge":
        n = max(M.merge_workspace_bytes(A.rows, A.nnz, 8), M.merge_workspace_bytes(A.cols, A.nnz, 8))
        st["ws"] = torch.empty(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    return st


def _project(st):
    m, algo = st["m"], st["case"]["algo"]
    rp, ci, va, rpT, ciT, vaT = st["arrays"]
    f, g, sens, ratio, image = (st[k].data_ptr() for k in ("f", "g", "sens", "ratio", "image"))
    s = torch.cuda.current_stream().cuda_stream
    if algo == "merge":
        ws, n = st["ws"].data_ptr(), st["ws"].numel()
        M.fp_merge(rp, ci, va, f, ratio, 8, m.rows, m.nnz, ws, n, stream=s)
    else:
        M.fp_csr_vector(rp, ci, va, f, ratio, m.rows, m.nnz, stream=s)
    M.ratio(g, ratio, m.rows, stream=s)
    if algo == "merge":
        M.bp_merge(rpT, ciT, vaT, ratio, image, 8, m.cols, m.nnz, ws, n, stream=s)
    elif algo == "csr_vector":
        M.bp_csr_vector(rpT, ciT, vaT, ratio, image, m.cols, m.nnz, stream=s)
    else:
        M.bp_scatter(rp, ci, va, ratio, image, m.rows, m.cols, m.nnz, stream=s)
    M.update(f, sens, image, m.cols, stream=s)
    return st["ratio"], st["image"]


def run(st):
    case = st["case"]
    if case["use"] == "project":
        return _project(st)
    if case["use"] == "run":
        return M.mlem_run(st["m"], st["sinos"][0], st["f0"], case["iters"], sens=st["s32"], options=st["options"])
    if case["use"] == "batch":
        b = st["batch"]
        for k, g in enumerate(st["sinos"]):
            b.set(k, g, st["f0"])
        b.iterate(case["iters"])
        return [b.image(k) for k in range(case["slots"])]
    with M.ResidentMatrix(st["A"]) as m:
        m.build_transpose()
        s32, s64 = m.sensitivity()
        return M.mlem_run(m, st["sinos"][0], st["f0"], case["iters"], sens=s32, options=st["options"]), s64


@functools.lru_cache(maxsize=None)
def _nonzeros(key):
    """The scanner's nonzeros, from up to 256 evenly spaced stretches of its rows."""
    geo = _geometry(dict(key))
    rows = M.geometry_rows(geo)
    if rows <= 65536:
        return M.gen_system_matrix(geo, seed=1).nnz
    n = 64
    starts = np.linspace(0, rows - n, 256).astype(int)
    return int(sum(M.gen_system_matrix(geo, seed=1, row_begin=int(r), row_end=int(r) + n).nnz for r in starts)
               * (rows / (n * len(starts))))


def work(case):
    """Per iteration: A for the forward and (transposed or not) for the back projection, the counts, the image and
    the sensitivity once; one multiply-add per nonzero, direction and sinogram.  Batches read A once per iteration
    whatever the number of slots."""
    geo = _geometry(case)
    rows, cols = M.geometry_rows(geo), M.geometry_cols(geo)
    nnz = _nonzeros(tuple(sorted((k, case[k]) for k in ("rings", "per_ring", "nx", "ny", "nz", "sub"))))
    slots, iters = _slots(case), case.get("iters", 1)
    per_value = 8 if case.get("values", "f32") == "f32" else 6  # value and column
    matrix = per_value * nnz + 8 * rows + (8 * cols if case.get("algo") != "scatter" else 8 * rows)
    total = iters * (matrix + per_value * nnz + slots * (8 * rows + 8 * cols) + 4 * cols)
    if case["use"] == "oneshot":
        total += 8 * nnz + 8 * rows  # the matrix from the host
    return {"bytes": int(total), "flops": int(4 * nnz * slots * iters)}


# --------------------------------------------------------------------------
# the same results in 64 bits
# --------------------------------------------------------------------------
class _Exact:
    """A in plain torch, projected in float64 over stretches of rows."""

    def __init__(self, A):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev, self.rows, self.cols = dev, A.rows, A.cols
        rowptr = A.rowptr.astype(np.int64)
        self.col = torch.from_numpy(A.col.view(np.int32)).to(dev)
        self.val = torch.from_numpy(np.ascontiguousarray(A.val)).to(dev)
        self.parts = []  # (first row, end row, first nonzero, end nonzero, row pointers within)
        r = 0
        while r < A.rows:
            e = int(np.searchsorted(rowptr, rowptr[r] + (1 << 25), side="right")) - 1
            e = min(A.rows, max(e, r + 1))
            b0, b1 = int(rowptr[r]), int(rowptr[e])
            self.parts.append((r, e, b0, b1, torch.from_numpy(rowptr[r:e + 1] - b0).to(dev)))
            r = e

    def forward(self, x):
        y = torch.zeros(self.rows, dtype=torch.float64, device=self.dev)
        for r, e, b0, b1, ptr in self.parts:
            c = torch.zeros(b1 - b0 + 1, dtype=torch.float64, device=self.dev)
            torch.cumsum(self.val[b0:b1].double() * x[self.col[b0:b1].long()], 0, out=c[1:])
            y[r:e] = c[ptr[1:]] - c[ptr[:-1]]
        return y

    def backward(self, y):
        out = torch.zeros(self.cols, dtype=torch.float64, device=self.dev)
        for r, e, b0, b1, ptr in self.parts:
            w = torch.repeat_interleave(y[r:e], ptr[1:] - ptr[:-1])
            out.index_add_(0, self.col[b0:b1].long(), self.val[b0:b1].double() * w)
        return out

    def step(self, f, g, sens):
        y = self.forward(f)
        ratio = torch.where(y != 0, g / torch.where(y != 0, y, torch.ones_like(y)), y)
        v = f * self.backward(ratio)
        return ratio, torch.where(sens == 0, v, v / torch.where(sens == 0, torch.ones_like(sens), sens))


def exact(case, seed):
    A = _matrix(case, seed)
    sinos = _counts(case, A, seed, _slots(case))
    E = _Exact(A)
    sens = E.backward(torch.ones(A.rows, dtype=torch.float64, device=E.dev))
    if case["use"] == "project":
        f = torch.from_numpy(0.5 + np.random.default_rng(seed).random(A.cols)).float().double().to(E.dev)
        return E.step(f, torch.from_numpy(sinos[0]).double().to(E.dev), sens)

    def image(k):
        g = torch.from_numpy(sinos[k]).double().to(E.dev)
        f = torch.ones(A.cols, dtype=torch.float64, device=E.dev)
        for _ in range(case["iters"]):
            f = E.step(f, g, sens)[1]
        return f.cpu().numpy()

    if case["use"] == "run":
        return image(0)
    if case["use"] == "oneshot":
        return image(0), sens.cpu().numpy()
    # a batch: its first slot and its last; the ones between would take minutes
    return [image(k) if k in (0, case["slots"] - 1) else None for k in range(case["slots"])]
