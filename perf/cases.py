"""The work that users have this framework do, as cases that can be timed.

listed() names the cases, draw() gives more of the same ranges, prepare() makes
what a program has in hand before the call, run() is one pass through the
public entry points, work() the bytes and operations the path cannot do
without, exact() the same outputs in 64 bits by plain torch.

A case is one of six kinds:
  recon     one sinogram reconstructed with a matrix held in HBM (mlem)
  project   one forward and one backprojection on host vectors, the step
            functions of a caller with an update rule of its own
  batch     a dynamic series against one matrix (Batch)
  unrolled  unrolled iterations and their gradients (Unrolled, backward)
  streamed  reconstruction with a matrix kept in host memory
  open      matrix loading, column sums and a reconstruction: one run of the
            command line driver from host memory
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mlem_amd as M
from mlem_amd import synth

KINDS = ("recon", "project", "batch", "unrolled", "streamed", "open")


def _case(kind, grid, lines, iterations=0, **more):
    c = {"kind": kind, "nx": grid[0], "ny": grid[1], "nz": grid[2], "lines": lines,
         "iterations": iterations, "mode": "fast", "precision": "fp32"}
    c.update(more)
    return c


def listed():
    pet = (128, 128, 48)
    return [
        # The smallest scanner of the tests, with the per-iteration statistics:
        # launches and latency, as in parameter studies and unit tests.
        _case("recon", (8, 8, 8), 4096, 20, name="recon_tiny_stats", stats=True),
        # The 32^3 workload: phantom studies, small animal frames.
        _case("recon", (32, 32, 32), 262144, 60, name="recon_small"),
        # The benchmark's clinical matrix (168.5M nonzeros), its 60 iterations.
        _case("recon", pet, 1327104, 60, name="recon_pet"),
        # Bit-exact mode for users who replace the sequential driver; grid not a
        # multiple of bricks or boxes, odd line count.
        _case("recon", (101, 99, 35), 600001, 20, name="recon_odd_exact", mode="exact"),
        # The largest matrix of the benchmark (789.8M nonzeros), fp16 values.
        _case("recon", (192, 192, 64), 4194304, 10, name="recon_large_fp16", precision="fp16"),
        # Forward projection and backprojection called on their own (penalised or
        # subset methods written by the caller).
        _case("project", (111, 111, 37), 700001, name="project_pair"),
        # A dynamic series on the clinical matrix: 32 frames, 10 to 40 iterations.
        _case("batch", pet, 1327104, 40, name="batch_pet_32", frames=32, width=32, least=10),
        # A short gated series in bit-exact mode on a ragged grid, 13 gates.
        _case("batch", (75, 77, 31), 200003, 20, name="batch_exact_13", frames=13, width=16,
              least=5, mode="exact"),
        # Training through unrolled reconstruction: the benchmark's 8 frames, 20
        # iterations, a checkpoint every 5, gradients of counts and images.
        _case("unrolled", pet, 1327104, 20, name="unrolled_pet_8", frames=8, every=5),
        # The same entry point as it comes by default (exact products, default
        # checkpoints), 3 frames.
        _case("unrolled", (64, 60, 24), 150001, 10, name="unrolled_exact_3", frames=3, every=0,
              mode="exact"),
        # A matrix larger than the memory given to it, streamed in row blocks.
        _case("streamed", (96, 96, 40), 700001, 5, name="streamed_64mib", block_mib=64),
        # Load a matrix, take its column sums, reconstruct.
        _case("open", (96, 100, 33), 500001, 30, name="open_recon"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    grid = (_log(rng, 8, 160), _log(rng, 8, 160), _log(rng, 8, 56))
    lines = _log(rng, 4000, 1300000)
    per_line = 0.42 * sum(grid)
    # a pass costs no more than the clinical reconstruction's 60 iterations
    most = 60 * 1.68e8
    if kind == "recon":
        its = max(1, min(rng.randint(5, 60), int(most / (lines * per_line))))
        precision = rng.choice(("fp32", "fp32", "fp16", "bf16"))
        return _case(kind, grid, lines, its, mode=rng.choice(("fast", "fast", "exact")),
                     precision=precision, stats=rng.random() < 0.3)
    if kind == "project":
        return _case(kind, grid, lines, mode=rng.choice(("fast", "fast", "exact")))
    if kind == "batch":
        width = rng.choice((4, 8, 16, 32))
        frames = rng.randint(2, 40)
        lines = min(lines, int(1327104 * 32 / max(frames, 32)))
        return _case(kind, grid, lines, rng.randint(8, 30), frames=frames, width=width, least=4,
                     mode=rng.choice(("fast", "fast", "exact")))
    if kind == "unrolled":
        frames = rng.randint(1, 16)
        lines = min(lines, int(1327104 * 8 / max(frames, 8)))
        return _case(kind, grid, lines, rng.randint(3, 15), frames=frames,
                     every=rng.choice((0, 0, 1, 4)), mode=rng.choice(("fast", "exact")))
    if kind == "streamed":
        return _case(kind, grid, min(lines, 700000), rng.randint(2, 6),
                     block_mib=rng.choice((8, 32, 64, 200)))
    return _case(kind, grid, min(lines, 700000), rng.randint(5, 40))


# ------------------------------------------------------------------ inputs --
def _grid(case):
    return case["nx"], case["ny"], case["nz"]


def _matrix(case, seed):
    return synth.make_matrix(_grid(case), case["lines"], 1000 + seed)


def _phantom(case, seed, scale=None):
    g = _grid(case)
    r = max(1.5, min(g) / 12.0), max(3.0, min(g[:2]) / 6.0)
    return synth.make_phantom(g, 12, 2000 + seed, r, scale=scale)


def _counts(case, m, seed):
    """One sinogram of about 75 counts a line."""
    return synth.poisson(synth.project(m, _phantom(case, seed)), 75.0 * case["lines"], 3000 + seed)


def _frames(case, m, seed):
    """Sinograms of a dynamic series: the phantom's parts scaled frame by frame,
    total counts spread over three decades."""
    n = case["frames"]
    total = synth.uniform(4000 + seed, 0, n)
    y = np.empty((n, m.rows), np.int32)
    for f in range(n):
        scale = (0.2 + 1.8 * synth.uniform(5000 + seed * 101 + f, 0, 12)).astype(np.float32)
        ybar = synth.project(m, _phantom(case, seed, scale))
        y[f] = synth.poisson(ybar, case["lines"] * 0.075 * 1000.0 ** total[f], 6000 + seed * 101 + f)
    return y


def _budgets(case, seed):
    lo, hi = case["least"], case["iterations"]
    u = synth.uniform(7000 + seed, 0, case["frames"])
    return (lo + np.floor(u * (hi - lo + 1))).astype(np.int32)


def _vectors(case, m, seed):
    """An image and a ratio sinogram as they occur inside an iteration."""
    x = _phantom(case, seed) + 0.05
    r = (0.5 + synth.uniform(8000 + seed, 0, m.rows)).astype(np.float32)
    return x.astype(np.float32), r


def _unrolled_inputs(case, m, seed):
    n = case["frames"]
    y = np.empty((n, m.rows), np.float32)
    target = np.empty((n, m.cols), np.float32)
    for f in range(n):
        scale = (0.2 + 1.8 * synth.uniform(5000 + seed * 101 + f, 0, 12)).astype(np.float32)
        target[f] = _phantom(case, seed, scale)
        ybar = synth.project(m, target[f])
        total = 75.0 * case["lines"]
        y[f] = synth.poisson(ybar, total, 6000 + seed * 101 + f)
        target[f] *= total / max(ybar.sum(), 1.0)
    x0 = np.full((n, m.cols), 0.5 * float(target.mean()) + 0.1, np.float32)
    return y, x0, target


def _open(case, m, **more):
    return M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid,
                                    precision=case["precision"], **more)


def prepare(case, seed):
    m = _matrix(case, seed)
    s = {"case": case}
    kind = case["kind"]
    if kind == "open":
        s.update(matrix=m, y=_counts(case, m, seed))
    elif kind == "streamed":
        s.update(A=_open(case, m, stream_block_bytes=case["block_mib"] << 20),
                 y=_counts(case, m, seed))
    elif kind == "recon":
        s.update(A=_open(case, m), y=_counts(case, m, seed))
    elif kind == "project":
        x, r = _vectors(case, m, seed)
        s.update(A=_open(case, m), x=x, r=r)
    elif kind == "batch":
        s.update(A=_open(case, m), y=_frames(case, m, seed), budgets=_budgets(case, seed))
        # the handle has served a series of this width before
        M.Batch(s["A"], s["y"][:1], [0], block_width=case["width"], mode=case["mode"]).close()
    else:
        y, x0, target = _unrolled_inputs(case, m, seed)
        s.update(A=_open(case, m), y=y, x0=x0)
        # dL/dx_K of a quadratic loss, about at the images a training run meets
        s["g"] = (x0 - target).astype(np.float32)
        M.Unrolled(s["A"], y, x0, 1, keep_tape=False, mode=case["mode"])
    return s


# --------------------------------------------------------------------- run --
def run(state):
    case = state["case"]
    kind, its, mode = case["kind"], case["iterations"], case["mode"]
    if kind in ("recon", "streamed"):
        if case.get("stats"):
            x, ll, total = M.mlem(state["A"], state["y"], None, its, mode=mode, stats=True)
            return {"image": x, "loglik": ll, "total": total}
        return {"image": M.mlem(state["A"], state["y"], None, its, mode=mode)}
    if kind == "project":
        return {"f": M.calcFwProj(state["A"], state["x"], mode=mode),
                "u": M.calcBkProj(state["A"], state["r"], mode=mode)}
    if kind == "batch":
        b = M.Batch(state["A"], state["y"], state["budgets"], block_width=case["width"], mode=mode)
        b.run(its)
        images = np.stack([b.image(f) for f in range(b.frames)])
        loglik = np.zeros((b.frames, its))  # a frame's history, zeros after its last iteration
        for f in range(b.frames):
            n, ll = b.frame_info(f)
            loglik[f, :n] = ll
        b.close()
        return {"images": images, "loglik": loglik}
    if kind == "unrolled":
        u = M.Unrolled(state["A"], state["y"], state["x0"], its,
                       checkpoint_interval=case["every"], mode=mode)
        gy, gx0 = u.backward(state["g"])
        u.close()
        return {"xK": u.xK, "gy": gy, "gx0": gx0}
    A = _open(case, state["matrix"])
    norm = M.calcColumnSums(A)
    x = M.mlem(A, state["y"], None, its, mode=mode)
    A.close()
    return {"norm": norm, "image": x}


# -------------------------------------------------------------------- work --
def _nnz(case):
    n = min(case["lines"], 2000)
    return synth.make_matrix(_grid(case), n, 1).nnz * (case["lines"] / n)


def work(case):
    """A product reads every matrix element once (index and value: 8 bytes, 6
    with 16-bit values) for all the right-hand sides of a block, and its
    vectors; loading and streaming read the host's 8-byte records."""
    rows, cols, nnz = case["lines"], case["nx"] * case["ny"] * case["nz"], _nnz(case)
    el = 8 if case["precision"] == "fp32" else 6
    kind, its = case["kind"], case["iterations"]
    one = 2 * el * nnz + 16 * rows + 20 * cols  # one iteration of one frame
    ops = 4 * nnz
    if kind in ("recon", "streamed"):
        return {"bytes": its * one + 4 * rows + 4 * cols, "flops": its * ops}
    if kind == "open":
        return {"bytes": 8 * nnz + its * one + 12 * rows + 8 * cols, "flops": its * ops}
    if kind == "project":
        return {"bytes": 2 * el * nnz + 8 * rows + 8 * cols, "flops": ops}
    f = case["frames"]
    if kind == "batch":
        mean = 0.5 * (case["least"] + its)
        blocks = -(-f // case["width"])
        return {"bytes": its * blocks * 2 * el * nnz + mean * f * (16 * rows + 20 * cols),
                "flops": mean * f * ops}
    # K iterations forward; recomputed once and two adjoint products backward
    return {"bytes": 3 * its * (2 * el * nnz + f * (16 * rows + 20 * cols)),
            "flops": 3 * its * f * ops}


# ------------------------------------------------------------------- exact --
class _System:
    """The matrix in 64 bits (16-bit cases: row scale times 16-bit quotient, as
    documented for those files) and its transpose, on the GPU."""

    def __init__(self, case, m):
        dev = "cuda"
        rowidx = torch.from_numpy(m.rowidx.astype(np.int64)).to(dev)
        crow = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), rowidx])
        col = torch.from_numpy(m.elements["column"].astype(np.int32)).to(dev)
        val = torch.from_numpy(np.ascontiguousarray(m.elements["value"])).to(dev)
        row = torch.repeat_interleave(torch.arange(m.rows, dtype=torch.int32, device=dev),
                                      torch.diff(crow))
        if case["precision"] == "fp32":
            val = val.double()
        else:
            s = torch.zeros(m.rows, device=dev).scatter_reduce_(0, row.long(), val, "amax")
            s = torch.where(s > 0, s, torch.ones_like(s))[row.long()]
            half = torch.float16 if case["precision"] == "fp16" else torch.bfloat16
            val = (val / s).to(half).double() * s.double()
        self.A = torch.sparse_csr_tensor(crow.int(), col, val, (m.rows, m.cols),
                                         check_invariants=False)
        order = torch.argsort(col, stable=True)
        ccol = torch.zeros(m.cols + 1, dtype=torch.int64, device=dev)
        ccol[1:] = torch.cumsum(torch.bincount(col.long(), minlength=m.cols), 0)
        self.T = torch.sparse_csr_tensor(ccol.int(), row[order], val[order], (m.cols, m.rows),
                                         check_invariants=False)
        self.norm = (self.T @ torch.ones(m.rows, 1, dtype=torch.float64, device=dev))

    def step(self, x, y):
        f = self.A @ x
        r = torch.where(f != 0, y / torch.where(f != 0, f, torch.ones_like(f)), torch.zeros_like(f))
        u = self.T @ r
        return f, r, u, x * torch.where(self.norm != 0, u / self._n(), u)

    def _n(self):
        return torch.where(self.norm != 0, self.norm, torch.ones_like(self.norm))


def _loglik(f, y):
    one = torch.ones_like(f)
    return torch.where(f > 0, y * torch.log(torch.where(f > 0, f, one)) - f, 0 * f).sum(0)


def _mlem64(S, y, its, last=None):
    """Images [cols, frames] after `its` iterations (frame f after last[f]),
    and the log-likelihoods and totals of every iteration."""
    x = (y.sum(0) / S.norm.sum()) * torch.ones(S.A.shape[1], 1, dtype=torch.float64, device="cuda")
    ll, total = [], []
    for k in range(its):
        f, _, _, xn = S.step(x, y)
        ll.append(_loglik(f, y))
        total.append(f.sum(0))
        x = xn if last is None else torch.where(last[None, :] > k, xn, x)
    return x, torch.stack(ll), torch.stack(total)


def _unrolled64(S, y, x, g, its):
    kept = []
    for _ in range(its):
        f, r, u, xn = S.step(x, y)
        kept.append((x, f, r, u))
        x = xn
    xK, gy, some = x, torch.zeros_like(y), S.norm != 0
    for x, f, r, u in reversed(kept):
        gu = torch.where(some, g * x / S._n(), g * x)
        g = torch.where(some, g * u / S._n(), g * u)
        gr = S.A @ gu
        d = torch.where(f != 0, gr / torch.where(f != 0, f, torch.ones_like(f)), 0 * gr)
        gy = gy + d
        g = g - S.T @ (d * r)
    return xK, gy, g


def exact(case, seed):
    kind, its = case["kind"], case["iterations"]
    m = _matrix(case, seed)
    S = _System(case, m)

    def dev(a):  # [frames, n] or [n] -> [n, frames] in 64 bits
        t = torch.from_numpy(np.atleast_2d(np.asarray(a))).to("cuda").double()
        return t.t().contiguous()

    if kind == "project":
        x, r = _vectors(case, m, seed)
        return {"f": (S.A @ dev(x))[:, 0], "u": (S.T @ dev(r))[:, 0]}
    if kind == "unrolled":
        y, x0, target = _unrolled_inputs(case, m, seed)
        g = (x0 - target).astype(np.float32)
        return dict(zip(("xK", "gy", "gx0"),
                        (t.t().contiguous() for t in _unrolled64(S, dev(y), dev(x0), dev(g), its))))
    if kind == "batch":
        y, last = _frames(case, m, seed), _budgets(case, seed)
        last = torch.from_numpy(last).to("cuda")
        x, ll, _ = _mlem64(S, dev(y), its, last)
        done = torch.arange(its, device="cuda")[:, None] >= last[None, :]
        return {"images": x.t().contiguous(),
                "loglik": torch.where(done, 0 * ll, ll).t().contiguous()}
    x, ll, total = _mlem64(S, dev(_counts(case, m, seed)), its)
    if kind == "open":
        return {"norm": S.norm[:, 0], "image": x[:, 0]}
    if case.get("stats"):
        return {"image": x[:, 0], "loglik": ll[:, 0], "total": total[:, 0]}
    return {"image": x[:, 0]}
