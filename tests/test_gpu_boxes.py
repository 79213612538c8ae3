"""FAST block products through 16x16x4 boxes: octets of pieces, windows of up to
1024 pieces per box and sums collected in LDS (4 and 8 frames) or stored piece
by piece (16 and 32), against FP64 MLEM.

Sizes at the edges: partial boxes, one box, no grid, windows of less than 8,
less than 64, 1023 to 1025 and several thousand pieces, an odd number of
windows, rows that fill a box (pieces are split at 512 elements) and empty ones.
"""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _matrix(grid, rows, dense, seed):
    nx, ny, nz = grid
    cols = nx * ny * nz
    rng = np.random.default_rng(seed)
    lists = []
    for r in range(rows):
        if r % 11 == 5 and rows > 11:
            lists.append(np.zeros(0, np.int64))
        elif r % 97 == 3 and dense:                      # every voxel of a 16x16x4 corner and more
            lists.append(np.arange(min(cols, 1500)))
        else:
            n = int(rng.integers(1, 1 + min(cols, 24)))
            at = int(rng.integers(0, cols))
            lists.append(np.unique((at + rng.integers(0, 3 * n, n)) % cols))
    lists[0] = np.unique(np.concatenate([lists[0], rng.integers(0, cols, 4)]))
    rowidx = np.cumsum([a.size for a in lists]).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = np.concatenate(lists)
    el["value"] = rng.random(el.size, dtype=np.float32) + np.float32(0.25)
    return rowidx, el, cols


@pytest.mark.parametrize("width", [4, 8, 16, 32])
@pytest.mark.parametrize("grid,rows,dense,with_grid", [
    ((16, 16, 4), 7, False, True),
    ((16, 16, 4), 1023, True, True),
    ((16, 16, 4), 1130, False, True),       # 1027 or so rows that have elements: a second window
    ((16, 16, 4), 2600, True, True),        # an odd number of windows
    ((17, 15, 5), 63, True, True),          # partial boxes
    ((33, 31, 9), 6000, True, True),
    ((33, 31, 9), 3000, False, False),      # no grid
    ((3, 2, 1), 40, False, True),           # a box of 6 voxels
])
def test_block_images_against_fp64(grid, rows, dense, with_grid, width):
    rowidx, el, cols = _matrix(grid, rows, dense, rows + width)
    rng = np.random.default_rng(3)
    Y = rng.poisson(20.0, (width, rows)).astype(np.int32)
    lengths = np.diff(np.concatenate([[0], rowidx.astype(np.int64)]))
    hits = np.bincount(el["column"], minlength=cols)
    # All terms are positive, so a sum of n terms in any order is within n-1
    # roundings (2^-24 each). An iteration's x * u / n has the row sums inside u
    # (at most `longest` roundings and one division), u's own sum and the column
    # sum (`most` each), a product, a quotient and the products of both passes;
    # the second iteration starts from the first one's relative error, which
    # enters f, u and x once each at most: three times in all.
    one = (lengths.max() + 2 * hits.max() + 8) * 2.0 ** -24
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, grid=grid if with_grid else None) as A:
        for iterations, tol in ((1, one), (2, 4 * one)):
            B = M.Batch(A, Y, np.full(width, iterations, np.int32), block_width=width, mode="fast")
            B.run(10)
            got = [B.image(f) for f in range(width)]
            B.close()
            for f in range(width):
                ref, _, _ = orc.f64_mlem(rowidx, el, cols, Y[f], iterations)
                assert np.array_equal(got[f] == 0, ref == 0), f
                on = ref != 0
                assert np.abs(got[f][on] / ref[on] - 1).max() <= tol, f


@pytest.mark.parametrize("frames", [1, 5, 13, 20])          # blocks of 4, 8, 16 and 32 frames
@pytest.mark.parametrize("grid,rows,dense,with_grid", [
    ((16, 16, 4), 7, False, True),          # rows of one piece
    ((33, 31, 9), 600, True, True),         # rows of 0 to 18 pieces
    ((33, 31, 9), 599, False, False),
])
def test_one_unrolled_iteration_against_fp64(grid, rows, dense, with_grid, frames):
    rowidx, el, cols = _matrix(grid, rows, dense, rows + frames)
    rng = np.random.default_rng(4)
    Y = rng.uniform(0.5, 20.0, (frames, rows)).astype(np.float32)
    X0 = rng.uniform(0.5, 2.0, (frames, cols)).astype(np.float32)
    G = rng.uniform(0.5, 2.0, (frames, cols)).astype(np.float32)
    lengths = np.diff(np.concatenate([[0], rowidx.astype(np.int64)]))
    hits = np.bincount(el["column"], minlength=cols)
    rowof = np.repeat(np.arange(rows), lengths)
    a = el["value"].astype(np.float64)

    def fwd(v):
        return np.bincount(rowof, a * v[el["column"]], rows)

    def bwd(r):
        return np.bincount(el["column"], a * r[rowof], cols)

    # Positive terms throughout (n-1 roundings for a sum of n terms, 2^-24
    # each): f and A(g x/n) have at most `longest` terms, n, u and A'(gf) at
    # most `most`; every output passes through at most three of each kind and
    # a dozen single operations. The gradient of the image is a difference of
    # two such terms: the bound is relative to their sum.
    tol = (3 * (lengths.max() + hits.max()) + 12) * 2.0 ** -24
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, grid=grid if with_grid else None) as A:
        u = M.Unrolled(A, Y, X0, K=1, mode="fast")
        gy, gx0 = u.backward(G)
        for k in range(frames):
            x, g = X0[k].astype(np.float64), G[k].astype(np.float64)
            n = np.where(hits > 0, bwd(np.ones(rows)), 1.0)
            f = fwd(x)
            on = f != 0
            fs = np.where(on, f, 1.0)
            r = np.where(on, Y[k] / fs, 0.0)
            b = bwd(r)
            gr = fwd(g * x / n)
            xK = orc.f64_unroll(rowidx, el, cols, Y[k], X0[k], 1)
            assert np.all(np.abs(u.xK[k] - xK) <= tol * np.abs(xK))
            want = np.where(on, gr / fs, 0.0)
            assert np.all(np.abs(gy[k] - want) <= tol * want)
            back = bwd(np.where(on, gr * r / fs, 0.0))
            assert np.all(np.abs(gx0[k] - (g * b / n - back)) <= tol * (g * b / n + back))
        u.close()
