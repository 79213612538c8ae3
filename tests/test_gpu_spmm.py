"""EXACT block products of 16 and 32 frames whose lanes read the records of
their row or column 16 at a time: batches and unrolled iterations bit for bit
against the fp32 restatement, gradients against the same frame in a block of 4.
Rows and columns of 0, 1, 15 to 17, 31 to 33 and thousands of elements; numbers
of them on both sides of a workgroup's 8 or 16 and of eight workgroups."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _matrix(rows, cols, seed):
    rng = np.random.default_rng(seed)
    n = rng.choice([0, 1, 15, 16, 17, 31, 32, 33, 40], rows)
    n[0] = 5000
    rowidx = np.cumsum(n).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    # a third of the elements on the first column, the last columns empty
    c = rng.integers(0, max(1, cols - 3), el.size)
    c[rng.random(el.size) < 0.33] = 0
    el["column"] = c
    el["value"] = rng.random(el.size, dtype=np.float32) + np.float32(0.1)
    return rowidx, el


SIZES = [(1, 1), (7, 9), (8, 17), (65, 127), (128, 129), (1000, 311)]


@pytest.mark.parametrize("width", [16, 32])
@pytest.mark.parametrize("rows,cols", SIZES)
def test_exact_batch_bitwise(rows, cols, width):
    rowidx, el = _matrix(rows, cols, rows + cols)
    rng = np.random.default_rng(7)
    frames = width - 3                                    # lanes without a frame
    Y = rng.poisson(12.0, (frames, rows)).astype(np.int32)
    budgets = rng.integers(0, 4, frames).astype(np.int32)
    budgets[0] = 3
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        B = M.Batch(A, Y, budgets, block_width=width, mode="exact")
        B.run(3)
        for f in range(frames):
            want = orc.mlem(rowidx, el, cols, Y[f], int(budgets[f]))[0]
            assert np.array_equal(B.image(f), want, equal_nan=True), f
        B.close()


@pytest.mark.parametrize("frames", [13, 29])
@pytest.mark.parametrize("rows,cols", SIZES)
def test_exact_unrolled_bitwise(rows, cols, frames):
    rowidx, el = _matrix(rows, cols, rows + cols)
    rng = np.random.default_rng(8)
    Y = rng.poisson(12.0, (frames, rows)).astype(np.float32)
    X0 = rng.uniform(0.5, 1.5, (frames, cols)).astype(np.float32)
    G = rng.standard_normal((frames, cols)).astype(np.float32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        u = M.Unrolled(A, Y, X0, K=3)
        gy, gx0 = u.backward(G)
        for f in (0, frames // 2, frames - 1):
            want = orc.mlem(rowidx, el, cols, Y[f].astype(np.int32), 3, x0=X0[f])[0]
            assert np.array_equal(u.xK[f], want, equal_nan=True), f
            one = M.Unrolled(A, Y[f:f + 1], X0[f:f + 1], K=3)
            gy1, gx1 = one.backward(G[f:f + 1])
            assert np.array_equal(gy[f], gy1[0], equal_nan=True), f
            assert np.array_equal(gx0[f], gx1[0], equal_nan=True), f
            one.close()
        u.close()
