"""How iterations are launched (direct, replayed graphs of several iterations)
and where the counts are summed (host loop, device integer sums): bitwise the
same results on either side of every line."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from mlem_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny():
    p = synth.make_problem("tiny")
    m = p.matrix
    A = M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid)
    yield p, A
    A.close()


# below, at and above one graph of 16 iterations and the 96-iteration line
@pytest.mark.parametrize("iterations", [1, 16, 95, 96, 113])
def test_replayed_runs_equal_direct_runs(tiny, iterations):
    p, A = tiny
    a, la, ta = M.mlem(A, p.y, None, iterations, use_graph=True, stats=True)
    b, lb, tb = M.mlem(A, p.y, None, iterations, use_graph=False, stats=True)
    assert np.array_equal(a, b) and np.array_equal(la, lb) and np.array_equal(ta, tb)
    R = M.Recon(A, p.y)  # the same iterations in two runs on one state
    R.run(iterations // 2)
    R.run(iterations - iterations // 2)
    assert np.array_equal(R.image(), a)


# statistics ring of 4096 results, batch ring of 1024: runs that wrap around
def test_statistics_past_the_ring(tiny):
    p, A = tiny
    n = 1024 + 130
    x, ll, _ = M.mlem(A, p.y, None, n, mode="exact", stats=True)
    B = M.Batch(A, p.y[None, :], block_width=4, mode="exact")
    assert B.run(100) == 100 and B.run(n - 100) == n - 100
    done, bl = B.frame_info(0)
    assert done == n and np.array_equal(B.image(0), x)
    np.testing.assert_allclose(bl, ll, rtol=1e-12)  # FP64 sums in another fixed order


def test_batch_budgets_in_one_run_and_single_steps(tiny):
    p, A = tiny
    Y = np.stack([p.y, p.y[::-1].copy(), np.roll(p.y, 7), p.y // 2, p.y + 3])
    budgets = np.array([5, 130, 0, 17, 17], np.int32)
    a = M.Batch(A, Y, budgets, block_width=4, use_graph=True)
    b = M.Batch(A, Y, budgets, block_width=4, use_graph=False)
    assert a.run(1000) == 130
    while b.run(1):
        pass
    for f in range(5):
        assert np.array_equal(a.image(f), b.image(f))
        ia, la = a.frame_info(f)
        ib, lb = b.frame_info(f)
        assert ia == ib == budgets[f] and np.array_equal(la, lb)


# host loop below 32768 counts, device sums from there on
@pytest.mark.parametrize("rows", [1, 32767, 32768, 70001])
def test_count_sums(rows):
    rng = np.random.default_rng(rows)
    y = rng.integers(-2**31, 2**31 - 1, rows).astype(np.int32)
    y[0] = -2**31
    rowidx = np.arange(1, rows + 1, dtype=np.uint64)
    el = np.zeros(rows, M.ELEMENT_DTYPE)
    el["column"] = np.arange(rows) % 3
    el["value"] = 1.0
    with M.Csr4Matrix.from_arrays(rows, 3, rowidx, el) as A:
        norm = M.calcColumnSums(A)
        want = orc.init_image(norm, y)[0]
        assert np.array_equal(M.mlem(A, y, None, 0), want)
        B = M.Batch(A, np.stack([y, y // 2]), [0, 0], block_width=4)
        assert np.array_equal(B.image(0), want)
        assert np.array_equal(B.image(1), orc.init_image(norm, y // 2)[0])


# matrices loaded by one thread and by several (from 16 MB on), of less than a
# chunk (2 MB), whole chunks and with a remainder
@pytest.mark.parametrize("rows,cols,per_row", [(4095, 4097, 3), (131072, 4096, 2), (131073, 5000, 2),
                                               (32768, 131071, 64), (33333, 131071, 75)])
def test_matrices_arrive_whole(rows, cols, per_row):
    rng = np.random.default_rng(rows)
    rowidx = np.arange(1, rows + 1, dtype=np.uint64) * per_row
    el = np.zeros(rows * per_row, M.ELEMENT_DTYPE)
    el["column"] = rng.integers(0, cols, el.size)
    el["value"] = rng.random(el.size, dtype=np.float32)
    x, r = rng.random(cols, dtype=np.float32), rng.random(rows, dtype=np.float32)
    y = rng.integers(0, 99, rows).astype(np.int32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        norm = M.calcColumnSums(A)
        assert np.array_equal(norm, orc.column_sums(rowidx, el, cols))
        assert np.array_equal(M.calcFwProj(A, x, mode="exact"), orc.fwproj(rowidx, el, x))
        assert np.array_equal(M.calcBkProj(A, r, mode="exact"), orc.bkproj(rowidx, el, r, cols))
        assert np.array_equal(M.calcCorrel(A, r, y), orc.correl(r, y))
        u = x.copy()
        assert np.array_equal(M.calcUpdate(A, norm, norm, u), orc.update(norm, norm, x))
        assert np.array_equal(M.mlem(A, y, x.copy(), 2, mode="exact", x0_given=True),
                              orc.mlem(rowidx, el, cols, y, 2, x0=x)[0])
