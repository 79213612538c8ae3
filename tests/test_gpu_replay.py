"""Replayed graphs (runs of 96 iterations or more): every kind of iteration from
a graph against the same iterations launched directly, bit for bit, over several
replays, and graphs dropped when what they hold has changed."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from mlem_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

RUN = 112            # seven replays of 16 iterations


@pytest.fixture(scope="module")
def tiny():
    p = synth.make_problem("tiny")
    m = p.matrix
    A = M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid)
    Y = np.stack([np.roll(p.y, 5 * f) for f in range(20)])
    yield p, A, Y
    A.close()


def _same_batches(a, b, frames):
    for f in range(frames):
        ia, la = a.frame_info(f)
        ib, lb = b.frame_info(f)
        assert ia == ib and np.array_equal(la, lb)
        assert np.array_equal(a.image(f), b.image(f)), f


@pytest.mark.parametrize("family", [("dict", 8), ("dict512", 32), ("tiles", 8), ("groups", 16)])
@pytest.mark.parametrize("mode", ["fast", "exact"])
def test_recon_families(tiny, mode, family):
    p, A, _ = tiny
    at_open = A.launch()
    try:
        A.set_launch(family, family)
        a, la, ta = M.mlem(A, p.y, None, RUN + 3, mode=mode, stats=True)
        b, lb, tb = M.mlem(A, p.y, None, RUN + 3, mode=mode, stats=True, use_graph=False)
        assert np.array_equal(a, b) and np.array_equal(la, lb) and np.array_equal(ta, tb)
        R = M.Recon(A, p.y, mode=mode)
        for n in (RUN, 5, RUN, 96):       # replays, direct iterations, replays of the same graph
            R.run(n)
        want = M.mlem(A, p.y, None, 2 * RUN + 101, mode=mode, use_graph=False)
        assert np.array_equal(R.image(), want)
        R.close()
    finally:
        A.set_launch(**at_open)


def test_recon_atomic(tiny):
    # sums in any order: both ways within the bound that ATOMIC mode has against
    # FP64 after 60 iterations (1e-4), in proportion
    p, A, _ = tiny
    m = p.matrix
    x64 = orc.f64_mlem(m.rowidx, m.elements, m.cols, p.y.astype(np.float64), RUN)[0]
    floor = 1e-6 * x64.max()
    for use_graph in (True, False):
        x, ll, _ = M.mlem(A, p.y, None, RUN, mode="atomic", use_graph=use_graph, stats=True)
        assert np.max(np.abs(x - x64) / np.maximum(x64, floor)) < 1e-4 * RUN / 60
        assert np.all(np.diff(ll) > -1e-6 * np.abs(ll[1:]))


def test_recon_graph_dropped_after_launch_change(tiny):
    # the graph holds the first tiles' buffers, which set_launch releases, and
    # the statistics partials of the first grid
    p, A, _ = tiny
    at_open = A.launch()
    changes = [("dict512", 32), ("tiles", 8), ("dict", 8), ("groups", 64)]
    try:
        R = M.Recon(A, p.y, mode="exact")
        E = M.Recon(A, p.y, mode="exact", use_graph=False)
        for family in changes:
            A.set_launch(family, family)
            R.run(RUN)
            E.run(RUN)
            assert np.array_equal(R.image(), E.image()), family
        m = p.matrix
        want = orc.mlem(m.rowidx, m.elements, m.cols, p.y, RUN * len(changes))[0]
        assert np.array_equal(R.image(), want)
        R.close()
        E.close()
    finally:
        A.set_launch(**at_open)


# two and more tiled blocks on two streams (FAST, from 8 frames on), EXACT
# blocks, blocks of a single frame; a frame without a budget and one that stops
# inside the replays, after which the blocks may be packed anew
@pytest.mark.parametrize("mode,width,frames", [("fast", 4, 8), ("fast", 4, 20), ("fast", 8, 17),
                                               ("fast", 16, 20), ("exact", 4, 9), ("exact", 16, 13),
                                               ("fast", 1, 3), ("exact", 1, 3)])
def test_batch(tiny, mode, width, frames):
    _, A, Y = tiny
    budgets = np.full(frames, 2 * RUN + 5, np.int32)
    budgets[0], budgets[1] = 0, RUN + 3
    a = M.Batch(A, Y[:frames], budgets, block_width=width, mode=mode, use_graph=True)
    b = M.Batch(A, Y[:frames], budgets, block_width=width, mode=mode, use_graph=False)
    assert a.run(10000) == b.run(10000) == 2 * RUN + 5
    _same_batches(a, b, frames)
    c = M.Batch(A, Y[:frames], budgets, block_width=width, mode=mode, use_graph=True)
    while c.run(100):                     # runs that end between two replays
        pass
    _same_batches(c, b, frames)
    for x in (a, b, c):
        x.close()


@pytest.mark.parametrize("mode,width", [("fast", 4), ("fast", 1), ("exact", 1)])
def test_batch_graph_dropped_after_launch_change(tiny, mode, width):
    _, A, Y = tiny
    at_open = A.launch()
    frames = 9 if width > 1 else 3
    budgets = np.full(frames, 3 * RUN, np.int32)
    try:
        a = M.Batch(A, Y[:frames], budgets, block_width=width, mode=mode, use_graph=True)
        b = M.Batch(A, Y[:frames], budgets, block_width=width, mode=mode, use_graph=False)
        for family in (("dict512", 32), ("tiles", 8), ("dict", 16)):
            A.set_launch(family, family)
            assert a.run(RUN) == b.run(RUN) == RUN
        _same_batches(a, b, frames)
        a.close()
        b.close()
    finally:
        A.set_launch(**at_open)


def test_tolerance_stops_are_found_with_and_without_graphs(tiny):
    _, A, Y = tiny
    a = M.Batch(A, Y[:9], rel_tol=1e-5, block_width=4, use_graph=True)
    b = M.Batch(A, Y[:9], rel_tol=1e-5, block_width=4, use_graph=False)
    assert a.run(3000) == b.run(3000) > 1
    _same_batches(a, b, 9)
    a.close()
    b.close()


def test_statistics_ring_wraps(tiny):
    # a reconstruction's ring holds 4096 results (its second part starts at the
    # ring's first slot again), a batch's 1024: runs that end at, before and
    # across the ring's end
    p, A, _ = tiny
    n = 4096 + 300
    x, ll, tot = M.mlem(A, p.y, None, n, mode="exact", stats=True)
    d, ld, td = M.mlem(A, p.y, None, n, mode="exact", stats=True, use_graph=False)
    assert np.array_equal(x, d) and np.array_equal(ll, ld) and np.array_equal(tot, td)
    B = M.Batch(A, p.y[None, :], block_width=1, mode="exact")
    for k in (1000, 100, 2990, 3, 3, 3, n - 4099):
        assert B.run(k) == k
    done, bl = B.frame_info(0, n)
    assert done == n and np.array_equal(B.image(0), x) and np.array_equal(bl, ll)
    B.close()


def test_statistics_ring_of_a_streamed_matrix(tiny):
    # one result per block and iteration: 4096 is no multiple of the blocks, so
    # an iteration's results lie on both sides of the ring's end
    p, _, _ = tiny
    m = p.matrix
    block = 4 * (m.rows + 64) + 8 * (int(m.rowidx[-1]) // 3 + 400)
    with M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid,
                                  stream_block_bytes=block) as S:
        nb = S.stream_blocks()
        assert nb == 3
        n = 4096 // nb + 40
        x, ll, tot = M.mlem(S, p.y, None, n, mode="exact", stats=True)
        with M.Csr4Matrix.from_arrays(m.rows, m.cols, m.rowidx, m.elements, grid=m.grid) as A:
            y, lw, tw = M.mlem(A, p.y, None, n, mode="exact", stats=True)
        assert np.array_equal(x, y)
        np.testing.assert_allclose(ll, lw, rtol=1e-11)   # FP64 sums in another fixed order
        np.testing.assert_allclose(tot, tw, rtol=1e-11)


def test_counts_whose_sum_is_not_exact_in_a_double():
    # more than 2^53 counts in all: the running double sum in file order
    rows = 4_400_000
    rng = np.random.default_rng(1)
    y = rng.integers(2**31 - 1000, 2**31 - 1, rows).astype(np.int32)
    assert float(y.sum(dtype=np.float64)) > 2.0**53
    rowidx = np.arange(1, rows + 1, dtype=np.uint64)
    el = np.zeros(rows, M.ELEMENT_DTYPE)
    el["column"] = np.arange(rows) % 300
    el["value"] = 1.0
    with M.Csr4Matrix.from_arrays(rows, 300, rowidx, el) as A:
        want = orc.init_image(M.calcColumnSums(A), y)[0]
        assert np.array_equal(M.mlem(A, y, None, 0), want)
        B = M.Batch(A, np.stack([y, y]), [0, 0], block_width=4, mode="exact")
        assert np.array_equal(B.image(0), want) and np.array_equal(B.image(1), want)
        B.close()
