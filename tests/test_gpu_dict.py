"""Dictionary tiles built from bitmap slabs of 2^18 indices: EXACT projections
(every element's position and value used once) against the fp32 restatement,
bit for bit, with indices at the slab edges, tiles of exactly the tile size,
empty tiles and dimensions on either side of a slab."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SLAB = 1 << 18


def _matrix(rows, cols, per_row, seed):
    rng = np.random.default_rng(seed)
    n = rng.integers(0, 2 * per_row + 1, rows)
    n[: rows // 8] = 0                                 # tiles without elements
    n[rows // 8: rows // 8 + 64] = 256                 # 16384 = 64 * 256, 2048 = 8 * 256
    rowidx = np.cumsum(n).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    c = rng.integers(0, cols, el.size)
    edges = np.array([0, 1, 31, 32, SLAB - 1, SLAB, SLAB + 1, 2 * SLAB - 1, 2 * SLAB, cols - 1])
    at = rng.integers(0, el.size, el.size // 5)
    c[at] = np.minimum(rng.choice(edges, at.size), cols - 1)
    el["column"] = c
    el["value"] = rng.random(el.size, dtype=np.float32)
    return rowidx, el


@pytest.mark.parametrize("family", [("dict", 8), ("dict", 24), ("dict", 64), ("dict512", 32)])
@pytest.mark.parametrize("rows,cols", [(3000, 1), (3000, 33), (4000, SLAB), (4001, SLAB + 1),
                                       (SLAB + 5, 3 * SLAB + 7), (2 * SLAB, 900)])
def test_exact_projections_over_slab_edges(rows, cols, family):
    rowidx, el = _matrix(rows, cols, 6 if rows > 10000 else 40, rows + cols)
    rng = np.random.default_rng(1)
    x = rng.random(cols, dtype=np.float32)
    r = rng.random(rows, dtype=np.float32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        A.set_launch(family, family)
        assert np.array_equal(M.calcFwProj(A, x, mode="exact"), orc.fwproj(rowidx, el, x))
        assert np.array_equal(M.calcBkProj(A, r, mode="exact"), orc.bkproj(rowidx, el, r, cols))


# Small matrices take smaller tiles (2048 elements up to 2.5M elements, 8192 up
# to 20M, 16384 above, or where a segment does not fit): FAST sums are the same
# bit for bit as with 16384-element tiles, whatever is chosen.
@pytest.mark.parametrize("rows,cols,per_row,longest,expect", [
    (300, 40, 3, 0, ("dict", 8)),            # one tile
    (5000, 700, 8, 0, ("dict", 8)),          # tiles end at their segment limit
    (9000, 3000, 60, 0, ("dict", 8)),
    (9000, 3000, 60, 2045, ("dict", 8)),     # the longest row that fits
    (9000, 3000, 60, 2046, ("dict512", 16)),
    (9000, 3000, 60, 8190, ("dict512", 32)),
    (40000, 30000, 80, 0, ("dict512", 16)),
])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_default_tiles_keep_the_sums(rows, cols, per_row, longest, expect, precision):
    rng = np.random.default_rng(rows + longest)
    n = rng.integers(0, 2 * per_row + 1, rows)
    n[rows // 3: rows // 3 + 900] = 0
    if longest:
        n[rows // 2] = longest
    rowidx = np.cumsum(n).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = rng.integers(0, cols, el.size)
    el["value"] = rng.random(el.size, dtype=np.float32)
    x = rng.random(cols, dtype=np.float32)
    r = rng.random(rows, dtype=np.float32)
    y = rng.integers(0, 50, rows).astype(np.int32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, precision=precision) as A:
        assert A.launch()["fwd"] == expect
        got = [M.calcFwProj(A, x), M.calcBkProj(A, r), *M.mlem(A, y, None, 4, stats=True)]
        exact = M.mlem(A, y, None, 4, mode="exact")
        A.set_launch(("dict512", 32), ("dict512", 32))
        want = [M.calcFwProj(A, x), M.calcBkProj(A, r), *M.mlem(A, y, None, 4, stats=True)]
        for a, b in zip(got[:3], want[:3]):
            assert np.array_equal(a, b)
        for a, b in zip(got[3:], want[3:]):  # FP64 sums over other workgroups
            np.testing.assert_allclose(a, b, rtol=1e-12)
        assert np.array_equal(exact, M.mlem(A, y, None, 4, mode="exact"))
