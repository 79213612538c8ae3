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
