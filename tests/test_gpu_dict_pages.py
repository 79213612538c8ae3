"""Dictionary tiles whose indices spread over many pages and several slabs of the
bitmap they are ranked in: EXACT projections against the fp32 restatement, bit
for bit."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SMALLEST = (1 << 14) * 32          # indices whose pages hold 32 of them


@pytest.mark.parametrize("family", [("dict", 8), ("dict", 48), ("dict512", 32)])
@pytest.mark.parametrize("cols", [SMALLEST, SMALLEST + 1, (1 << 24) + 3])
@pytest.mark.parametrize("spread", ["random", "corner"])
def test_exact_projections_over_pages(cols, family, spread):
    rows = 500
    rng = np.random.default_rng(cols)
    rowidx = np.cumsum(rng.integers(1, 200, rows)).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    c = rng.integers(0, cols, el.size)
    if spread == "corner":         # few pages, at both ends of the indices
        c = np.where(c % 2, cols - 1 - c % 300, c % 300)
    el["column"] = c
    el["value"] = rng.random(el.size, dtype=np.float32)
    x = rng.random(cols, dtype=np.float32)
    r = rng.random(rows, dtype=np.float32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        A.set_launch(family, family)
        assert np.array_equal(M.calcFwProj(A, x, mode="exact"), orc.fwproj(rowidx, el, x))
        assert np.array_equal(M.calcBkProj(A, r, mode="exact"), orc.bkproj(rowidx, el, r, cols))
