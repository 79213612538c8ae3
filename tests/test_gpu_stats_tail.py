"""Statistics summed by the backprojection's own launch (dictionary kernels of
256 and 512 lanes) against the separate kernel that lane-group backprojections
leave it to: EXACT images do not depend on the launch configuration, so every
iteration's log-likelihood and total must be the same bits. Sizes: one partial,
fewer and more than the 1024 lanes of the sum, more than two per lane."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fwd", [("dict", 8), ("dict", 64), ("dict512", 16), ("dict512", 32)])
@pytest.mark.parametrize("rows", [5, 900, 2049, 300000, 700000])     # 1 to 2735 tiles of 256 rows
def test_statistics_same_bits_as_separate_sum(rows, fwd):
    cols = 700
    rng = np.random.default_rng(rows)
    rowidx = np.cumsum(rng.integers(0, 4, rows)).astype(np.uint64)
    if not rowidx[-1]:
        rowidx[-1] = 1
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = rng.integers(0, cols, el.size)
    el["value"] = rng.random(el.size, dtype=np.float32) + np.float32(0.1)
    y = rng.poisson(9.0, rows).astype(np.int32)
    got = []
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        for bwd in (("groups", 8), ("dict", 8), ("dict", 48), ("dict512", 24)):
            A.set_launch(fwd, bwd)
            got.append(M.mlem(A, y, None, 4, mode="exact", stats=True))
    want = orc.mlem(rowidx, el, cols, y, 4)[0]
    for x, ll, total in got:
        assert np.array_equal(x, want)
        assert np.array_equal(ll, got[0][1]) and np.array_equal(total, got[0][2])
        assert ll.size == 4 and np.all(np.isfinite(ll))
