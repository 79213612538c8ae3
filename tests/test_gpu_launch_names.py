"""launch() and set_launch(): what launch() returned can be set again, at once or
after other families, and gives the same FAST sums bit for bit (small matrices
are opened with tiles nested in the 16384-element ones)."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M

pytestmark = pytest.mark.gpu


# matrices opened with 2048-, 8192- and 16384-element tiles
@pytest.mark.parametrize("rows,cols,longest,expect", [
    (9000, 3000, 0, ("dict", 8)), (9000, 3000, 4000, ("dict512", 16)),
    (9000, 3000, 9000, ("dict512", 32))])
def test_launch_can_be_set_again(rows, cols, longest, expect):
    rng = np.random.default_rng(rows + longest)
    n = rng.integers(0, 121, rows)
    if longest:
        n[rows // 2] = longest
    rowidx = np.cumsum(n).astype(np.uint64)
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = rng.integers(0, cols, el.size)
    el["value"] = rng.random(el.size, dtype=np.float32)
    x, r = rng.random(cols, dtype=np.float32), rng.random(rows, dtype=np.float32)
    y = rng.integers(0, 50, rows).astype(np.int32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        at_open = A.launch()
        assert at_open["fwd"] == expect

        def products():
            return [M.calcFwProj(A, x), M.calcBkProj(A, r), M.mlem(A, y, None, 4)]

        want = products()
        A.set_launch(**A.launch())
        assert A.launch() == at_open
        assert all(np.array_equal(a, b) for a, b in zip(products(), want))
        A.set_launch(("groups", 16), ("tiles", 8))
        A.set_launch(**at_open)
        assert A.launch() == at_open
        assert all(np.array_equal(a, b) for a, b in zip(products(), want))
