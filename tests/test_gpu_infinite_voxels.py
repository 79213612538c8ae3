"""FAST block products with an infinite voxel: rows that do not cross it stay
finite, whatever its place in the box (the numbers of elements are such that no
chunk ends at a multiple of 4, 8 or 32 elements)."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,frames", [(4, 4), (6, 6), (12, 12), (24, 24)])  # blocks of 4 ... 32
@pytest.mark.parametrize("extra", [1, 2, 3])     # elements beyond a multiple of 4
def test_rows_beside_an_infinite_voxel(cols, frames, extra):
    rng = np.random.default_rng(cols)
    lists = [rng.choice(cols, rng.integers(1, 4), replace=False) for _ in range(39)]
    while sum(map(len, lists)) % 4 != (extra + 2) % 4:
        lists.append(rng.choice(cols, 1))
    lists += [[0], [cols - 1]]                   # the shortest pieces come last
    rows = len(lists)
    rowidx = np.cumsum([len(a) for a in lists]).astype(np.uint64)
    assert int(rowidx[-1]) % 4 == extra % 4
    el = np.zeros(int(rowidx[-1]), M.ELEMENT_DTYPE)
    el["column"] = np.concatenate(lists)
    el["value"] = rng.random(el.size, dtype=np.float32) + np.float32(0.25)
    D = np.zeros((rows, cols))
    for i, b in enumerate(np.concatenate([[0], rowidx[:-1].astype(int)])):
        for k in range(int(b), int(rowidx[i])):
            D[i, el["column"][k]] += float(el["value"][k])
    y = rng.integers(1, 50, (frames, rows)).astype(np.float32)
    x0 = (rng.random((frames, cols)) + 0.5).astype(np.float32)
    for f in range(frames):
        x0[f, f % cols] = np.inf
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el) as A:
        n = M.calcColumnSums(A).astype(np.float64)
        x1 = M.Unrolled(A, y, x0, 1, mode="fast").xK
    for f in range(frames):
        v = f % cols
        x = x0[f].astype(np.float64)
        x[v] = 0.0
        r = np.where(D[:, v] != 0, 0.0, y[f] / np.where(D[:, v] != 0, 1.0, D @ x))  # y / inf = 0
        want = x * (D.T @ r) / np.where(n != 0, n, 1.0)
        keep = np.arange(cols) != v
        # positive sums of fewer than 50 terms, in fp32: below 64 roundings
        np.testing.assert_allclose(x1[f, keep], want[keep], rtol=64 * 2.0**-24)
