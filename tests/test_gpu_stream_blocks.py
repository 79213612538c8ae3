"""Streamed blocks packed to column codes: EXACT projections and iterations
(every element's row, column and value used once, in order) against the fp32
restatement, bit for bit: blocks on both sides of the smallest packed size,
whole and partial last chunks of 4096 elements, columns that pack and columns
that do not, blocks resident or not."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

CHUNK = 4096
MIN = 1 << 20          # elements of the smallest block that is packed


def _matrix(kind, nnz, cols, seed):
    rng = np.random.default_rng(seed)
    rows = max(1, nnz // 37)
    cuts = np.sort(rng.integers(0, nnz + 1, rows - 1))       # rows of any length, some empty
    rowidx = np.concatenate([cuts, [nnz]]).astype(np.uint64)
    el = np.zeros(nnz, M.ELEMENT_DTYPE)
    if kind == "steps":          # ascending, few distinct steps
        c = np.cumsum(rng.choice([0, 1, 1, 1, 2, 96], nnz)) % cols
    elif kind == "many":         # ascending, many distinct steps: most are escapes
        c = np.cumsum(rng.integers(0, 2000, nnz)) % cols
    elif kind == "random":       # does not pack
        c = rng.integers(0, cols, nnz)
    else:                        # chunk by chunk one or the other
        c = np.cumsum(rng.choice([1, 5, cols - 3], nnz)) % cols
        k = (np.arange(nnz) // CHUNK) % 2 == 1
        c[k] = rng.integers(0, cols, int(k.sum()))
    el["column"] = c
    el["value"] = rng.random(nnz, dtype=np.float32) + np.float32(0.1)
    return rows, rowidx, el


@pytest.mark.parametrize("resident", [False, True])
@pytest.mark.parametrize("kind,cols", [("steps", 1), ("steps", 7001), ("many", 90001),
                                       ("random", 90001), ("mixed", 30011)])
@pytest.mark.parametrize("nnz", [MIN - 1, MIN, MIN + 1, MIN + CHUNK - 1, 3 * MIN + 777])
def test_exact_results_of_packed_blocks(nnz, kind, cols, resident):
    rows, rowidx, el = _matrix(kind, nnz, cols, nnz + cols)
    rng = np.random.default_rng(5)
    x = rng.random(cols, dtype=np.float32) + np.float32(0.5)
    r = rng.random(rows, dtype=np.float32)
    y = rng.poisson(30.0, rows).astype(np.int32)
    # one block, or two packed ones and a smaller last one that is not
    block = 4 * (max(rows, cols) + 64) + 8 * (MIN + MIN // 3)
    keep = 2 * block if resident else 0              # the first block stays on the device
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, stream_block_bytes=block,
                                  stream_resident_bytes=keep) as A:
        assert A.stream_blocks() == (3 if nnz > 2 * MIN else 1)
        assert np.array_equal(M.calcFwProj(A, x, mode="exact"), orc.fwproj(rowidx, el, x))
        assert np.array_equal(M.calcBkProj(A, r, mode="exact"), orc.bkproj(rowidx, el, r, cols))
        assert np.array_equal(M.mlem(A, y, None, 3, mode="exact"),
                              orc.mlem(rowidx, el, cols, y, 3)[0])


# The transpose of small blocks is sorted by merging up to 131072 elements and
# digit by digit above.
@pytest.mark.parametrize("nnz", [131071, 131072, 131073, 400000])
def test_exact_results_of_small_blocks(nnz):
    cols = 5003
    rows, rowidx, el = _matrix("random", nnz, cols, nnz)
    y = np.random.default_rng(6).poisson(30.0, rows).astype(np.int32)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, stream_block_bytes=8 << 20) as A:
        assert np.array_equal(M.mlem(A, y, None, 3, mode="exact"),
                              orc.mlem(rowidx, el, cols, y, 3)[0])
