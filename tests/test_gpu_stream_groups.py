"""Streamed blocks packed by several threads in groups of chunks, blocks with many
escaped steps, and blocks left unpacked: EXACT results against the fp32
restatement, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import mlem_amd as M
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

MIN = 1 << 20          # elements of the smallest block that is packed


def _columns(kind, nnz, cols, rng):
    if kind == "steps":
        return np.cumsum(rng.choice([1, 1, 2, 96], nnz)) % cols
    if kind == "random":                       # not packed
        return rng.integers(0, cols, nnz)
    few = rng.choice([1, 3, 77], nnz)          # four in ten steps are escaped
    any_ = rng.integers(0, cols, nnz)
    return np.cumsum(np.where(rng.random(nnz) < 0.4, any_, few)) % cols


@pytest.mark.parametrize("kind", ["steps", "escapes", "random"])
@pytest.mark.parametrize("nnz", [2 * MIN - 1, 2 * MIN, 3 * MIN + 777, 5 * MIN + 4095])
@pytest.mark.parametrize("blocks", [1, 2])
def test_exact_results(nnz, kind, blocks):
    cols = 70001
    rng = np.random.default_rng(nnz)
    rows = nnz // 41
    cuts = np.sort(rng.integers(0, nnz + 1, rows - 1))
    rowidx = np.concatenate([cuts, [nnz]]).astype(np.uint64)
    el = np.zeros(nnz, M.ELEMENT_DTYPE)
    el["column"] = _columns(kind, nnz, cols, rng)
    el["value"] = rng.random(nnz, dtype=np.float32) + np.float32(0.1)
    x = rng.random(cols, dtype=np.float32) + np.float32(0.5)
    r = rng.random(rows, dtype=np.float32)
    y = rng.poisson(30.0, rows).astype(np.int32)
    block = 4 * (max(rows, cols) + 64) + 8 * (nnz // blocks + 1000)
    with M.Csr4Matrix.from_arrays(rows, cols, rowidx, el, stream_block_bytes=block) as A:
        assert A.stream_blocks() == blocks
        assert np.array_equal(M.calcFwProj(A, x, mode="exact"), orc.fwproj(rowidx, el, x))
        assert np.array_equal(M.calcBkProj(A, r, mode="exact"), orc.bkproj(rowidx, el, r, cols))
        assert np.array_equal(M.mlem(A, y, None, 3, mode="exact"),
                              orc.mlem(rowidx, el, cols, y, 3)[0])
