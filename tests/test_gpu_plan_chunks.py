"""Device tile plans of matrices with more start rows than one chunk of the
planner's chain (1024 starts of 32 rows), against the oracle's sequential plan,
bit for bit: row counts on both sides of the chunk edge, runs of long rows
(tiles that end between the 32-row starts) inside a chunk and across its edge,
and rows too long for a tile among them."""
import numpy as np
import pytest

from plan_tools import EVEN, ROUNDS, assert_same_plan, device_plan, raw_regridder

pytestmark = pytest.mark.gpu

CHUNK_ROWS = 1024 * 32


def _matrix(nrows, seed):
    rng = np.random.default_rng(seed)
    ncols = nrows + 100
    n = rng.integers(0, 9, nrows)
    for a, m in ((500, 60), (CHUNK_ROWS - 20, 50), (2 * CHUNK_ROWS + 3, 40), (nrows - 30, 30)):
        if 0 <= a and a + m <= nrows:
            n[a:a + m] = rng.integers(100, 1000, m)
            n[a + m // 2] = 2500  # over both geometries' column limit
    row = np.repeat(np.arange(nrows), n)
    start = np.minimum(np.arange(nrows), ncols - n)
    rp = np.concatenate(([0], np.cumsum(n))).astype(np.int64)
    col = (start[row] + np.arange(rp[-1]) - rp[row]).astype(np.int32)
    return rp, col, rng.random(rp[-1]) + 0.1, ncols


@pytest.mark.parametrize("nrows", [CHUNK_ROWS - 1, CHUNK_ROWS, CHUNK_ROWS + 1, CHUNK_ROWS + 33, 70001])
def test_plan_over_chunks(cr, orc, nrows):
    rp, col, val, ncols = _matrix(nrows, nrows)
    h = raw_regridder(cr._lib, nrows, ncols, rp, col, val)
    try:
        for style, geom in ((ROUNDS, 0), (ROUNDS, 1), (EVEN, 0), (EVEN, 1)):
            print(f"[case] plan chunks nrows={nrows} style={style} geom={geom}", flush=True)
            dev = device_plan(cr._lib, h, 0, style, geom, orc.empty_tile_plan)
            assert_same_plan(dev, orc.tile_plan(style, geom, rp, col, val, ncols))
    finally:
        cr._lib.lib.cr_regridder_destroy(h)


@pytest.mark.parametrize("ncols", [1, 40, 1500])
def test_plan_long_columns(cr, orc, ncols):
    """Columns that hundreds to thousands of rows hold (the earlier row is looked up
    in the transposed matrix): repeats inside a row, empty rows, columns last held
    more than a tile's rows ago or only by rows too long for a tile."""
    rng = np.random.default_rng(ncols)
    nrows = 4000
    n = rng.integers(0, 7, nrows)
    n[1000:2200] = 0
    n[::97] = 2500
    rp = np.concatenate(([0], np.cumsum(n))).astype(np.int64)
    col = rng.integers(0, ncols, rp[-1]).astype(np.int32)
    val = rng.random(rp[-1]) + 0.1
    h = raw_regridder(cr._lib, nrows, ncols, rp, col, val)
    try:
        for style, geom in ((ROUNDS, 0), (ROUNDS, 1), (EVEN, 0), (EVEN, 1)):
            print(f"[case] plan columns ncols={ncols} style={style} geom={geom}", flush=True)
            dev = device_plan(cr._lib, h, 0, style, geom, orc.empty_tile_plan)
            assert_same_plan(dev, orc.tile_plan(style, geom, rp, col, val, ncols))
    finally:
        cr._lib.lib.cr_regridder_destroy(h)
