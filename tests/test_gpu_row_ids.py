"""Matrices of few, long rows, whose non-zeros' rows are found by a wave a row: the tile
plans against the oracle's sequential plan bit for bit, both directions, with the mean
row on both sides of the switch, rows too long for a tile and empty rows among them."""
import numpy as np
import pytest

from plan_tools import EVEN, ROUNDS, assert_same_plan, device_plan, raw_regridder

pytestmark = pytest.mark.gpu


def _matrix(nrows, mean, seed):
    rng = np.random.default_rng(seed)
    ncols = max(3 * mean, 200)
    n = rng.integers(0, 2 * mean + 1, nrows)
    n[0] = 0
    n[-1] = 0
    n[nrows // 2] += nrows * mean - n.sum() if nrows * mean > n.sum() else 0  # the mean row is `mean` or just above
    ncols = max(ncols, int(n.max()))
    rp = np.concatenate(([0], np.cumsum(n))).astype(np.int64)
    col = np.concatenate([np.sort(rng.choice(ncols, m, replace=False)) for m in n]).astype(np.int32)
    return rp, col, rng.random(rp[-1]) + 0.1, ncols


@pytest.mark.parametrize("nrows,mean", [(700, 32), (700, 33), (5, 64), (257, 200), (9, 3000)])
def test_plans_of_long_rows(cr, orc, nrows, mean):
    rp, col, val, ncols = _matrix(nrows, mean, nrows + mean)
    h = raw_regridder(cr._lib, nrows, ncols, rp, col, val)
    try:
        t = np.lexsort((np.repeat(np.arange(nrows), np.diff(rp)), col))
        trow = np.repeat(np.arange(nrows), np.diff(rp))[t].astype(np.int32)
        trp = np.concatenate(([0], np.cumsum(np.bincount(col, minlength=ncols)))).astype(np.int64)
        for style, geom in ((ROUNDS, 1), (EVEN, 0)):
            print(f"[case] long rows {nrows} x {mean} style={style} geom={geom}", flush=True)
            dev = device_plan(cr._lib, h, 0, style, geom, orc.empty_tile_plan)
            assert_same_plan(dev, orc.tile_plan(style, geom, rp, col, val, ncols))
            dev = device_plan(cr._lib, h, 1, style, geom, orc.empty_tile_plan)
            assert_same_plan(dev, orc.tile_plan(style, geom, trp, trow, val[t], nrows))
    finally:
        cr._lib.lib.cr_regridder_destroy(h)
