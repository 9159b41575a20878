"""Columns whose row 0 alone holds the maximum (GPU): the header's range counts
row 0 only as a minimum, so its maximum is the largest row that is not below
every row before it."""
import numpy as np
import pytest

import buff_amd
from buff_amd import _native as N
from oracle import refcpu

pytestmark = pytest.mark.gpu

TILE = 1024


@pytest.fixture(scope="module")
def ctx():
    return buff_amd.Context(0)


# a workgroup's range of at most four tiles (one a wave) up to 1024 tiles, then rounds of four; new minima all along, in
# the first rows only, and at the edges of groups of 64 rows, tiles, rounds and ranges
@pytest.mark.parametrize("rows", [3, 64, 65, TILE, TILE + 1, 4 * TILE - 1, 4 * TILE + 63, 9 * TILE + 5, 1024 * TILE,
                                  1024 * TILE + 1, 9 * 1024 * TILE + 77])
@pytest.mark.parametrize("kind", ["fall", "flat", "edges"])
def test_stream(ctx, rows, kind):
    rng = np.random.default_rng(rows)
    x = np.round(rng.normal(0, 1, rows), 2)
    if kind == "fall":
        x += np.round(-np.arange(rows) * 0.01, 2)
    elif kind == "edges":
        at = np.arange(1, rows // 64 + 1) * 64
        at = np.unique(np.concatenate([at[rng.integers(0, len(at), 40)] - 1, at[rng.integers(0, len(at), 40)],
                                       np.arange(TILE, rows, 5 * TILE)])) if len(at) else np.array([1])
        at = at[at < rows]
        x[at] = -10.0 - np.arange(len(at))   # each a new minimum
        x[-1] = 3.0
    x[0] = x.max() + 2
    x = np.round(x, 2)
    try:
        want = refcpu.encode(x, 100)
    except refcpu.RefPanic:   # no row counts into the maximum
        with pytest.raises(N.RefPanic):
            ctx.encode(x, 100)
        return
    ch = ctx.encode(x, 100)
    assert np.array_equal(ch.serialize(), want)
    ch.free()


# the replay of a column of 1024 tiles (ranges of four) against one row more (ranges of two): a range's tiles run side by
# side, so four are no slower than two
def test_time(ctx):
    def device_us(rows):
        x = np.round(np.random.default_rng(1).uniform(-10, 10, rows), 2)
        x[0] = 20.0
        xd = ctx.alloc(8 * rows)
        xd.upload(x)
        best = np.inf
        for _ in range(8):
            ctx.prof_reset()
            ctx.prof_enable(True)
            ctx.encode_device(xd.ptr, rows, 100).free()
            ctx.synchronize()
            best = min(best, ctx.prof_query("k_minmax_prefix")[1] * 1e3)
            ctx.prof_enable(False)
        xd.free()
        return best

    a, b = device_us(1024 * TILE), device_us(1024 * TILE + 1)
    assert a < 1.2 * b, (a, b)
