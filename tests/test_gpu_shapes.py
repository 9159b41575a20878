"""Kernels at the sizes where their launch shape changes (GPU): edges of tiles
and waves, remainders, the smallest and largest of a rule's range. Answers are
whole numbers, so every comparison is exact."""
import numpy as np
import pytest

import buff_amd
from buff_amd import datagen

pytestmark = pytest.mark.gpu

TILE = 1024


@pytest.fixture(scope="module")
def ctx():
    return buff_amd.Context(0)


def fixed(x, dlen):
    return np.trunc(np.asarray(x) * 2.0 ** dlen).astype(np.int64)


# one tile a wave up to 8192 waves, then two: every tile of the uniform column holds the top byte; the walk's maximum
# lies in a run of such tiles
@pytest.mark.parametrize("rows", [2, TILE - 1, TILE, TILE + 1, 64 * TILE + 5, 8192 * TILE, 8192 * TILE + 1,
                                  16384 * TILE + 777])
@pytest.mark.parametrize("data", ["uniform", "walk"])
def test_max_ties(ctx, rows, data):
    x = datagen.uniform(rows, -1000, 1000, 4, 11) if data == "uniform" else datagen.random_walk(rows, 4, 12)
    x[0] = x[1:].min() - 1.5   # row 0 is not the maximum: the header's range holds it
    ch = ctx.encode(x, 10 ** 4)
    info = ch.info()
    want = int(fixed(x, info.dlen).max())
    value, off = ch.max()
    assert off == want - info.base and value == want / 2.0 ** info.dlen
    ch.free()
