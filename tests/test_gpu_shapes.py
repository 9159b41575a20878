"""Kernels at the sizes where their launch shape changes (GPU): edges of tiles
and waves, remainders, the smallest and largest of a rule's range. Answers are
whole numbers, so every comparison is exact."""
import numpy as np
import pytest

import buff_amd
from buff_amd import _native as N
from buff_amd import datagen
from buff_amd.split_double import SplitBDDoubleCompress
from oracle import refcpu, refcsv

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


def bits(words, n):
    return np.unpackbits(np.asarray(words, dtype="<u4").view(np.uint8), bitorder="little")[:n].astype(bool)


# one launch for windows of 16 .. 8192 rows (one tile a wave up to 2048 tiles, then four); the general path around it
@pytest.mark.parametrize("decimals,rows", [(1, 40), (1, 5000), (3, 70_001), (4, 2048 * TILE), (4, 2048 * TILE + 3),
                                           (6, 2100 * TILE - 1)])
@pytest.mark.parametrize("window", [15, 16, 17, 1000, 1023, 1024, 1025, 8192, 8193])
def test_windowed_max(ctx, decimals, rows, window):
    x = datagen.random_walk(rows, decimals, 21)
    ch = ctx.encode(x, 10 ** decimals)
    dlen = ch.info().dlen
    f = fixed(x, dlen)
    for s, e in {(0, rows), (min(17, rows - 1), rows), (rows // 3, rows - rows // 5), (min(1500, rows - 1), rows - 1)}:
        if e <= s:
            continue
        vals, words = ch.max_range(s, e, window, flags=buff_amd.BUFF_SEMANTIC)
        at = np.arange(0, e - s, window)
        want = np.maximum.reduceat(f[s:e], at)
        assert np.array_equal(vals, want / 2.0 ** dlen), (s, e)
        hit = np.zeros(rows, dtype=bool)
        hit[s:e] = f[s:e] == np.repeat(want, window)[: e - s]
        assert np.array_equal(bits(words, rows), hit), (s, e)
    ch.free()


# the decode of sparse columns: one, two and more dense planes, tiles with no outlier, a few, and more than one a lane
@pytest.mark.parametrize("layout", ["major", "residue"])
@pytest.mark.parametrize("decimals", [1, 2, 3, 4, 6, 8])
@pytest.mark.parametrize("rows", [2000, 40 * TILE + 7])
def test_sparse_decode(ctx, layout, decimals, rows):
    rng = np.random.default_rng(5)
    x = np.round(rng.normal(100.0, 0.5, rows), decimals)
    # the leading rows decide which columns are sparse; later tiles hold none, few, or a third of outliers
    share = np.where(np.arange(rows) < 2000, 0.02, (np.arange(rows) // TILE % 3) / 6.0)
    hit = rng.random(rows) < share
    hit[7] = True
    x[hit] = np.round(100.0 + 10.0 ** rng.uniform(5, 7, int(hit.sum())), decimals)
    ch = ctx.encode(x, 10 ** decimals, flags=buff_amd.BUFF_MAJORITY if layout == "major" else buff_amd.BUFF_RESIDUE)
    info = ch.info()
    assert info.sparse_cols > 0
    want = fixed(x, info.dlen) / 2.0 ** info.dlen
    assert np.array_equal(ch.materialize(flags=buff_amd.BUFF_SEMANTIC), want)
    ch.free()


# the filter of sparse columns: up to three columns deposited together, then more; predicates on a majority value (the
# dense planes are prefetched), an outlier value, and beyond the column
@pytest.mark.parametrize("decimals", [3, 6, 8, 10])
@pytest.mark.parametrize("rows", [2000, 3 * TILE, 41 * TILE + 5])
def test_sparse_filter(ctx, decimals, rows):
    rng = np.random.default_rng(6)
    x = np.round(rng.normal(100.0, 0.001, rows), decimals)
    hit = rng.random(rows) < 0.1
    hit[:2] = True
    x[hit] = np.round(10.0 ** rng.uniform(2, 5, int(hit.sum())), decimals)
    x[1] = 0.0
    ch = ctx.encode(x, 10 ** decimals, flags=buff_amd.BUFF_MAJORITY)
    stream = refcpu.major_encode(x, 10 ** decimals)
    info = ch.info()
    f = fixed(x, info.dlen)
    for pred in (float(x[~hit][3]), 100.0, float(x[hit][5]), 0.0, -1.0, 2e5):
        p = int(fixed(pred, info.dlen))
        for op, want in (("range", f > p), ("equal", f == p)):
            words, count = ch.filter(op, pred, flags=buff_amd.BUFF_SEMANTIC)
            assert np.array_equal(bits(words, rows), want) and count == want.sum(), (op, pred, info.sparse_cols)
            words, count = ch.filter(op, pred)
            w_ref, c_ref = refcpu.major_filter(stream, 10 ** decimals, op, pred)[:2]
            assert count == c_ref and np.array_equal(words, w_ref), (op, pred, info.sparse_cols)
    ch.free()


# short decimals (up to 8 digits, a point, up to 8 digits: the byte-parallel parse), the forms next to them, forms that
# are none, and every item position relative to a 4 KiB block; more blocks than one round of the scan
@pytest.mark.parametrize("skip", [0, 2])
@pytest.mark.parametrize("seed,count,line", [(1, 3, 3), (2, 5000, 7), (3, 40_000, 1000), (4, 40_000, 10 ** 9)])
def test_csv_short_decimals(ctx, skip, seed, count, line):
    rng = np.random.default_rng(seed)
    items = []
    for _ in range(count):
        a = "".join(rng.choice(list("0123456789"), rng.integers(0, 11)))
        b = "".join(rng.choice(list("0123456789"), rng.integers(0, 11)))
        form = rng.integers(0, 12)
        s = {0: a, 1: "." + b, 2: a + ".", 3: a + "." + b + "e3", 4: a + ".." + b, 5: a + "x" + b}.get(form, a + "." + b)
        items.append(("", "", "-", "+")[rng.integers(0, 4)] + s)
    text = "".join(t + (("\r\n" if i % 3 else "\n") if (i + 1) % line == 0 else ",") for i, t in enumerate(items))
    for tail in ("", "7.25", "\n"):
        t = (text + tail).encode()
        got = ctx.csv_parse(t, b",", skip)
        want = np.array(refcsv.construct_file_iterator_skip_newline(t, skip), dtype=np.float64)
        assert np.array_equal(got.view(np.uint64), want.view(np.uint64))


def test_csv_many_blocks(ctx):
    k = np.arange(4_500_000, dtype=np.int64) % 9973 * 1009   # 8193 blocks and more
    body = np.char.zfill(k.astype("U8"), 8)
    text = np.full((len(k), 9), ord(","), dtype=np.uint8)
    text[:, :8] = np.frombuffer(body.astype("S8").tobytes(), dtype=np.uint8).reshape(-1, 8)
    text[99::100, 8] = ord("\n")
    assert np.array_equal(ctx.csv_parse(text.tobytes()), k.astype(np.float64))
    assert np.array_equal(ctx.csv_parse(text.tobytes(), skip_val=3), k.reshape(-1, 100)[:, 3:].ravel().astype(np.float64))


# sums, maxima and encodes whose result the last workgroup hands over (one workgroup, a few, 256), and the ones around
# that take a second launch; interleaved, so that every call finds the slots as the one before left them
@pytest.mark.parametrize("decimals", [1, 4, 8])
def test_handover(ctx, decimals):
    cols = []
    for i, rows in enumerate((3, TILE, 4 * TILE + 1, 1000 * TILE, 1024 * TILE, 1024 * TILE + 1, 4096 * TILE, 4100 * TILE)):
        x = datagen.random_walk(rows, decimals, 31 + i)
        f = fixed(x, ctx_dlen := {1: 5, 4: 15, 8: 28}[decimals])
        cols.append((x, f, ctx_dlen))
    for rep in range(3):
        for x, f, dlen in cols[::-1] if rep == 1 else cols:
            ch = ctx.encode(x, 10 ** decimals)
            info = ch.info()
            assert info.base == f.min() and info.dlen == dlen
            _, exact, _ = ch.sum()
            assert exact == float(f.sum()) / 2.0 ** dlen
            if f[0] < f.max():   # row 0 as the unique maximum is the header's own rule
                assert ch.max()[0] == f.max() / 2.0 ** dlen
            assert ch.sum()[1] == exact
            ch.free()


# batch after batch on one context (the second and third take over the first's executor), two alive at once, larger
# and smaller query lists: every answer from its own batch's chunks; chunk handles made on demand
def test_batch_after_batch(ctx):
    def encode(seed, lens):
        cols = [datagen.uniform(n, -1000, 1000, 3, seed + i) for i, n in enumerate(lens)]
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
        xd = ctx.alloc(8 * int(off[-1]))
        xd.upload(np.concatenate(cols))
        b = ctx.batch_encode_device(xd.ptr, off, np.full(len(lens), 1000, dtype=np.uint64))
        xd.free()
        return b, cols

    def check(b, cols, reps):
        qs = [(N.BUFF_Q_SUM, k % len(cols), 0.0, -1, 0) for k in range(len(cols) * reps)]
        qs += [(N.BUFF_Q_GT, k, float(c[0]), -1, N.BUFF_SEMANTIC) for k, c in enumerate(cols)]
        res = b.query(qs)
        for k, r in enumerate(res):
            f = fixed(cols[k % len(cols)], 11)
            if k < len(cols) * reps:
                assert r.exact == float(f.sum()) / 2.0 ** 11
            else:
                assert r.count == (f > f[0]).sum()
                assert np.array_equal(bits(b.bitmap(r, len(f)), len(f)), f > f[0])

    first, a = encode(1, [1500, 30, 40_000])
    check(first, a, 1)
    last = first.chunks[-1]
    assert len(first.chunks) == 3 and last is first.chunks[2] and last.info().n == 40_000
    assert [c.info().n for c in first.chunks] == [1500, 30, 40_000]
    with pytest.raises(IndexError):
        first.chunks[3]
    first.free()
    assert last.handle is None
    second, b = encode(50, [70_001, 20])
    third, c = encode(90, [1024] * 9)
    for reps in (1, 300, 1):
        check(second, b, reps)
        check(third, c, reps)
    third.free()
    second.free()
    fourth, d = encode(130, [50, 2_000_000])
    check(fourth, d, 20)
    fourth.free()


# the host codec's streams, whatever their length against the room their first call gives
@pytest.mark.parametrize("rows", [2, 3, 63, 64, 65, 1024, 5000])
@pytest.mark.parametrize("decimals", [1, 3, 12])
def test_codec_sizes(ctx, rows, decimals):
    scale = 10 ** decimals
    comp = SplitBDDoubleCompress(rows, rows, scale)
    x = np.append(datagen.uniform(rows - 1, -1000, 1000, min(decimals, 4), rows), 1000.25)
    for name, flags in (("byte_fixed_encode", 0), ("byte_residue_encode", buff_amd.BUFF_RESIDUE),
                        ("buff_encode_majority", buff_amd.BUFF_MAJORITY)):
        if flags == buff_amd.BUFF_MAJORITY and rows < 2000:   # its sample
            continue
        ch = ctx.encode(x, scale, flags=flags)
        got = getattr(comp, name)(x)
        assert got.flags.owndata and np.array_equal(got, ch.serialize())
        ch.free()


# chunks whose row 0 alone holds the maximum: new minima in the first rows only, all along (the fall of a walk) and at
# the edges of groups, tiles, waves and 16-tile items; several such chunks among ordinary ones in one batch
def test_batch_row0_max(ctx):
    rng = np.random.default_rng(5)
    cols = []
    for n in (3, 64, 65, TILE, TILE + 1, 4 * TILE, 4 * TILE + 63, 15 * TILE + 1, 16 * TILE, 16 * TILE + 1, 64 * TILE + 9,
              70 * TILE - 1):
        fall = np.round(-np.arange(n) * 0.01 + rng.normal(0, 1, n), 2)
        flat = np.round(rng.normal(0, 1, n), 2)
        at = np.unique(np.clip([63, 64, TILE - 1, TILE, 4 * TILE - 1, 4 * TILE, 16 * TILE - 1, 16 * TILE], 1, n - 1))
        edges = flat.copy()
        edges[at] = -10.0 - np.arange(len(at))   # each a new minimum, the last but one row's maximum not
        for x in (fall, flat, edges):
            top = x.copy()
            top[0] = x.max() + 2
            cols += [top] if rng.random() < 0.9 else [top, x]
    keep = []
    for x in cols:
        try:
            keep.append((x, ctx.encode(x, 100)))
        except N.RefPanic:   # no row counts into the maximum
            pass
    assert len(keep) > 30
    off = np.concatenate([[0], np.cumsum([len(x) for x, _ in keep])]).astype(np.uint64)
    xd = ctx.alloc(8 * int(off[-1]))
    xd.upload(np.concatenate([x for x, _ in keep]))
    b = ctx.batch_encode_device(xd.ptr, off, np.full(len(keep), 100, dtype=np.uint64))
    xd.free()
    for (x, ch), got in zip(keep, b.chunks):
        assert np.array_equal(got.serialize(), ch.serialize()), len(x)
        ch.free()
    b.free()


# the values of a condition's rows: offsets staged in 32 and in 64 bits (decimals), more tiles than waves, one range of
# 64 tiles and many; dense, sparse and clustered conditions
@pytest.mark.parametrize("decimals,rows", [(1, 1), (2, 1000), (2, 64 * TILE), (2, 64 * TILE + 1), (4, 8192 * TILE + 5),
                                           (5, 5121 * TILE), (6, 6000 * TILE - 3), (12, 70 * TILE + 9)])
def test_condition_values(ctx, decimals, rows):
    rng = np.random.default_rng(rows)
    x = rng.integers(-10 ** 5, 10 ** 5, rows) / 100.0
    x[0] = x.min() - 1.5
    if rows == 1:
        with pytest.raises(N.RefPanic):
            ctx.encode(x, 10 ** decimals)
        return
    ch = ctx.encode(x, 10 ** decimals)
    dlen = ch.info().dlen
    f = fixed(x, dlen)
    for kind in ("dense", "sparse", "clustered", "none", "last"):
        cond = np.zeros(rows, dtype=bool)
        if kind == "dense":
            cond[:] = rng.random(rows) < 0.9
        elif kind == "sparse":
            cond[rng.integers(0, rows, max(1, rows // 50))] = True
        elif kind == "clustered":
            cond[rows // 3: rows // 3 + rows // 7 + 1] = True
        if kind != "none":
            cond[-1] = True
        words = np.packbits(cond, bitorder="little")
        words = np.pad(words, (0, -len(words) % 8)).view(np.uint32)[: (rows + 31) // 32]
        got = ch.materialize_cond(words, flags=buff_amd.BUFF_SEMANTIC)
        assert np.array_equal(got, f[cond] / 2.0 ** dlen), kind
    ch.free()


# as many ranges as a wave adds up by itself, and one more
@pytest.mark.parametrize("rows", [4096 * 64 * TILE, 4096 * 64 * TILE + 65])
def test_condition_values_largest(ctx, rows):
    x = (np.arange(rows, dtype=np.int32) * 7919 % 2001).astype(np.float64)
    x[0] = -1.5
    words = np.zeros((rows + 63) // 64, dtype=np.uint64)
    at = np.random.default_rng(rows).integers(0, len(words) - 1, 100_000)
    words[at] = 1 << 17   # a row of each of these words
    words[-1] = 1
    want = x[np.append(np.unique(at) * 64 + 17, (len(words) - 1) * 64)]
    ch = ctx.encode(x, 10)
    got = ch.materialize_cond(words.view(np.uint32)[: (rows + 31) // 32], flags=buff_amd.BUFF_SEMANTIC)
    assert np.array_equal(got, want)
    ch.free()


# the sums' launch shapes: by tiles (up to 1024, 2048, 4096, 32768 and more) and planes (one, two, more), with the
# hand-over in the launch and by two launches
@pytest.mark.parametrize("decimals,high", [(1, 50), (2, 1000), (4, 1000)])
@pytest.mark.parametrize("rows", [1024 * TILE, 1024 * TILE + 1, 2048 * TILE, 2048 * TILE + 1, 4096 * TILE + 3,
                                  32768 * TILE, 32768 * TILE + 1])
def test_sum(ctx, decimals, high, rows):
    x = datagen.uniform(rows, -high, high, decimals, rows)
    x[0] = -high - 1.5
    ch = ctx.encode(x, 10 ** decimals)
    info = ch.info()
    f = fixed(x, info.dlen)
    want = float(f.sum()) / 2.0 ** info.dlen
    a, b = ch.sum(), ch.sum_noalloc()
    assert a[1] == want and b[1] == want and a[0] == b[0] and np.array_equal(a[2], b[2])
    kept = min(5, info.dlen)   # the fraction bits of one decimal
    exact = ch.sum_precision(1, flags=buff_amd.BUFF_SEMANTIC)[1]
    drop = info.dlen - kept
    assert exact == float((((f - info.base) >> drop << drop) + info.base).sum()) / 2.0 ** info.dlen
    ch.free()


# a narrow column's sum takes the time of its bytes: 13 bits a row against 26
def test_sum_time(ctx):
    rows = 1 << 26
    us = []
    for decimals, high in ((1, 50), (4, 1000)):
        x = datagen.uniform(rows, -high, high, decimals, 3)
        x[0] = -high - 1.5
        ch = ctx.encode(x, 10 ** decimals)
        best = np.inf
        for _ in range(8):
            ctx.prof_reset()
            ctx.prof_enable(True)
            ch.sum()
            best = min(best, ctx.prof_query("k_sum")[1] * 1e3)
            ctx.prof_enable(False)
        us.append(best)
        ch.free()
    assert us[0] < 0.65 * us[1], us


# the filter on a condition's rows: its grid does not follow the plain filter's shapes (up to 8192 tiles, to 32768, more)
@pytest.mark.parametrize("rows", [TILE + 1, 8192 * TILE, 8192 * TILE + 1, 32768 * TILE, 32768 * TILE + 65])
def test_condition_filter(ctx, rows):
    rng = np.random.default_rng(rows)
    x = rng.integers(-10 ** 5, 10 ** 5, rows) / 100.0
    x[0] = x.min() - 1.5
    ch = ctx.encode(x, 100)
    f = fixed(x, ch.info().dlen)
    for share in (0.02, 0.9):
        cond = np.repeat(rng.random((rows + 63) // 64) < share, 64)[:rows]
        cond[-1] = True
        words = np.packbits(cond, bitorder="little")
        words = np.pad(words, (0, -len(words) % 4)).view(np.uint32)
        for op, hit in (("range", f > f[rows // 2]), ("equal", f == f[rows // 2])):
            got, count = ch.filter_cond(op, float(x[rows // 2]), words, flags=buff_amd.BUFF_SEMANTIC)
            assert np.array_equal(bits(got, rows), hit & cond) and count == (hit & cond).sum(), (op, share)
    ch.free()


# twice the tiles, few of them with a condition row: 1.35 times the time (1.8 on more workgroups than are resident)
def test_condition_filter_time(ctx):
    us = []
    for rows in (32768 * TILE, 65536 * TILE):
        x = datagen.random_walk(rows, 4, 5)
        ch = ctx.encode(x, 10 ** 4)
        pred = float(np.quantile(x[::97], 0.9))
        cond, words = (ctx.alloc(rows // 8) for _ in range(2))
        ch.filter_device("range", float(np.quantile(x[::97], 0.98)), cond.ptr, flags=buff_amd.BUFF_SEMANTIC)
        best = np.inf
        for _ in range(12):
            ctx.prof_reset()
            ctx.prof_enable(True)
            ch.filter_cond_device("range", pred, cond.ptr, words.ptr, flags=buff_amd.BUFF_SEMANTIC)
            ctx.synchronize()
            best = min(best, ctx.prof_query("k_filter_cond_gt")[1] * 1e3)
            ctx.prof_enable(False)
        us.append(best)
        for b in (ch, cond, words):
            b.free()
    assert us[1] < 1.6 * us[0], us


# the filters' grids: resident workgroups up to 49152 tiles, then more of them with a group of tiles a wave
@pytest.mark.parametrize("rows", [49152 * TILE, 49152 * TILE + 1])
def test_filter_lines(ctx, rows):
    x = (np.arange(rows, dtype=np.int64) * 7919 % 200_003 - 100_000) / 100.0
    x[0] = -1001.5
    ch = ctx.encode(x, 100)
    for pred in (999.0, 0.5):
        for op, want in (("range", x > pred), ("equal", x == pred)):
            words, count = ch.filter(op, pred, flags=buff_amd.BUFF_SEMANTIC)
            assert np.array_equal(bits(words, rows), want) and count == want.sum(), (op, pred)
    ch.free()


# encode and decode: up to 16384 workgroups of four tiles, then a tile a wave; sparse columns loop there
@pytest.mark.parametrize("layout", [0, buff_amd.BUFF_MAJORITY])
@pytest.mark.parametrize("rows", [65536 * TILE, 65536 * TILE + 1])
def test_decode_lines(ctx, layout, rows):
    x = np.tile(np.random.default_rng(3).integers(-4000, 4000, 999_983) / 8.0, rows // 999_983 + 1)[:rows]
    if layout:
        x[::37] = 1e6
    x[0] = x.min() - 1.5
    ch = ctx.encode(x, 10 ** 3, flags=layout)
    assert (ch.info().sparse_cols > 0) == bool(layout)
    assert np.array_equal(ch.materialize(flags=buff_amd.BUFF_SEMANTIC), x)
    ch.free()


# windowed maxima on columns of four planes: the longest windows of the one-launch form at a size, one row more, and
# windows that divide its 16 tiles
@pytest.mark.parametrize("rows,windows", [(16385 * TILE, (6144, 6145, 8192)), (65537 * TILE, (1536, 1537, 4096))])
def test_windowed_max_lines(ctx, rows, windows):
    x = datagen.random_walk(rows, 6, 23)
    ch = ctx.encode(x, 10 ** 6)
    info = ch.info()
    assert info.planes == 4
    f = fixed(x, info.dlen)
    for window in windows:
        for s in (0, 17):
            vals, words = ch.max_range(s, rows, window, flags=buff_amd.BUFF_SEMANTIC)
            want = np.maximum.reduceat(f[s:], np.arange(0, rows - s, window))
            assert np.array_equal(vals, want / 2.0 ** info.dlen), (window, s)
            hit = np.zeros(rows, dtype=bool)
            hit[s:] = f[s:] == np.repeat(want, window)[: rows - s]
            assert np.array_equal(bits(words, rows), hit), (window, s)
    ch.free()


# windows of 7001 rows against 1000 on a large column of four planes: the halo of the one-launch form is not read
def test_windowed_max_time(ctx):
    rows = 1 << 27
    x = datagen.random_walk(rows, 6, 23)
    ch = ctx.encode(x, 10 ** 6)
    vals, words = ctx.alloc(8 * (rows // 1000 + 1)), ctx.alloc(rows // 8)
    us = []
    for window in (1000, 7001):
        best = np.inf
        for _ in range(6):
            ctx.prof_reset()
            ctx.prof_enable(True)
            ch.max_range_device(0, rows, window, vals.ptr, rows // 1000 + 1, words.ptr, flags=buff_amd.BUFF_SEMANTIC)
            ctx.synchronize()
            best = min(best, ctx.prof_query("k_wmax")[1] * 1e3)
            ctx.prof_enable(False)
        us.append(best)
    for b in (ch, vals, words):
        b.free()
    assert us[1] < 1.17 * us[0], us


def batch_of(ctx, cols, scale):
    off = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.uint64)
    xd = ctx.alloc(8 * int(off[-1]))
    xd.upload(np.concatenate(cols))
    b = ctx.batch_encode_device(xd.ptr, off, np.full(len(cols), scale, dtype=np.uint64))
    xd.free()
    return b


# batched queries of as many work items as a wave folds, one more, and thousands (a workgroup folds them), beside small ones
@pytest.mark.parametrize("tiles", [511, 512, 513, 4096])
def test_batch_fold(ctx, tiles):
    cols = [datagen.uniform(n, -1000, 1000, 3, 5 + n) for n in (tiles * TILE, 40, 70_000)]
    for c in cols:
        c[0] = -1001.5
    b = batch_of(ctx, cols, 1000)
    f = [fixed(c, 11) for c in cols]
    for chunks in ((0,), (0, 1, 2), (1, 0, 2, 0, 1)):
        qs = [(op, k, 250.0, -1, N.BUFF_SEMANTIC) for op in (N.BUFF_Q_SUM, N.BUFF_Q_MAX, N.BUFF_Q_GT) for k in chunks]
        for part in (qs, qs[len(chunks): 2 * len(chunks)]):   # all of them, the maxima alone
            for (op, k, *_), r in zip(part, b.query(part)):
                if op == N.BUFF_Q_SUM:
                    assert r.exact == float(f[k].sum()) / 2.0 ** 11
                elif op == N.BUFF_Q_MAX:
                    assert r.value == f[k].max() / 2.0 ** 11
                else:
                    assert r.count == (f[k] > fixed(250.0, 11)).sum()
    b.free()


# one query on a large chunk has thousands of items: folding them takes little beside the scan
def test_batch_fold_time(ctx):
    import time

    x = datagen.uniform(1 << 24, -1000, 1000, 4, 3)
    x[0] = -1001.5
    us = {}
    for op, rows in ((N.BUFF_Q_GT, 1 << 24), (N.BUFF_Q_SUM, 1 << 24), (N.BUFF_Q_SUM, 1 << 22), (N.BUFF_Q_MAX, 1 << 22)):
        # every tile holds the top byte: the max is refined everywhere
        b = batch_of(ctx, [x[:rows]], 10 ** 4)
        q = N.prepare_queries([(op, 0, 100.0, -1, N.BUFF_SEMANTIC)])
        best = np.inf
        for _ in range(60):
            t = time.perf_counter()
            b.query(q)
            best = min(best, (time.perf_counter() - t) * 1e6)
        us[op, rows] = best
        b.free()
    assert us[N.BUFF_Q_SUM, 1 << 24] < 1.55 * us[N.BUFF_Q_GT, 1 << 24], us
    assert us[N.BUFF_Q_MAX, 1 << 22] < 1.2 * us[N.BUFF_Q_SUM, 1 << 22], us


# equality on sparse columns: all bytes the majority's with one dense plane or none, a first or a later byte that is not,
# bytes that no row has together; tiles of no outlier, one, 64, 65 and hundreds
@pytest.mark.parametrize("decimals", [1, 2, 3, 6])
@pytest.mark.parametrize("rows", [2000, 60 * TILE + 13])
def test_sparse_equality(ctx, decimals, rows):
    rng = np.random.default_rng(decimals)
    x = np.round(100.0 + 0.1 * rng.integers(-3, 4, rows), decimals)
    at = [np.array([5, 7])]   # the leading rows decide which columns are sparse
    for tile, count in zip(range(2, rows // TILE + 1), (0, 1, 64, 65, 700) * 12):
        at.append(tile * TILE + rng.choice(min(TILE, rows - tile * TILE), min(count, rows - tile * TILE), replace=False))
    at = np.concatenate(at).astype(int)
    x[at] = np.round(rng.choice([1e5, 1e5 + 7, 3e5, 7e6], len(at)), decimals)
    x[5], x[7], x[0] = 7e6, 1e5, 0.0
    ch = ctx.encode(x, 10 ** decimals, flags=buff_amd.BUFF_MAJORITY)
    stream = refcpu.major_encode(x, 10 ** decimals)
    info = ch.info()
    assert info.sparse_cols > 0
    f = fixed(x, info.dlen)
    for pred in (100.0, float(x[3]), 1e5, 1e5 + 7, 3e5, 7e6, 3e5 + 7, 5e6, 0.0):
        want = f == fixed(pred, info.dlen)
        words, count = ch.filter("equal", pred, flags=buff_amd.BUFF_SEMANTIC)
        assert np.array_equal(bits(words, rows), want) and count == want.sum(), (pred, info.sparse_cols)
        words, count = ch.filter("equal", pred)
        w_ref, c_ref = refcpu.major_filter(stream, 10 ** decimals, "equal", pred)[:2]
        assert count == c_ref and np.array_equal(words, w_ref), (pred, info.sparse_cols)
    ch.free()


# an outlier's value where a tile has more than 64 outliers against the majority's value, which reads every dense plane
def test_sparse_equality_time(ctx):
    rows = 1 << 26
    rng = np.random.default_rng(2)
    base = np.round(100.0 + 0.01 * rng.standard_normal(1 << 20), 3)
    hit = rng.random(1 << 20) < 0.09
    base[hit] = np.round(10.0 ** rng.uniform(6, 9, int(hit.sum())), 3)
    x = np.tile(base, rows >> 20)
    x[0], x[1] = 0.0, 1e9
    ch = ctx.encode(x, 1000, flags=buff_amd.BUFF_MAJORITY)
    assert ch.info().sparse_cols >= 2
    words = ctx.alloc(rows // 8)
    us = []
    for pred in (float(base[hit][3]), float(base[~hit][3])):
        best = np.inf
        for _ in range(8):
            ctx.prof_reset()
            ctx.prof_enable(True)
            ch.filter_device("equal", pred, words.ptr, flags=buff_amd.BUFF_SEMANTIC)
            ctx.synchronize()
            best = min(best, ctx.prof_query("k_major_filter_eq")[1] * 1e3)
            ctx.prof_enable(False)
        us.append(best)
    for b in (ch, words):
        b.free()
    assert us[0] < 1.08 * us[1], us


# the reference's decode of sparse columns (a later column's majority byte at twice its shift, up to its last outlier):
# tiles of no outlier, one, 64, 65 and hundreds; the last outlier at either end of a lane's 16 rows and between
@pytest.mark.parametrize("decimals", [1, 2, 3, 4])
@pytest.mark.parametrize("last", [0, 1, 7, 15])
def test_sparse_decode_reference(ctx, decimals, last):
    rows = 60 * TILE + 13
    rng = np.random.default_rng(decimals)
    x = np.round(100.0 + 0.1 * rng.integers(-3, 4, rows), decimals)
    at = [np.array([5, 7])]   # the leading rows decide which columns are sparse
    for tile, count in zip(range(2, 50), (0, 1, 64, 65, 700) * 10):
        at.append(tile * TILE + rng.choice(TILE, count, replace=False))
    at = np.concatenate(at + [[52 * TILE + 16 * 21 + last]]).astype(int)
    x[at] = np.round(rng.choice([1e5, 1e5 + 7, 3e5, 7e6], len(at)), decimals)
    x[at[-1]], x[5], x[7], x[0] = 3e5 + 1, 7e6, 1e5, 0.0
    ch = ctx.encode(x, 10 ** decimals, flags=buff_amd.BUFF_MAJORITY)
    assert ch.info().sparse_cols > 0
    assert {ch.sparse_col(j)[2] for j in range(ch.info().sparse_cols)} & {int(at[-1])}
    try:
        want = refcpu.major_decode(refcpu.major_encode(x, 10 ** decimals), 10 ** decimals)
    except refcpu.RefPanic:
        with pytest.raises(N.RefPanic):
            ch.materialize()
    else:
        assert np.array_equal(ch.materialize().view(np.uint64), want.view(np.uint64))
    ch.free()
