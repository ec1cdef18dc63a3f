"""Per-zone statistics: the split of a raster into chunks of tiles and its queue (emulated on the
CPU), and on the GPU the accumulation of runs, their commits and the fold of the partial records,
for zone patterns from one zone to a new zone at every cell. Data are whole numbers small enough
that every FP64 sum is exact, so all statistics are compared for equality."""
import numpy as np
import pytest


# ---- chunks of a launch and the queue (device/mapx_dev.hiph run_chunks, Sched; runtime.cpp Task) ----

def chunk_counts(ds, bs, tile, ch):
    nb = [-(-ds[i] // bs[i]) for i in (0, 1)]

    def chunks(l0, l1):
        e = [ds[i] - (nb[i] - 1) * bs[i] if last else bs[i] for i, last in ((0, l0), (1, l1))]
        return -(-(-(-e[0] // tile[0]) * -(-e[1] // tile[1])) // ch)
    return nb, chunks(False, False), chunks(True, False), chunks(False, True), chunks(True, True)


def first_chunk(nb, c, b):
    by, bx = divmod(b, nb[0])
    full = min(by, nb[1] - 1) * ((nb[0] - 1) * c[0] + c[1])
    if by == nb[1]:
        return full + (nb[0] - 1) * c[2] + c[3]
    return full + bx * (c[2] if by == nb[1] - 1 else c[0])


def chunk_of(nb, c, cl):
    by = bx = 0
    if nb[1] > 1:
        by = min(cl // ((nb[0] - 1) * c[0] + c[1]), nb[1] - 1)
    cl -= by * ((nb[0] - 1) * c[0] + c[1])
    per = c[2] if by == nb[1] - 1 else c[0]
    if nb[0] > 1:
        bx = min(cl // per, nb[0] - 1)
    return bx, by, cl - bx * per


@pytest.mark.parametrize("ds,bs,tile,ch", [((1, 1), (64, 64), (64, 64), 1), ((2100, 1037), (1024, 1024), (256, 16), 2),
                                           ((1024, 2048), (1024, 1024), (256, 16), 16), ((3001, 90), (512, 64), (256, 16), 3),
                                           ((90, 3001), (64, 512), (64, 64), 5), ((513, 513), (256, 256), (256, 16), 64)])
def test_chunks_cover_every_tile_once(ds, bs, tile, ch):
    nb, *c = chunk_counts(ds, bs, tile, ch)
    total = first_chunk(nb, c, nb[0] * nb[1])
    seen = set()
    for cl in range(total):
        bx, by, band = chunk_of(nb, c, cl)
        assert first_chunk(nb, c, by * nb[0] + bx) + band == cl  # the slots of a launch per block
        e = [min(bs[i], ds[i] - b * bs[i]) for i, b in ((0, bx), (1, by))]
        t0, t1 = -(-e[0] // tile[0]), -(-e[1] // tile[1])
        for down in (False, True):  # both orders visit the same tiles: dividing and stepping agree
            nbr = t1 if down else t0
            q, r = divmod(band * ch, nbr)
            x, y = (q, r) if down else (r, q)
            for tt in range(band * ch, min((band + 1) * ch, t0 * t1)):
                assert (x, y) == (divmod(tt, nbr) if down else divmod(tt, nbr)[::-1])
                if not down:
                    assert (bx, by, x, y) not in seen
                    seen.add((bx, by, x, y))
                if down:
                    x, y = (x, y + 1) if y + 1 < t1 else (x + 1, 0)
                else:
                    x, y = (x + 1, y) if x + 1 < t0 else (0, y + 1)
        assert min((band + 1) * ch, t0 * t1) > band * ch  # no empty chunk
    assert len(seen) == sum(-(-min(bs[0], ds[0] - i * bs[0]) // tile[0]) for i in range(nb[0])) * \
        sum(-(-min(bs[1], ds[1] - i * bs[1]) // tile[1]) for i in range(nb[1]))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 100, 4095, 4096, 4099, 20000])
def test_queue_deals_every_chunk_once(n):
    run = 3 if n >= 4096 else 0
    seen = []
    for x in range(8):
        k, last = 0, -1
        while True:
            c = ((((k >> run) << 3) + x) << run) + (k & ((1 << run) - 1))
            assert c > last  # chunk numbers increase, so the first one past the end is the last taken
            if c >= n:
                break
            seen.append(c)
            last, k = c, k + 1
    assert sorted(seen) == list(range(n))


# ---- statistics on the GPU -----------------------------------------------------------------

def zone_pattern(name, h, w, nz, rng):
    y, x = np.mgrid[0:h, 0:w]
    if name == "noise":  # a new zone at almost every cell
        return rng.integers(0, nz, (h, w))
    if name == "stripes":  # borders inside the threads' vectors, the same in every row
        return (x // 3) % nz
    if name == "diagonal":
        return ((x + 2 * y) // 37) % nz
    if name == "outside":  # ids that belong to no zone, single cells and whole vectors
        z = ((x // 8 + y // 5) % (nz + 2)) - 1
        return np.where((x + y) % 11 == 0, nz + 100, z)
    return np.zeros((h, w), np.int64)  # one zone


def check(t, v, z, nz):
    ok = (z >= 0) & (z < nz)
    v64, zz = v[ok].astype(np.float64), z[ok]
    cnt = np.bincount(zz, minlength=nz)
    assert np.array_equal(t["count"], cnt)
    assert np.array_equal(t["sum"], np.bincount(zz, weights=v64, minlength=nz))
    with np.errstate(invalid="ignore"):
        assert np.array_equal(t["mean"], np.where(cnt > 0, t["sum"] / np.maximum(cnt, 1), np.nan), equal_nan=True)
    mn, mx = np.full(nz, np.inf), np.full(nz, -np.inf)
    np.minimum.at(mn, zz, v64)
    np.maximum.at(mx, zz, v64)
    has = cnt > 0
    assert np.array_equal(np.asarray(t["min"], np.float64)[has], mn[has])
    assert np.array_equal(np.asarray(t["max"], np.float64)[has], mx[has])


def table(G, s):
    G.eval(s)
    return s.table()


SHAPES = [(1, 1, 64), (5, 3, 64), (33, 257, 64), (300, 201, 64), (1100, 1030, 1024), (2090, 2101, 512), (4096, 4352, 1024)]


@pytest.mark.gpu
@pytest.mark.parametrize("pattern,nz,dtype", [("noise", 16, np.float32), ("stripes", 17, np.float32), ("diagonal", 256, np.uint8),
                                              ("outside", 16, np.int16), ("one", 1, np.int32), ("stripes", 64, np.uint8)])
def test_statistics_of_zone_patterns(G, pattern, nz, dtype):
    rng = np.random.Generator(np.random.PCG64(5))
    for h, w, b in SHAPES:
        if pattern == "noise" and h > 2000:
            continue
        print("case zones", pattern, nz, dtype.__name__, h, w, b, flush=True)
        z = zone_pattern(pattern, h, w, nz, rng)
        lo = 0 if dtype is np.uint8 else -100
        v = rng.integers(lo, 101, (h, w)).astype(dtype)
        R, Z = G.from_array(v, (b, b)), G.from_array(z.astype(np.int32), (b, b))
        check(table(G, G.zstats(R, Z, nz)), v, z, nz)
        # reduced in the kernel of a 3x3 sum (windows in LDS); whole numbers, exact in FP32
        try:
            G.set_option("focal_zonal", 1)
            f = G.convolve(G.astype(R, G.F32), [[1, 2, 1], [0, 3, 0], [1, 0, 2]])
            tf = table(G, G.zstats(f, Z, nz))
            again = table(G, G.zstats(f + 0.0, Z, nz))
        finally:
            G.set_option("focal_zonal", 0)
        check(tf, G.to_array(f), z, nz)
        assert np.array_equal(tf["sum"], again["sum"])


@pytest.mark.gpu
def test_statistics_of_floats_repeat_bit_for_bit(G):
    """FP32 data of both signs with infinities: the FP64 sums within their rounding bound
    (n 2^-53 sum |v|), the same in every evaluation."""
    rng = np.random.Generator(np.random.PCG64(6))
    h, w, nz = 1500, 1333, 40
    v = rng.standard_normal((h, w)).astype(np.float32)
    z = zone_pattern("diagonal", h, w, nz, rng)
    v[(z == 3) & (rng.random((h, w)) < 0.01)] = np.inf
    R, Z = G.from_array(v, (512, 512)), G.from_array(z.astype(np.int32), (512, 512))
    S = G.zstats(R, Z, nz)
    runs = []
    for _ in range(3):
        G.eval(S)
        runs.append(S.table()["sum"].copy())
    assert all(np.array_equal(r, runs[0]) for r in runs)
    for i in range(nz):
        c = v[z == i].astype(np.float64)
        if i == 3:
            assert runs[0][i] == np.inf
        else:
            assert abs(runs[0][i] - np.sum(c)) <= 2 * c.size * 2.0 ** -53 * np.abs(c).sum(), i
