"""The bands of map_amd/csrc/radial.hip: every cell is stored by a band that follows those it reads, and the
aligned bands stay inside one row or column of blocks (host emulation of the launches); the scans on the
GPU at sizes with several wavefronts per octant, with and without vectors, against the oracle."""
import numpy as np
import pytest

from parity import assert_exact

DIRS = [(0, -1, 1, 0), (1, 0, 0, -1), (1, 0, 0, 1), (0, 1, 1, 0), (0, 1, -1, 0), (-1, 0, 0, 1), (-1, 0, 0, -1), (0, -1, -1, 0)]
OWN = 64


def bands(ds, bs, s, K):
    """Per launch: (octant, first column, p0, p1, smallest x or y of an aligned band, wavefronts)."""
    octs = []
    for fx, fy, sx, sy in DIRS:
        far = lambda u, o, n: n - 1 - o if u > 0 else o  # noqa: E731
        L0 = far(fx, s[0], ds[0]) if fx else far(fy, s[1], ds[1])
        L1 = far(sx, s[0], ds[0]) if sx else far(sy, s[1], ds[1])
        octs.append((fx, fy, sx, sy, L0, L1))
    b = 0
    while True:
        launch = []
        for o, (fx, fy, sx, sy, L0, L1) in enumerate(octs):
            axis, f = (0, fx) if fx else (1, fy)
            aligned = bs[axis] % K == 0
            ua = (s[axis] // K + f * b) * K
            cb = K * b if not aligned else ua - s[axis] if f > 0 else s[axis] - (ua + K - 1)
            p0, p1 = max(0, -cb), min(K, L0 - cb + 1)
            if cb > L0:
                continue
            launch.append((octs[o], cb, p0, p1, ua if aligned else None, min(cb + p1 - 1, L1) // OWN + 1))
        if not launch:
            return
        yield launch
        b += 1


@pytest.mark.parametrize("ds,bs,s,K", [((300, 220), (128, 64), (150, 73), 64), ((700, 90), (256, 32), (0, 0), 64),
                                      ((257, 129), (64, 64), (256, 128), 32), ((33, 17), (16, 16), (16, 0), 64),
                                      ((520, 390), (128, 128), (200, 150), 64), ((5, 300), (4, 64), (2, 299), 32),
                                      ((400, 40), (64, 8), (63, 20), 64), ((400, 40), (64, 8), (64, 39), 64)])
def test_bands_cover_the_raster(ds, bs, s, K):
    nb = [-(-d // b) for d, b in zip(ds, bs)]
    stored = set()
    for launch in bands(ds, bs, s, K):
        now = set()
        for (fx, fy, sx, sy, L0, L1), cb, p0, p1, ua, waves in launch:
            cell = lambda c, r: (s[0] + c * fx + r * sx, s[1] + c * fy + r * sy)  # noqa: E731
            assert 0 <= p0 < p1 <= K
            if ua is not None:  # the K cells from ua lie in one row or column of blocks
                axis, f = (0, fx) if fx else (1, fy)
                assert 0 <= ua and ua + K <= nb[axis] * bs[axis] and ua // bs[axis] == (ua + K - 1) // bs[axis]
                for p in (p0, p1 - 1):
                    assert cell(cb + p, 0)[axis] == (ua + p if f > 0 else ua + K - 1 - p)
            for w in range(waves):
                r0 = (w - 1) * OWN
                for r in range(max(0, r0), min(r0 + 2 * OWN, L1 + 1)):
                    if cb + p0 > 0 and r <= cb + p0 - 1:
                        assert cell(cb + p0 - 1, r) in stored
                    if r < r0 + OWN:
                        continue
                    for c in range(max(r, cb + p0), cb + p1):
                        x, y = cell(c, r)
                        assert 0 <= x < ds[0] and 0 <= y < ds[1]
                        now.add((x, y))
        stored |= now
    assert len(stored) == ds[0] * ds[1]


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,bs,dt", [(700, 520, (128, 64), np.float32), (650, 300, (96, 50), np.float32), (400, 333, (64, 33), np.float64),
                                       (1, 300, (64, 64), np.float32), (300, 1, (64, 64), np.float32)])
def test_scans_of_several_bands(G, O, w, h, bs, dt):
    rng = np.random.default_rng(w)
    a = (rng.standard_normal((h, w)) * 3).astype(dt)
    a[rng.random((h, w)) < 0.02] = np.nan
    a[rng.random((h, w)) < 0.01] = -np.inf
    A, oa = G.from_array(a, bs), O.from_array(a, bs)
    for s in ((w // 2, h // 2), (0, h - 1), (w - 1, 0), (min(w - 1, bs[0]), h // 3), (min(w - 1, 63), 0)):
        for red in ("rmax", "rsum"):
            print("case bands", w, h, bs, np.dtype(dt).name, red, s, flush=True)
            assert_exact(G.to_array(getattr(G, red)(A, list(s))), getattr(O, red)(oa, s).val, "%s from %s" % (red, s))
