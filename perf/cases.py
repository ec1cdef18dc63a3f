"""The measured workloads: what users of the framework evaluate, through its public entry points.

Every case is a map-algebra script of `map_amd/workloads.py` (or the example scripts they follow) over
rasters that are already resident in HBM, evaluated with `map.eval` or served with `map.Server`. A result
raster is read back with the C ABI's `ma_fetch` into a pinned buffer that the program keeps (block-tiled,
as the framework stores it); zonal results are read with `table()`. Each pass releases what it computed, so
the next one computes it again.

Sizes are those of the benchmark, the tests and the workload descriptions: Life boards from 256 cells a
side to 16384^2, DEMs of 512 to 16384 cells a side, blocks of 64 to 1024, up to 256 zones.
"""
import contextlib
import ctypes as ct
import math

import numpy as np
import torch

from map_amd import map as M
from map_amd import workloads as W

_ready = False


def _device():
    global _ready
    if not _ready:
        M.setupDevices("", M.DEV_GPU, "")
        _ready = True
    return torch.device("cuda")


# ---- the cases ------------------------------------------------------------------------


def listed():
    return [
        # an interactive board: a few generations, launches and host latency count
        {"name": "life_small", "kind": "life", "w": 320, "h": 256, "block": 64, "gens": 8, "graph": False},
        # a board of odd size in the middle of the range: ragged edge blocks
        {"name": "life_ragged", "kind": "life", "w": 3001, "h": 2003, "block": 512, "gens": 64, "graph": False},
        # the headline: 200 generations of a 16384^2 board, replayed from a graph
        {"name": "life_large", "kind": "life", "w": 16384, "h": 16384, "block": 1024, "gens": 200, "graph": True},
        # one hillshade of a DEM, the result read back (python/hill.py)
        {"name": "hillshade", "kind": "hillshade", "w": 4096, "h": 4096, "block": 512},
        # hillshade reduced per zone in one fused kernel, over a large DEM
        {"name": "hillshade_zonal", "kind": "hillshade_zonal", "w": 16384, "h": 16384, "block": 1024, "zones": 256},
        # many independent tiles evaluated together: 5x5 weighted sum, slope, threshold, per-zone sums
        {"name": "tiles", "kind": "tiles", "tiles": 128, "lo": 256, "hi": 4096, "block": 1024, "zones": 16},
        # ten requests of the served mix (hillshade, slope + aspect, 7x7 mean, zonal) in flight together
        {"name": "served", "kind": "served", "requests": 10, "lo": 512, "hi": 2048, "block": 1024},
        # a weighted overlay of four rasters (python/wsum.py) summarised per zone
        {"name": "overlay_zonal", "kind": "overlay", "w": 8191, "h": 6001, "block": 1024, "zones": 64, "dtype": "f32"},
        # the viewshed of python/view.py from one observer, the height above the line of sight read back
        {"name": "viewshed", "kind": "viewshed", "w": 1500, "h": 1100, "block": 256, "ox": 0.3, "oy": 0.6, "mask": False},
        # the visible cells of a large DEM from its centre
        {"name": "viewshed_large", "kind": "viewshed", "w": 16384, "h": 16384, "block": 1024, "ox": 0.5, "oy": 0.5, "mask": True},
        # rainfall accumulated along D8 directions, the amounts read back
        {"name": "flow", "kind": "flow", "w": 2048, "h": 1536, "block": 256, "dtype": "f32", "mask": False},
        # the stream network (cells with enough accumulated rain) of a large DEM
        {"name": "flow_large", "kind": "flow", "w": 16384, "h": 16384, "block": 1024, "dtype": "f32", "mask": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(n, block):
    """n, changed so that the last block of an axis is no narrower than the widest halo (3 cells)."""
    return n + 3 if 0 < n % block < 3 else n


def draw(rng):
    kind = rng.choice(["life", "hillshade", "hillshade_zonal", "tiles", "served", "overlay", "viewshed", "flow"])
    if kind == "tiles":
        n = _log(rng, 8, 128)
        return {"kind": kind, "tiles": n, "lo": 256, "hi": 4096, "block": rng.choice([512, 1024]), "zones": rng.choice([4, 16, 64])}
    if kind == "served":
        return {"kind": kind, "requests": rng.randint(1, 10), "lo": 512, "hi": 2048, "block": rng.choice([256, 512, 1024])}
    top = {"life": 16000, "hillshade": 8000, "hillshade_zonal": 16000, "overlay": 8000, "viewshed": 12000, "flow": 12000}[kind]
    w = _log(rng, 250, top)
    h = max(250, min(top, int(w * math.exp(rng.uniform(-0.7, 0.7)))))
    block = rng.choice([b for b in (64, 128, 256, 512, 1024) if max(w, h) / 64 <= b <= max(w, h)])
    c = {"kind": kind, "w": _fit(w, block), "h": _fit(h, block), "block": block}
    if kind == "life":
        c.update(gens=_log(rng, 4, 200), graph=rng.random() < 0.5)
    if kind in ("hillshade_zonal", "overlay"):
        c["zones"] = rng.choice([16, 64, 256])
    if kind == "overlay":
        c["dtype"] = rng.choice(["f32", "f32", "f64", "s32"])
    if kind == "viewshed":
        c.update(ox=round(rng.random(), 3), oy=round(rng.random(), 3), mask=w * h > 4e6)
    if kind == "flow":
        c.update(dtype=rng.choice(["f32", "f32", "s32", "f64"]), mask=w * h > 4e6)
    return c


# ---- inputs, made from the seed alone -----------------------------------------------------


def _gen(seed, k=0):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed) * 1000003 + k)
    return g


def _dem(seed, w, h):
    """A DEM in metres, F32: 64 Gaussian hills and eight octaves of value noise of 256 cells and less (the
    shape of the framework's own synthetic DEM)."""
    d, g = _device(), _gen(seed, 1)
    s = max(w, h) / 4096.0
    u = torch.rand(4, 64, generator=g, device=d, dtype=torch.float64)
    sig = (50 + 750 * u[2]) * s
    x = torch.arange(w, device=d, dtype=torch.float64)[None] - (u[0] * w)[:, None]
    y = torch.arange(h, device=d, dtype=torch.float64)[None] - (u[1] * h)[:, None]
    gx = torch.exp(-x * x / (2 * sig * sig)[:, None])
    gy = torch.exp(-y * y / (2 * sig * sig)[:, None]) * (3000 * u[3])[:, None]
    z = (gy.t() @ gx).float()
    for o in range(8):
        p = 256 >> o
        nh, nw = h // p + 1, w // p + 1
        lat = (torch.rand(1, 1, nh + 1, nw + 1, generator=g, device=d) * 2 - 1) * (10.0 / (1 << o))
        z += torch.nn.functional.interpolate(lat, size=(nh * p + 1, nw * p + 1), mode="bilinear", align_corners=True)[0, 0, :h, :w]
    return z


def _zones(seed, w, h, nz, dtype):
    """Voronoi zones of nz points (at an eighth of the resolution where the raster is large)."""
    d, g = _device(), _gen(seed, 2)
    f = 1 if max(w, h) <= 2048 else 8
    zw, zh = -(-w // f), -(-h // f)
    p = torch.rand(2, nz, generator=g, device=d) * torch.tensor([[zw], [zh]], device=d)
    x = torch.arange(zw, device=d, dtype=torch.float32)
    best = torch.full((zh, zw), float("inf"), device=d)
    z = torch.zeros((zh, zw), device=d, dtype=dtype)
    for i in range(nz):
        q = (torch.arange(zh, device=d, dtype=torch.float32) - p[1, i])[:, None] ** 2 + (x - p[0, i])[None] ** 2
        m = q < best
        best = torch.where(m, q, best)
        z.masked_fill_(m, i)
    return z.repeat_interleave(f, 0).repeat_interleave(f, 1)[:h, :w].contiguous() if f > 1 else z


def _d8(z):
    """Steepest-descent D8 codes: the first neighbour (E, SE, S, SW, W, NW, N, NE) with the largest drop
    per unit distance, 0 where none inside the raster is lower."""
    h, w = z.shape
    pad = torch.nn.functional.pad(z[None, None], (1, 1, 1, 1), value=float("inf"))[0, 0]
    best = torch.zeros_like(z)
    code = torch.zeros_like(z, dtype=torch.uint8)
    for (dx, dy), c in W.D8_CODES:
        drop = (z - pad[1 + dy:1 + dy + h, 1 + dx:1 + dx + w]) / (math.sqrt(2.0) if dx and dy else 1.0)
        m = drop > best
        best = torch.where(m, drop, best)
        code.masked_fill_(m, c)
    return code


_CODE = {torch.float32: M.F32, torch.float64: M.F64, torch.uint8: M.U8, torch.int32: M.S32}
_TORCH = {"f32": torch.float32, "f64": torch.float64, "s32": torch.int32}


def _input(a, block):
    """The framework's raster of a 2D GPU tensor, resident in HBM."""
    h, w = a.shape
    n0, n1 = -(-w // block), -(-h // block)
    if n0 * block != w or n1 * block != h:
        a = torch.nn.functional.pad(a, (0, n0 * block - w, 0, n1 * block - h))
    t = a.reshape(n1, block, n0, block).permute(0, 2, 1, 3).contiguous().cpu()
    r = M.Raster(M._lib.ma_input(ct.c_void_p(t.data_ptr()), ct.c_size_t(t.numel() * t.element_size()), M.Array([w, h]),
                                 _CODE[t.dtype], M.Array([block, block])))
    M.eval(r)
    return r


class _Result:
    """A pinned host buffer for one raster result (block-tiled), and its valid cells as views: the whole
    blocks, and the edge blocks of a ragged raster without their padding."""

    def __init__(self, w, h, block, dtype):
        n0, n1 = -(-w // block), -(-h // block)
        self.buf = torch.empty((n1, n0, block, block), dtype=dtype, pin_memory=True)
        self.nbytes = ct.c_size_t(self.buf.numel() * self.buf.element_size())
        self.ptr = ct.c_void_p(self.buf.data_ptr())
        e0, e1, f0, f1 = w - (n0 - 1) * block, h - (n1 - 1) * block, w // block, h // block
        b = self.buf
        v = [b[:f1, :f0], b[:f1, f0:, :, :e0], b[f1:, :f0, :e1], b[f1:, f0:, :e1, :e0]]
        self.views = [x for x in v if x.numel()]

    def fetch(self, raster):
        if M._lib.ma_fetch(raster, self.ptr, self.nbytes) != 0:
            raise RuntimeError(M._lib.ma_lastError().decode())
        return self.views


def _split(a, block):
    """A 2D tensor as the views of _Result lay it out."""
    h, w = a.shape
    n0, n1 = -(-w // block), -(-h // block)
    p = torch.nn.functional.pad(a, (0, n0 * block - w, 0, n1 * block - h))
    b = p.reshape(n1, block, n0, block).permute(0, 2, 1, 3)
    e0, e1, f0, f1 = w - (n0 - 1) * block, h - (n1 - 1) * block, w // block, h // block
    return [x for x in (b[:f1, :f0], b[:f1, f0:, :, :e0], b[f1:, :f0, :e1], b[f1:, f0:, :e1, :e0]) if x.numel()]


def _options(case):
    """The options a program with this workload sets (the rest stays at its default)."""
    M.set_option("graph", 1 if case.get("graph") else 0)
    M.set_option("focal_zonal", 1 if case["kind"] in ("hillshade_zonal", "tiles") else 0)


REQUESTS = ("hillshade", "slope_aspect", "mean7", "hillshade", "slope_aspect", "zstats", "hillshade", "mean7",
            "slope_aspect", "hillshade")  # 4 : 3 : 2 : 1


def _sides(seed, n, lo, hi):
    r = np.random.Generator(np.random.PCG64([seed, 11]))
    return [tuple(int(round(math.exp(r.uniform(math.log(lo), math.log(hi))))) for _ in range(2)) for _ in range(n)]


def _tile_inputs(case, seed):
    """(DEM, zones, 5x5 weights) of every tile."""
    for i, (w, h) in enumerate(_sides(case["tiles"], case["tiles"], case["lo"], case["hi"])):
        w, h = _fit(w, case["block"]), _fit(h, case["block"])
        r = np.random.Generator(np.random.PCG64([seed, i]))
        wts = (r.integers(-64, 65, (5, 5)) / 64.0).tolist()
        yield _dem(seed * 4099 + i, w, h), _zones(seed * 4099 + i, w, h, case["zones"], torch.uint8), wts


def _request_inputs(case, seed):
    """(kind, DEM, zones) of every request."""
    for i, (w, h) in enumerate(_sides(case["requests"] + 77, case["requests"], case["lo"], case["hi"])):
        w, h = _fit(w, case["block"]), _fit(h, case["block"])
        kind = REQUESTS[i]
        yield kind, _dem(seed * 4099 + i, w, h), _zones(seed * 4099 + i, w, h, 64, torch.int32) if kind == "zstats" else None


def _observer(case):
    return [min(case["w"] - 1, int(case["ox"] * case["w"])), min(case["h"] - 1, int(case["oy"] * case["h"]))]


OBSERVER_HEIGHT = 0.01  # above the ground, in the units of the normalised DEM
HIDDEN = 1e-4  # a cell this little below the line of sight counts as visible
STREAM = 1000  # accumulated rain that makes a stream


def _norm(seed, w, h):
    z = _dem(seed, w, h)
    return (z - z.min()) / (z.max() - z.min())


def _eye(norm, obs):
    """Height of the observer's eye in the normalised DEM (an F32 value)."""
    return float(np.float32(float(norm[obs[1], obs[0]]) + OBSERVER_HEIGHT))


def _life(case, seed):
    return (torch.rand(case["h"], case["w"], generator=_gen(seed, 3), device=_device()) < 0.3).to(torch.uint8)


def _layer(case, seed, k):
    """One layer of an overlay: a suitability score in [0, 100), smooth with some noise."""
    z = _norm(seed * 7 + k, case["w"], case["h"]) * 100.0
    return z.to(_TORCH[case["dtype"]])


def _rain(case, seed):
    r = torch.rand(case["h"], case["w"], generator=_gen(seed, 4), device=_device())
    return (r * 2).to(_TORCH[case["dtype"]]) if case["dtype"] != "s32" else (r * 3).to(torch.int32)


def prepare(case, seed):
    _device()
    _options(case)
    k = case["kind"]
    s = {"case": case}
    if k == "tiles":
        keep = [(_input(d, case["block"]), _input(z, case["block"]), wts) for d, z, wts in _tile_inputs(case, seed)]
        s["in"] = keep
        s["out"] = [W.batch_tile_sums(M, d, z, wts, case["zones"]) for d, z, wts in keep]
    elif k == "served":
        s["in"] = []
        for kind, d, z in _request_inputs(case, seed):
            h, w = d.shape
            n = {"hillshade": 1, "mean7": 1, "slope_aspect": 2, "zstats": 0}[kind]
            s["in"].append((kind, _input(d, case["block"]), None if z is None else _input(z, case["block"]),
                            [_Result(w, h, case["block"], torch.float32) for _ in range(n)]))
    else:
        w, h, block = case["w"], case["h"], case["block"]
        if k == "life":
            s["in"] = _input(_life(case, seed), block)
            s["out"] = W.life(M, s["in"], case["gens"])
            s["host"] = _Result(w, h, block, torch.uint8)
        elif k == "hillshade":
            s["in"] = _input(_dem(seed, w, h), block)
            s["out"] = W.hillshade(M, s["in"])
            s["host"] = _Result(w, h, block, torch.float32)
        elif k == "hillshade_zonal":
            s["in"] = _input(_dem(seed, w, h), block), _input(_zones(seed, w, h, case["zones"], torch.int32), block)
            s["out"] = W.hillshade_zonal(M, *s["in"], case["zones"])
        elif k == "overlay":
            s["in"] = [_input(_layer(case, seed, i), block) for i in range(4)]
            s["zones"] = _input(_zones(seed, w, h, case["zones"], torch.int32), block)
            score = W.wsum(M, *s["in"])
            s["out"] = M.zstats(score if case["dtype"] != "f64" else M.astype(score, M.F32), s["zones"], case["zones"])
        elif k == "viewshed":
            a, obs = _norm(seed, w, h), _observer(case)
            eye = _eye(a, obs)
            s["in"] = norm = _input(a, block)
            dx, dy = obs[0] - M.index(norm, M.D1), obs[1] - M.index(norm, M.D2)
            s["dist"] = dist = M.sqrt(dx * dx + dy * dy + 0.0)
            M.eval(dist)
            view = (M.rmax((norm - eye) / dist, obs) * dist + eye) - norm
            s["out"] = M.astype(view < HIDDEN, M.U8) if case["mask"] else view
            s["host"] = _Result(w, h, block, torch.uint8 if case["mask"] else torch.float32)
            del dx, dy
        elif k == "flow":
            s["in"] = _input(_rain(case, seed), block), _input(_d8(_dem(seed, w, h)), block)
            acc = M.flow_accumulation(*s["in"])
            s["out"] = M.astype(acc > STREAM, M.U8) if case["mask"] else acc
            s["host"] = _Result(w, h, block, torch.uint8 if case["mask"] else _TORCH[case["dtype"]])
    return s


def _table(z):
    t = z.table()
    return {k: t[k] for k in ("sum", "min", "max", "count")}


def run(s):
    k = s["case"]["kind"]
    if k == "served":
        server = M.Server(max_inflight=64)
        ids, left = {}, 0
        for i, (kind, dem, zones, _) in enumerate(s["in"]):
            ids[server.submit(*W.serve_request(M, kind, dem, zones))] = i
            left += 1
        got = [None] * left
        while left:
            for rid, *_ in server.step(2000):
                got[ids[rid]] = server.result(rid)
                left -= 1
        out = []
        for targets, (kind, _, _, host) in zip(got, s["in"]):
            out.append(_table(targets[0]) if kind == "zstats" else [r.fetch(t) for r, t in zip(host, targets)])
            for t in targets:
                M.release(t)
        server.close()
        return out
    if k == "tiles":
        M.eval(*s["out"])
        t = [_table(z) for z in s["out"]]
        return {f: np.stack([x[f] for x in t]) for f in t[0]}
    if k in ("hillshade_zonal", "overlay"):
        M.eval(s["out"])
        return _table(s["out"])
    M.eval(s["out"])
    got = s["host"].fetch(s["out"])
    M.release(s["out"])
    return got


def work(case):
    """Bytes: every input raster read once and every result written once. Operations: those of the script."""
    k = case["kind"]
    if k == "tiles":
        cells = sum(w * h for w, h in _sides(case["tiles"], case["tiles"], case["lo"], case["hi"]))
        return {"bytes": 5.0 * cells, "flops": 100.0 * cells}
    if k == "served":
        per = {"hillshade": (8, 120), "slope_aspect": (12, 110), "mean7": (8, 98), "zstats": (8, 4)}
        b = f = 0.0
        for (w, h), kind in zip(_sides(case["requests"] + 77, case["requests"], case["lo"], case["hi"]), REQUESTS):
            b += per[kind][0] * float(w * h)
            f += per[kind][1] * float(w * h)
        return {"bytes": b, "flops": f}
    cells = float(case["w"]) * case["h"]
    if k == "life":
        return {"bytes": 2 * cells, "flops": 12 * cells * case["gens"]}
    if k == "hillshade":
        return {"bytes": 8 * cells, "flops": 120 * cells}
    if k == "hillshade_zonal":
        return {"bytes": 8 * cells, "flops": 124 * cells}
    size = {"f32": 4, "s32": 4, "f64": 8}.get(case.get("dtype"), 4)
    if k == "overlay":
        return {"bytes": (4 * size + 4) * cells, "flops": 13 * cells}
    if k == "viewshed":  # the normalised DEM and the distances read, the result written
        return {"bytes": (8 + (1 if case["mask"] else 4)) * cells, "flops": 15 * cells}
    return {"bytes": (size + 1 + (1 if case["mask"] else size)) * cells, "flops": 2 * cells}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------


def _axis(n, block, d):
    """Along one axis, for the neighbour at offset d of every cell: its coordinate inside the raster, whether
    it lies in the cell's own block or an existing neighbour block, and the coordinate mirrored in the own block."""
    x = torch.arange(n, device=_device())
    b = x // block
    ext = torch.clamp(n - b * block, max=block)
    lx = x - b * block + d
    ok = (x + d >= 0) & (x + d < n)
    inv = torch.where(lx < 0, -lx - 1, torch.where(lx >= ext, ext - (lx - ext + 1), lx))
    return torch.clamp(x + d, 0, n - 1), ok, b * block + inv


def _window(a, block, dx, dy):
    """The neighbour at (dx, dy) of every cell under the framework's border rule: outside the raster both
    coordinates mirror inside the cell's own block."""
    x, okx, ix = _axis(a.shape[1], block, dx)
    y, oky, iy = _axis(a.shape[0], block, dy)
    plain = a.index_select(0, y).index_select(1, x)
    if bool(okx.all()) and bool(oky.all()):
        return plain
    return torch.where(oky[:, None] & okx[None], plain, a.index_select(0, iy).index_select(1, ix))


@contextlib.contextmanager
def _f64():
    """Python scalars beside comparisons take part in 64 bits."""
    torch.set_default_dtype(torch.float64)
    try:
        yield
    finally:
        torch.set_default_dtype(torch.float32)


class _T:
    """The map-algebra calls of the workload scripts over 64-bit tensors."""

    def __init__(self, block):
        self.block = block

    def convolve(self, r, mask):
        n1, n0 = len(mask) // 2, len(mask[0]) // 2
        acc = None
        for y, row in enumerate(mask):
            for x, v in enumerate(row):
                if v:
                    t = _window(r, self.block, x - n0, y - n1) * float(v)
                    acc = t if acc is None else acc.add_(t)
        return acc

    def _f(name):
        def f(self, *a):
            if isinstance(a[0], torch.Tensor):
                return getattr(torch, name)(*a)
            return float(np.float32(getattr(math, name)(*a)))
        return f
    sin, cos, atan, atan2, sqrt = _f("sin"), _f("cos"), _f("atan"), _f("atan2"), _f("sqrt")

    def zstats(self, v, zones, nz):
        z = zones.reshape(-1).long()
        v = v.reshape(-1).double()
        new = lambda x: torch.full((nz,), x, dtype=torch.float64, device=v.device)  # noqa: E731
        return {"sum": new(0.0).index_add_(0, z, v), "min": new(math.inf).scatter_reduce_(0, z, v, "amin"),
                "max": new(-math.inf).scatter_reduce_(0, z, v, "amax"), "count": None}


def _exact_view(case, seed):
    """The viewshed recurrence of every octant in 64 bits, a column at a time."""
    norm, (ox, oy) = _norm(seed, case["w"], case["h"]), _observer(case)
    eye = _eye(norm, (ox, oy))
    norm = norm.double()
    h, w = norm.shape
    x = torch.arange(w, device=norm.device, dtype=torch.float64) - ox
    y = torch.arange(h, device=norm.device, dtype=torch.float64) - oy
    dist = torch.sqrt(x[None] ** 2 + y[:, None] ** 2)
    ang = (norm - eye) / dist
    out = torch.full_like(ang, -math.inf)
    if math.isfinite(float(ang[oy, ox])):
        out[oy, ox] = ang[oy, ox]
    for fx, fy, sx, sy in ((0, -1, 1, 0), (1, 0, 0, -1), (1, 0, 0, 1), (0, 1, 1, 0), (0, 1, -1, 0), (-1, 0, 0, 1), (-1, 0, 0, -1),
                           (0, -1, -1, 0)):
        far = lambda ux, uy: (w - 1 - ox if ux > 0 else ox) if ux else (h - 1 - oy if uy > 0 else oy)  # noqa: E731
        l0, l1 = far(fx, fy), far(sx, sy)
        prev = out[oy, ox].reshape(1)
        for c in range(1, l0 + 1):
            n = min(c, l1) + 1
            r = torch.arange(n, device=norm.device, dtype=torch.float64)
            ri = torch.arange(n, device=norm.device)
            a = torch.cat([prev, prev[-1:]])[:n]  # row r of the previous column (unused on the diagonal)
            b = torch.cat([prev[:1], prev])[:n]   # row r - 1 of it
            wt = r / c * (c - 1) - (r - 1)
            base = a * wt + b * (1 - wt)
            base = torch.where(ri == 0, a, torch.where(ri == c, b, base))
            iy, ix = oy + fy * c + sy * ri, ox + fx * c + sx * ri
            v = ang[iy, ix]
            prev = torch.where(torch.isfinite(v), torch.maximum(base, v), base)
            out[iy, ix] = prev
    return (out * dist + eye) - norm


def _exact_flow(case, seed):
    """Rain accumulated downstream in 64 bits, a layer of finished cells at a time."""
    d = _device()
    z = _dem(seed, case["w"], case["h"])
    code = _d8(z)
    h, w = z.shape
    n = h * w
    to = torch.full((n,), n, dtype=torch.int64, device=d)
    at = torch.arange(n, device=d)
    for (dx, dy), c in W.D8_CODES:
        m = code.reshape(-1) == c
        to[m] = at[m] + dy * w + dx
    tot = torch.cat([_rain(case, seed).double().reshape(-1), torch.zeros(1, dtype=torch.float64, device=d)])
    left = torch.bincount(to, minlength=n + 1)
    go = torch.nonzero(left[:n] == 0).reshape(-1)
    while go.numel():
        t = to[go]
        tot.index_add_(0, t, tot[go])
        left.index_add_(0, t, torch.full_like(t, -1))
        t = torch.unique(t)
        go = t[(left[t] == 0) & (t < n)]
    return torch.where(to < n, tot[:n], torch.zeros((), dtype=torch.float64, device=d)).reshape(h, w)


def exact(case, seed):
    k = case["kind"]
    if k == "life" or (k in ("flow", "viewshed") and case["mask"]):
        return None  # whole numbers
    if k == "tiles":
        T, got = _T(case["block"]), []
        for d, z, wts in _tile_inputs(case, seed):
            with _f64():
                got.append(W.batch_tile_sums(T, d.double(), z, wts, case["zones"]))
        return {f: None if f == "count" else torch.stack([x[f] for x in got]) for f in got[0]}
    if k == "served":
        T, out = _T(case["block"]), []
        for kind, d, z in _request_inputs(case, seed):
            with _f64():
                r = W.serve_request(T, kind, d.double(), z)
            out.append(r[0] if kind == "zstats" else [_split(x, case["block"]) for x in r])
        return out
    T = _T(case["block"])
    if k == "hillshade":
        d = _dem(seed, case["w"], case["h"]).double()
        with _f64():
            return _split(W.hillshade(T, d), case["block"])
    if k == "hillshade_zonal":
        w, h = case["w"], case["h"]
        d, z = _dem(seed, w, h).double(), _zones(seed, w, h, case["zones"], torch.int32)
        with _f64():
            return W.hillshade_zonal(T, d, z, case["zones"])
    if k == "overlay":
        c = [float(np.float32(v)) for v in (0.1, 0.2, 0.3, 0.4)]
        r = [_layer(case, seed, i).double() for i in range(4)]
        v = c[0] * r[0] + r[1] * c[1] + c[2] * r[2] + r[3] * c[3]
        return T.zstats(v, _zones(seed, case["w"], case["h"], case["zones"], torch.int32), case["zones"])
    if k == "viewshed":
        return _split(_exact_view(case, seed), case["block"])
    if case["dtype"] == "s32" or case["w"] * case["h"] > 4e6:
        return None
    return _split(_exact_flow(case, seed), case["block"])
