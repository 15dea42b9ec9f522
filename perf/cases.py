"""Workloads of the dexel morphology library, as a program that uses it runs them.

Each case is one call through a public entry point: an operation on a volume
kept in HBM (`Context.morph_device`), an operation on a host volume
(`VoronoiMorphoHip.apply`), a batch of uneven resident volumes
(`Context.morph_batch_device`), each kept with `Context.copy_device`, or a
mesh turned into dexels (`Context.rasterize`).  The inputs are

* ``poisson``: direct dexel columns of Poisson(lam) segments with exponential
  (mean 40 dexel) gaps and lengths, clipped to [0, 1024];
* ``balls``: the union of random solid balls (smooth surfaces, few segments
  per column, empty columns around them);
* ``tubes``: thin random tubes, rasterized from a triangle mesh (filigree).

``listed()`` gives the cases, ``draw(rng)`` one more of the same ranges,
``prepare`` / ``run`` one pass, ``work`` the bytes a pass cannot do without,
``exact`` the result in 64 bits by direct evaluation of the definition.
"""

import functools
import math

import numpy as np
import torch

from voroffset_amd import _native, mesh
from voroffset_amd.morpho import VoronoiMorphoHip
from voroffset_amd.volume import CompressedVolume

ZMAX = 1024.0    # z-extent of the Poisson columns
MEAN = 40.0      # mean gap and segment length
MARGIN = 80.0    # empty z-range below and above (erosions and closings need the radius plus one)
OPS = ("dilation", "erosion", "closing", "opening")


def listed():
    return [
        # a small part held on the device: launches and latency count
        {"name": "resident_64x48_r4", "kind": "resident", "input": "poisson", "nx": 64, "ny": 48, "lam": 6.0,
         "op": "dilation", "r": 4.0, "precision": "fp32"},
        # a host volume of the command line tool's size: 128 dexels and 8 of padding around them, FP64
        {"name": "host_balls_144_r4_fp64", "kind": "host", "input": "balls", "nx": 144, "ny": 144, "balls": 32,
         "op": "dilation", "r": 4.0, "precision": "fp64"},
        # filigree: 2000 tubes in a 512 box with padding 16, the gaps between them closed
        {"name": "tubes_544_close_r5", "kind": "resident", "input": "tubes", "box": 512, "tubes": 2000,
         "op": "closing", "r": 5.0, "precision": "fp32"},
        # the same filigree thickened, endpoints in FP64
        {"name": "tubes_544_r10_fp64", "kind": "resident", "input": "tubes", "box": 512, "tubes": 2000,
         "op": "dilation", "r": 10.0, "precision": "fp64"},
        # solids shrunk: long smooth segments, complements on a grown grid
        {"name": "balls_512_erode_r8", "kind": "resident", "input": "balls", "nx": 512, "ny": 512, "balls": 96,
         "op": "erosion", "r": 8.0, "precision": "fp32"},
        # the throughput workload
        {"name": "poisson_1024_r16", "kind": "resident", "input": "poisson", "nx": 1024, "ny": 1024, "lam": 6.0,
         "op": "dilation", "r": 16.0, "precision": "fp32"},
        # ... with FP64 endpoints
        {"name": "poisson_1024_r16_fp64", "kind": "resident", "input": "poisson", "nx": 1024, "ny": 1024, "lam": 6.0,
         "op": "dilation", "r": 16.0, "precision": "fp64"},
        # ... with a large radius
        {"name": "poisson_1024_r64", "kind": "resident", "input": "poisson", "nx": 1024, "ny": 1024, "lam": 6.0,
         "op": "dilation", "r": 64.0, "precision": "fp32"},
        # a ragged grid, sparse columns, a radius between whole dexels
        {"name": "ragged_1531x219_r7.3", "kind": "resident", "input": "poisson", "nx": 1531, "ny": 219, "lam": 2.5,
         "op": "dilation", "r": 7.3, "precision": "fp32"},
        # the largest request a server of resident volumes gets: two dilations and two complements
        {"name": "poisson_1896_close_r48", "kind": "resident", "input": "poisson", "nx": 1896, "ny": 1896, "lam": 8.0,
         "op": "closing", "r": 48.0, "precision": "fp32"},
        # many uneven volumes, radii and operations in one call
        {"name": "batch_24", "kind": "batch", "volumes": 24, "side_lo": 64, "side_hi": 512, "r_lo": 2.0, "r_hi": 32.0,
         "precision": "fp32"},
        # a mesh becoming a dexel volume (host arrays in and out)
        {"name": "rasterize_544", "kind": "raster", "box": 512, "tubes": 2000},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("resident",) * 7 + ("host", "batch", "raster"))
    precision = "fp32" if rng.random() < 0.7 else "fp64"
    if kind == "raster":
        box = int(_log(rng, 100, 640))
        return {"kind": kind, "box": box, "tubes": max(8, int(box * box * rng.uniform(0.003, 0.01)))}
    if kind == "batch":
        return {"kind": kind, "volumes": rng.randint(3, 30), "side_lo": 48, "side_hi": int(_log(rng, 100, 500)),
                "r_lo": 2.0, "r_hi": round(_log(rng, 4, 40), 1), "precision": precision}
    source = rng.choice(("poisson", "poisson", "balls", "tubes"))
    c = {"kind": kind, "input": source, "op": rng.choice(OPS), "precision": precision}
    most = 500 if kind == "host" else 1300
    if source != "balls" and c["op"] in ("erosion", "opening"):  # thin features erode to nothing: grow or fill them
        c["op"] = rng.choice(("dilation", "closing"))
    if source == "tubes":
        c["box"] = int(_log(rng, 100, min(most, 640)))
        c["tubes"] = max(8, int(c["box"] ** 2 * rng.uniform(0.003, 0.01)))
        c["r"] = round(_log(rng, 2, 24), 1)
        return c
    c["nx"], c["ny"] = int(_log(rng, 40, most)), int(_log(rng, 40, most))
    if source == "poisson":
        c["lam"] = round(rng.uniform(2, 10), 2)
    else:
        c["balls"] = rng.randint(16, 160)
        if c["op"] in ("erosion", "opening"):  # some of the solid has to stay
            c["nx"], c["ny"] = max(c["nx"], 100), max(c["ny"], 100)
            most = 0.08 * min(c["nx"], c["ny"])
    r = _log(rng, 2, min(64, most))
    c["r"] = round(r, 1) if rng.random() < 0.5 else float(round(r))
    return c


# -- inputs -------------------------------------------------------------------

def _poisson(nx, ny, lam, seed):
    """(offsets, endpoints) on the GPU, float64."""
    g = torch.Generator("cuda").manual_seed(seed)
    n = nx * ny
    k = torch.poisson(torch.full((n,), float(lam), device="cuda"), generator=g)
    most = int(k.max()) if n else 0
    z = torch.zeros(n, dtype=torch.float64, device="cuda")
    lo, hi, keep = [], [], []
    for i in range(most):
        u = torch.rand(2, n, dtype=torch.float64, device="cuda", generator=g)
        step = -MEAN * torch.log1p(-u)
        start = z + step[0]
        z = start + step[1]
        lo.append(start)
        hi.append(torch.clamp(z, max=ZMAX))
        keep.append((k > i) & (start < ZMAX))
    return _pack(torch.stack(lo, 1), torch.stack(hi, 1), torch.stack(keep, 1))


def _pack(lo, hi, keep):
    off = torch.zeros(lo.shape[0] + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(2 * keep.sum(1), 0, out=off[1:])
    return off, torch.stack((lo[keep], hi[keep]), 1).reshape(-1).contiguous()


def _merge(lo, hi):
    """Rows of intervals (empty ones at +inf, -inf) into (lo, hi, keep): each
    row's union, an interval at the place of its last piece."""
    lo, order = torch.sort(lo, 1)
    hi = torch.cummax(torch.gather(hi, 1, order), 1).values
    after = torch.cat((lo[:, 1:], torch.full_like(lo[:, :1], math.inf)), 1)
    before = torch.cat((torch.full_like(hi[:, :1], -math.inf), hi[:, :-1]), 1)
    starts = (lo > before) & (lo < math.inf)
    ends = (after > hi) & (lo < math.inf)
    place = torch.arange(lo.shape[1], device=lo.device).expand_as(lo)
    first = torch.cummax(torch.where(starts, place, torch.zeros_like(place)), 1).values
    return torch.gather(lo, 1, first), hi, ends


def _balls(nx, ny, count, seed):
    """The union of `count` balls in an nx x ny grid of z-extent ZMAX / 2."""
    rng = np.random.default_rng(seed)
    side = float(min(nx, ny))
    r = rng.uniform(0.04, 0.14, count) * side
    c = torch.tensor(np.stack((rng.uniform(0, nx, count), rng.uniform(0, ny, count),
                               rng.uniform(0.15, 0.85, count) * ZMAX / 2, r)), device="cuda")
    offs, zs, base = [torch.zeros(1, dtype=torch.int64, device="cuda")], [], 0
    rows = max(1, (1 << 24) // max(1, nx * count))
    for y0 in range(0, ny, rows):
        y = torch.arange(y0, min(ny, y0 + rows), dtype=torch.float64, device="cuda") + 0.5
        x = torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5
        q = (c[3] ** 2 - (x[None, :, None] - c[0]) ** 2 - (y[:, None, None] - c[1]) ** 2).reshape(-1, count)
        h = torch.sqrt(q.clamp(min=0))
        lo = torch.where(q > 0, (c[2] - h).clamp(min=0), math.inf)
        hi = torch.where(q > 0, (c[2] + h).clamp(max=ZMAX / 2), -math.inf)
        off, z = _pack(*_merge(lo, hi))
        offs.append(off[1:] + base)
        base += z.numel()
        zs.append(z)
    return torch.cat(offs), torch.cat(zs)


@functools.lru_cache(None)
def _context():
    """The context a program creates once and keeps."""
    return _native.Context(0)


@functools.lru_cache(None)
def _method(precision):
    return VoronoiMorphoHip(precision, device=0)


def _tube_mesh(case, seed):
    return mesh.prism_tubes(case["tubes"], box=float(case["box"]), seed=seed)


def _tube_grid(case):
    """Columns per side and padding of the grid around the tubes' box."""
    pad = max(16, int(case.get("r", 0)) + 2)
    return case["box"] + 2 * pad, pad


def _volume(case, seed):
    """(nx, ny, offsets, endpoints, z_lo, z_hi) of a case's input, absolute z, float64 on the GPU."""
    if case["input"] == "tubes":
        n, pad = _tube_grid(case)
        m = _tube_mesh(case, seed)
        off, z = _context().rasterize(m.vertices, m.triangles, n, n, -float(pad), -float(pad), 1.0)
        return n, n, torch.from_numpy(off).cuda(), torch.from_numpy(z).cuda(), -float(pad), float(n - pad)
    nx, ny = case["nx"], case["ny"]
    if case["input"] == "balls":
        return (nx, ny, *_balls(nx, ny, case["balls"], seed), -MARGIN, ZMAX / 2 + MARGIN)
    return (nx, ny, *_poisson(nx, ny, case["lam"], seed), -MARGIN, ZMAX + MARGIN)


def _resident(vol, precision):
    """The volume as the device entry points take it: endpoints of the storage type, relative to the shift."""
    nx, ny, off, z, zlo, zhi = vol
    shift = _native.storage_shift(zlo, zhi) if precision == "fp32" else 0.0
    z = (z - shift).to(torch.float32 if precision == "fp32" else torch.float64)
    return nx, ny, off, z, zlo - shift, zhi - shift


def _jobs(case):
    """(side, lam, op, radius) of a batch's volumes: sides spread over their logarithm, densities and radii evenly."""
    n, jobs = case["volumes"], []
    for k in range(n):
        t, u, v = (k + 0.5) / n, (k * 0.618034 + 0.31) % 1, (k * 0.754878 + 0.57) % 1
        side = case["side_lo"] * (case["side_hi"] / case["side_lo"]) ** t
        jobs.append((int(round(side)), 2 + 8 * u, OPS[k % 4], case["r_lo"] + (case["r_hi"] - case["r_lo"]) * v))
    return jobs


def _batch(case, seed):
    return [(op, r, _resident(_volume({"input": "poisson", "nx": side, "ny": side, "lam": lam}, seed + 7919 * k + 1),
                              case["precision"])) for k, (side, lam, op, r) in enumerate(_jobs(case))]


def _room(columns, source, lam=0.0):
    """Endpoints the buffer for a result holds, as a program reserves them before it knows the result."""
    return int(columns * {"poisson": 2 * lam + 4, "balls": 8, "tubes": 24}[source]) + 4096


def _results(columns, precision, source, lam=0.0):
    """Buffers of the program's own for one result (the library's live until its next call)."""
    return {"off": torch.zeros(columns + 1, dtype=torch.int64, device="cuda"),
            "z": torch.zeros(_room(columns, source, lam), dtype=torch.float32 if precision == "fp32" else torch.float64,
                             device="cuda")}


def prepare(case, seed):
    if case["kind"] == "raster":
        n, pad = _tube_grid(case)
        m = _tube_mesh(case, seed)
        return {"kind": "raster", "ctx": _context(), "z": np.zeros(_room(n * n, "tubes")),
                "call": (m.vertices, m.triangles, n, n, -float(pad), -float(pad), 1.0)}
    if case["kind"] == "batch":
        jobs = _batch(case, seed)
        return {"kind": "batch", "ctx": _context(), "precision": case["precision"], "keep": jobs,
                "out": [_results(side * side, case["precision"], "poisson", lam) for side, lam, _, _ in _jobs(case)],
                "jobs": [(op, r, nx, ny, off.data_ptr(), z.data_ptr(), zlo, zhi)
                         for op, r, (nx, ny, off, z, zlo, zhi) in jobs]}
    vol = _volume(case, seed)
    if case["kind"] == "host":
        nx, ny, off, z, zlo, zhi = vol
        host = CompressedVolume(nx, ny, off.cpu().numpy(), z.cpu().numpy(), origin=(0.0, 0.0, zlo),
                                extent=(float(nx), float(ny), zhi - zlo), spacing=1.0, padding=0)
        return {"kind": "host", "method": _method(case["precision"]), "volume": host, "op": case["op"], "r": case["r"],
                "z": np.zeros(_room(nx * ny, case["input"], case.get("lam", 0.0)))}
    nx, ny, off, z, zlo, zhi = _resident(vol, case["precision"])
    return {"kind": "resident", "ctx": _context(), "keep": (off, z),
            "out": _results(nx * ny, case["precision"], case["input"], case.get("lam", 0.0)),
            "call": (case["op"], case["precision"], case["r"], nx, ny, off.data_ptr(), z.data_ptr(), zlo, zhi)}


def _kept(ctx, pairs, size):
    """Results copied from the library's workspace into the program's buffers, with one wait."""
    copies = []
    for (out, count), own in pairs:
        if count > own["z"].numel():
            raise RuntimeError("a result of %d endpoints does not fit its buffer" % count)
        copies += [(own["off"].data_ptr(), out.offsets, 8 * own["off"].numel()), (own["z"].data_ptr(), out.z, size * count)]
    ctx.copy_device(copies)


def run(state):
    if state["kind"] == "resident":
        out, count, _ = state["ctx"].morph_device(*state["call"])
        _kept(state["ctx"], [((out, count), state["out"])], state["out"]["z"].element_size())
        return state["out"]
    if state["kind"] == "batch":
        outs, _ = state["ctx"].morph_batch_device(state["precision"], state["jobs"])
        _kept(state["ctx"], list(zip(outs, state["out"])), state["out"][0]["z"].element_size())
        return state["out"]
    if state["kind"] == "host":
        out, _, _ = state["method"].apply(state["op"], state["volume"], state["r"])
        off, z = out.off, out.z
    else:
        off, z = state["ctx"].rasterize(*state["call"])
    state["z"][:z.size] = z
    return {"off": off, "z": state["z"]}


# -- what a pass cannot do without ------------------------------------------------

def _volume_bytes(columns, endpoints, size):
    return 8 * (columns + 1) + size * endpoints


def work(case):
    """Offsets and endpoints of the input read once and of the output written
    once.  Segments per column are those of the input's distribution; a result
    is counted as one segment per column (what large radii leave)."""
    if case["kind"] == "raster":
        columns = _tube_grid(case)[0] ** 2
        return {"bytes": case["tubes"] * (16 * 24 + 28 * 12) + _volume_bytes(columns, 64 * case["tubes"], 8), "flops": 0}
    size = 4 if case["precision"] == "fp32" else 8
    if case["kind"] == "batch":
        return {"bytes": sum(_volume_bytes(side * side, 2 * lam * side * side, size) +
                             _volume_bytes(side * side, 2 * side * side, size) for side, lam, _, _ in _jobs(case)),
                "flops": 0}
    if case["input"] == "tubes":
        columns, endpoints = _tube_grid(case)[0] ** 2, 64 * case["tubes"]
    else:
        columns = case["nx"] * case["ny"]
        endpoints = 2 * columns * (case["lam"] if case["input"] == "poisson" else 0.5)
    if case["kind"] == "host":
        size = 8
    return {"bytes": _volume_bytes(columns, endpoints, size) + _volume_bytes(columns, 2 * columns, size), "flops": 0}


# -- the definition in 64 bits ------------------------------------------------------

def _rows(off, z):
    """CSR columns as padded rows (empty places at +inf, -inf)."""
    n = (off[1:] - off[:-1]) // 2
    most = max(1, int(n.max()))
    place = torch.arange(most, device=z.device)
    keep = place[None, :] < n[:, None]
    at = torch.where(keep, off[:-1, None] + 2 * place[None, :], torch.zeros_like(place)[None, :])
    if not z.numel():
        z = torch.zeros(2, dtype=torch.float64, device=off.device)
    return torch.where(keep, z[at], math.inf), torch.where(keep, z[at + 1], -math.inf)


def _dilate(nx, ny, off, z, r):
    """Union over the disk of radius r of the columns' segments grown by sqrt(r^2 - d^2)."""
    lo, hi = (v.reshape(ny, nx, -1) for v in _rows(off, z))
    k = int(math.floor(r))
    disk = [(dx, dy, math.sqrt(r * r - dx * dx - dy * dy)) for dy in range(-k, k + 1) for dx in range(-k, k + 1)
            if dx * dx + dy * dy <= r * r]
    S = lo.shape[2]
    if nx * ny * len(disk) * S > 4e8:
        return None
    grow = torch.nn.functional.pad
    lo, hi = grow(lo, (0, 0, k, k, k, k), value=math.inf), grow(hi, (0, 0, k, k, k, k), value=-math.inf)
    offs, zs, base = [torch.zeros(1, dtype=torch.int64, device="cuda")], [], 0
    rows = max(1, (1 << 25) // (nx * len(disk) * S))
    for y0 in range(0, ny, rows):
        m = min(rows, ny - y0)
        a = torch.cat([lo[y0 + k + dy:y0 + k + dy + m, k + dx:k + dx + nx] - h for dx, dy, h in disk], 2)
        b = torch.cat([hi[y0 + k + dy:y0 + k + dy + m, k + dx:k + dx + nx] + h for dx, dy, h in disk], 2)
        o, v = _pack(*_merge(a.reshape(m * nx, -1), b.reshape(m * nx, -1)))
        offs.append(o[1:] + base)
        base += v.numel()
        zs.append(v)
    return torch.cat(offs), torch.cat(zs)


def _complement(off, z, zlo, zhi):
    """Columns complemented within [zlo, zhi]."""
    lo, hi = _rows(off, z)
    a = torch.cat((torch.full_like(lo[:, :1], zlo), torch.where(hi > -math.inf, hi, math.inf)), 1)
    b = torch.cat((lo, torch.full_like(lo[:, :1], math.inf)), 1).clamp(max=zhi)
    a = a.clamp(min=zlo)
    return _pack(a, b, b > a)


def _erode(nx, ny, off, z, r, zlo, zhi):
    """Complement within [zlo - 1, zhi + 1] on a grid with a ring of full columns, dilated, cropped and complemented."""
    o, v = _complement(off, z, zlo - 1, zhi + 1)
    lo, hi = (t.reshape(ny, nx, -1) for t in _rows(o, v))
    full = torch.nn.functional.pad
    lo, hi = full(lo, (0, 0, 1, 1, 1, 1), value=math.inf), full(hi, (0, 0, 1, 1, 1, 1), value=-math.inf)
    ring = torch.ones(ny + 2, nx + 2, dtype=torch.bool, device="cuda")
    ring[1:-1, 1:-1] = False
    lo[..., 0] = torch.where(ring, zlo - 1, lo[..., 0])
    hi[..., 0] = torch.where(ring, zhi + 1, hi[..., 0])
    lo, hi = lo.reshape((nx + 2) * (ny + 2), -1), hi.reshape((nx + 2) * (ny + 2), -1)
    grown = _dilate(nx + 2, ny + 2, *_pack(lo, hi, hi >= lo), r)
    if grown is None:
        return None
    lo, hi = (t.reshape(ny + 2, nx + 2, -1)[1:-1, 1:-1].reshape(nx * ny, -1) for t in _rows(*grown))
    return _complement(*_pack(lo, hi, hi >= lo), zlo, zhi)


def _exact(op, r, vol, room):
    nx, ny, off, z, zlo, zhi = vol
    v = (off, z.to(torch.float64))
    for step in {"dilation": "d", "erosion": "e", "closing": "de", "opening": "ed"}[op]:
        v = _dilate(nx, ny, *v, r) if step == "d" else _erode(nx, ny, *v, r, zlo, zhi)
        if v is None:
            return None
    z = torch.zeros(room, dtype=torch.float64, device="cuda")
    z[:v[1].numel()] = v[1]
    return {"off": None, "z": z}


def exact(case, seed):
    if case["kind"] in ("raster", "batch") or case["input"] == "tubes":
        return None  # (their inputs are made by the library itself, or would take too long)
    vol = _volume(case, seed)
    room = _room(case["nx"] * case["ny"], case["input"], case.get("lam", 0.0))
    if case["kind"] == "host":
        if case["precision"] == "fp32":
            shift = _native.storage_shift(vol[4], vol[5])
            vol = (*vol[:3], (vol[3] - shift).to(torch.float32).to(torch.float64) + shift, *vol[4:])
        return _exact(case["op"], case["r"], vol, room)
    return _exact(case["op"], case["r"], _resident(vol, case["precision"]), room)
