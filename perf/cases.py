"""Workloads of the OWM ground-seed pipeline, as a user's program runs them
through fastowm_amd's Python interface.

A program keeps one Context (and, when it serves, one Server) for all of its
clouds, so every state here shares them; each state is another cloud.  The
clouds follow the generator of fastowm_amd.synth (terrain of sinusoids, 40 %
vegetation with exponential heights, optional clusters and flat roofs with
1-cm heights), made on the GPU by torch.  Point order is either random (as that
generator's) or along scan lines (as an airborne scanner delivers a strip);
`cm` rounds the coordinates to centimetres, as LiDAR files hold them.

Every output is a list of point ids, or counts: whole numbers.  Their number
depends on the cloud, so a program keeps them in buffers of its own, sized for
the largest answer its clouds can give (NONE behind the last id).
"""
import math

import numpy as np
import torch

from fastowm_amd import owm, synth

DEV = "cuda:0"
_held = {}


def _context():
    if "ctx" not in _held:
        _held["ctx"] = owm.Context(0)
    return _held["ctx"]


def _server():
    # a serving process gives its loop a fixed share of the device memory
    if "server" not in _held:
        _held["serve_ctx"] = owm.Context(0, hbm_budget=64 << 30)
        _held["server"] = owm.Server(_held["serve_ctx"], max_inflight=2, max_batch=64)
    return _held["server"]


# ------------------------------------------------------------------ cases --

def _tile(name, n, density, wsize, overlap, bsize, scene="plain", order="random", cm=False,
          box=False, source="device"):
    return {"name": name, "kind": "tile", "n": n, "density": density, "wsize": wsize,
            "overlap": overlap, "bsize": bsize, "scene": scene, "order": order, "cm": cm,
            "box": box, "source": source}


def listed():
    return [
        # the smallest request a serving client or an interactive crop sends:
        # latency of one call
        _tile("tile_10k", 10_000, 8.0, 10, 0.8, 20),
        # a small tile of a host program (numpy arrays, the file header's box),
        # odd sizes, an odd window side and half overlap
        _tile("tile_host_300k", 299_977, 4.3, 7, 0.5, 13, box=True, source="host"),
        # the 500 m x 500 m tile of 1M points
        _tile("tile_1m", 1_000_000, 4.0, 12, 0.8, 20),
        # a dense strip in scan order with centimetre coordinates; its window
        # side is not a whole number of window steps
        _tile("tile_8m_scan_cm", 7_999_993, 15.0, 12, 0.7, 25, order="scan", cm=True),
        # the 2 km x 2 km tile of 20M points with clusters
        _tile("tile_20m_clusters", 20_000_000, 5.0, 12, 0.8, 20, scene="clusters"),
        # the urban 3 km x 3 km tile of 120M points with 1-cm roofs (exact ties)
        _tile("tile_120m_roofs", 120_000_000, 13.3, 12, 0.8, 20, scene="roofs"),
        # a survey: 512 uneven tiles in one batch (329M points)
        {"name": "batch_512", "kind": "batch", "mix": "survey", "tiles": 512, "cm": False},
        # a batch of requests whose window and cell sizes all differ
        {"name": "batch_96_mixed", "kind": "batch", "mix": "requests", "tiles": 96, "cm": True},
        # a serving burst: resident tiles submitted one by one, then awaited
        {"name": "serve_192", "kind": "serve", "mix": "survey", "tiles": 192, "cm": False},
        # the stage interface: a resident tree, its stages one by one, and a
        # second query of the same tree with other parameters
        {"name": "stages_3m", "kind": "stages", "n": 3_000_001, "density": 6.0, "wsize": 10,
         "overlap": 0.8, "bsize": 20, "scene": "plain", "order": "random", "cm": False,
         "wsize2": 15, "overlap2": 0.6, "bsize2": 25},
        # a headed .xyz file read from its bytes and run
        {"name": "reader_1m", "kind": "reader", "n": 1_000_003, "density": 5.0, "wsize": 12,
         "overlap": 0.8, "bsize": 20, "scene": "plain", "order": "scan", "cm": True},
        # the quadtree statistics of the 20M-point tile
        {"name": "stats_20m", "kind": "stats", "n": 20_000_000, "density": 5.0,
         "scene": "clusters", "order": "random", "cm": False, "policy": "maxnumber",
         "max_number": 32, "min_radius": 0.0, "level": 5},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def _overlap(rng):
    return rng.choice([0.5, 0.6, 0.75, 0.8, 0.8, 0.9, round(rng.uniform(0.5, 0.9), 2)])


def draw(rng):
    kind = rng.choice(["tile"] * 8 + ["large"] * 3 + ["batch"] * 4 + ["serve", "stages", "stages",
                                                                     "reader", "stats", "stats"])
    cloud = {"density": round(rng.uniform(1.0, 20.0), 2), "scene": rng.choice(["plain", "plain", "clusters", "roofs"]),
             "order": rng.choice(["random", "random", "scan"]), "cm": rng.random() < 0.4}
    query = {"wsize": rng.randint(5, 20), "overlap": _overlap(rng), "bsize": rng.randint(10, 30)}
    if kind == "tile":
        n = _log(rng, 10_000, 8_000_000)
        host = n <= 1_000_000 and rng.random() < 0.25
        return {"kind": "tile", "n": n, **cloud, **query, "box": rng.random() < 0.3,
                "source": "host" if host else "device"}
    if kind == "large":  # a survey in one tile
        cloud["density"] = round(rng.uniform(4.0, 16.0), 2)
        query.update(wsize=rng.randint(8, 16), overlap=rng.choice([0.5, 0.6, 0.75, 0.8, 0.8]))
        return {"kind": "tile", "n": _log(rng, 8_000_000, 120_000_000), **cloud, **query,
                "box": rng.random() < 0.3, "source": "device"}
    if kind == "batch":
        mix = rng.choice(["survey", "requests"])
        tiles = _log(rng, 4, 256) if mix == "survey" else _log(rng, 4, 96)
        return {"kind": "batch", "mix": mix, "tiles": tiles, "cm": rng.random() < 0.4}
    if kind == "serve":
        return {"kind": "serve", "mix": rng.choice(["survey", "requests"]),
                "tiles": _log(rng, 8, 96), "cm": rng.random() < 0.4}
    if kind == "stages":
        return {"kind": "stages", "n": _log(rng, 10_000, 8_000_000), **cloud, **query,
                "wsize2": rng.randint(5, 20), "overlap2": _overlap(rng), "bsize2": rng.randint(10, 30)}
    if kind == "reader":
        cloud["cm"] = True
        return {"kind": "reader", "n": _log(rng, 10_000, 1_000_000), **cloud, **query}
    by_radius = rng.random() < 0.4
    return {"kind": "stats", "n": _log(rng, 100_000, 20_000_000), **cloud,
            "policy": "minradius" if by_radius else "maxnumber", "max_number": rng.choice([16, 32, 64, 128]),
            "min_radius": rng.choice([0.5, 1.0, 2.0]) if by_radius else 0.0, "level": rng.randint(3, 6)}


# ----------------------------------------------------------------- clouds --

def _uniform(g, n):
    return torch.rand(n, dtype=torch.float64, device=DEV, generator=g)


def _terrain(x, y, side, g, which=None):
    """Sum of four sinusoids of 2-40 m wavelength, amplitude 3 m in all; `which`
    maps points to tiles (each with phases and wavelengths of its own)."""
    tiles = side.numel()
    z = torch.full_like(x, 300.0)
    for _ in range(4):
        k = 2.0 * math.pi / (2.0 + 38.0 * _uniform(g, tiles))
        a = 2.0 * math.pi * _uniform(g, tiles)
        p = 2.0 * math.pi * _uniform(g, tiles)
        kx, ky = k * torch.cos(a), k * torch.sin(a)
        if which is not None:
            kx, ky, p = kx[which], ky[which], p[which]
        z += 0.75 * torch.sin(x * kx + y * ky + p)
    return z


def _vegetation(z, g):
    n = z.numel()
    high = _uniform(g, n) < 0.4
    return z + torch.where(high, -6.0 * torch.log1p(-_uniform(g, n)), torch.zeros_like(z))


def _cloud(case, seed):
    """x, y, z of one tile (float64, on the GPU)."""
    n = case["n"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    side = math.sqrt(n / case["density"])
    x = _uniform(g, n) * side
    y = _uniform(g, n)
    if case["order"] == "scan":  # lines across the strip, one after another
        y = (torch.arange(n, dtype=torch.float64, device=DEV) + y) / n
    y *= side
    if case["scene"] == "clusters":  # a tenth of the points, sigma 3 m
        m = max(1, n // 20_000)
        cx, cy = _uniform(g, m) * side, _uniform(g, m) * side
        own = torch.randint(0, m, (n,), device=DEV, generator=g)
        at = _uniform(g, n) < 0.1
        dx = torch.randn(n, dtype=torch.float64, device=DEV, generator=g) * 3.0
        dy = torch.randn(n, dtype=torch.float64, device=DEV, generator=g) * 3.0
        x = torch.where(at, (cx[own] + dx).clamp_(0.0, side), x)
        y = torch.where(at, (cy[own] + dy).clamp_(0.0, side), y)
    z = _vegetation(_terrain(x, y, torch.tensor([side], dtype=torch.float64, device=DEV), g), g)
    if case["scene"] == "roofs":  # 30 m blocks, three in ten of them built over
        m = max(1, int(side / 30.0))
        cell = (x / side * m).long().clamp_(max=m - 1) * m + (y / side * m).long().clamp_(max=m - 1)
        built = _uniform(g, m * m) < 0.3
        height = torch.round((305.0 + 35.0 * _uniform(g, m * m)) * 100.0) / 100.0
        z = torch.where(built[cell], height[cell], z)
    x += 512_000.0
    y += 4_700_000.0
    if case["cm"]:
        x, y, z = (torch.round(a * 100.0) / 100.0 for a in (x, y, z))
    return x, y, z


def _mix(case):
    """The tiles of a batch: fastowm_amd.synth's uneven survey or request
    parameters (sizes, densities, windows)."""
    if case["mix"] == "survey":
        return synth.batch_tiles(case["tiles"], seed=0)
    return [t for _, t in synth.serve_requests(case["tiles"], 1000.0, seed=1)]


def _mix_cloud(tiles, cm, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    counts = torch.tensor([t.n for t in tiles], device=DEV)
    side = torch.tensor([t.width for t in tiles], dtype=torch.float64, device=DEV)
    which = torch.repeat_interleave(torch.arange(len(tiles), device=DEV), counts)
    n = which.numel()
    x = _uniform(g, n) * side[which]
    y = _uniform(g, n) * side[which]
    z = _vegetation(_terrain(x, y, side, g, which), g)
    x += torch.tensor([t.x0 for t in tiles], dtype=torch.float64, device=DEV)[which]
    y += torch.tensor([t.y0 for t in tiles], dtype=torch.float64, device=DEV)[which]
    if cm:
        x, y, z = (torch.round(a * 100.0) / 100.0 for a in (x, y, z))
    return x, y, z


# ------------------------------------------------------------ the passes --

def _query(case, key=""):
    return {k: case[k + key] for k in ("wsize", "overlap", "bsize")}


def _windows(n, density, wsize, overlap, bsize):
    """At most as many windows as a tile of these parameters has."""
    side = math.sqrt(n / density)
    return (int((side + 2 * wsize * overlap) / round(wsize * (1 - overlap), 2)) + 2) ** 2


def _ids(count):
    return np.full(count, owm.NONE, dtype=np.uint32)


def _seed_buffer(n, density, wsize, overlap, bsize):
    """Every seed is the minimum of two windows or the addition of a cell."""
    cells = (int(math.sqrt(n / density) / bsize) + 2) ** 2
    return _ids(min(n, _windows(n, density, wsize, overlap, bsize) // 2 + cells))


def _keep(buffer, values):
    buffer[:len(values)] = values
    return buffer


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch" or kind == "serve":
        tiles = _mix(case)
        xyz = _mix_cloud(tiles, case["cm"], seed)
        state = {"kind": kind, "xyz": xyz}
        params = [{"wsize": t.wsize, "overlap": t.overlap, "bsize": t.bsize} for t in tiles]
        state["seeds"] = np.concatenate([_seed_buffer(t.n, t.n / t.width ** 2, **p)
                                         for t, p in zip(tiles, params)])
        if kind == "batch":
            state["ctx"] = _context()
            state["desc"] = owm.batch_desc(list(zip((t.n for t in tiles), params)))
        else:
            state["server"] = _server()
            ends = np.cumsum([t.n for t in tiles])
            state["requests"] = [([a[e - t.n:e] for a in xyz], p)
                                 for t, e, p in zip(tiles, ends.tolist(), params)]
        return state
    x, y, z = _cloud(case, seed)
    state = {"kind": kind, "ctx": _context()}
    if kind == "stats":
        state["xy"] = (x, y)
        state["args"] = {k: case[k] for k in ("policy", "max_number", "min_radius", "level")}
        state["classes"] = np.zeros((4096, 3), dtype=np.int64)
        return state
    state["query"] = _query(case)
    state["seeds"] = _seed_buffer(case["n"], case["density"], **state["query"])
    if kind == "reader":
        host = [a.cpu().numpy() for a in (x, y, z)]
        box = synth.bbox(host[0], host[1])
        head = "%d\n%.17g\n%.17g\n%.17g\n%.17g\n" % ((case["n"],) + box)
        state["text"] = head.encode() + synth.format_xyz(*host, 2)
        return state
    if kind == "stages":
        state["query2"] = _query(case, "2")
        state["minima"] = _ids(_windows(case["n"], case["density"], **state["query"]))
        state["llp"] = state["seeds"].copy()
        state["adds"] = state["seeds"].copy()
        state["seeds"] = _seed_buffer(case["n"], case["density"], **state["query2"])
    elif case["box"]:
        state["query"]["bbox"] = tuple(float(v) for v in (x.min(), x.max(), y.min(), y.max()))
    if kind == "tile" and case["source"] == "host":
        x, y, z = (a.cpu().numpy() for a in (x, y, z))
    state["xyz"] = (x, y, z)
    return state


def run(state):
    kind = state["kind"]
    if kind == "tile":
        seeds = state["ctx"].run_tile(*state["xyz"], **state["query"])
        return _keep(state["seeds"], seeds), len(seeds)
    if kind == "batch":
        seeds, ends = state["ctx"].batch_run(*state["xyz"], state["desc"], split=False)
        return _keep(state["seeds"], seeds), ends
    if kind == "serve":
        server = state["server"]
        ids = [server.submit(*xyz, **params) for xyz, params in state["requests"]]
        seeds = [server.wait(i)[0] for i in ids]
        return _keep(state["seeds"], np.concatenate(seeds)), np.array([len(s) for s in seeds])
    if kind == "stages":
        ctx, q = state["ctx"], state["query"]
        tree = ctx.parallel_qtree(*state["xyz"])
        minima, _ = ctx.stage1(tree, **q)
        llp = ctx.stage2(tree, minima, **q)
        adds = ctx.stage3(tree, llp, **q)
        again = ctx.tree_run(tree, **state["query2"])
        tree.free()
        return [(_keep(state[k], v), len(v)) for k, v in (("minima", minima), ("llp", llp),
                                                          ("adds", adds), ("seeds", again))]
    if kind == "reader":
        ctx = state["ctx"]
        seeds = ctx.run_cloud(ctx.parse_xyz(state["text"]), **state["query"])
        return _keep(state["seeds"], seeds), len(seeds)
    classes, summary = state["ctx"].qtree_stats(*state["xy"], **state["args"])
    return _keep(state["classes"], classes), summary["leaves"], summary["depth"]


def work(case):
    """Each point's coordinates read once and the ids written (about one seed
    per 20 m x 20 m, small beside the input)."""
    kind = case["kind"]
    if kind == "batch" or kind == "serve":
        return {"bytes": 24.0 * sum(t.n for t in _mix(case)), "flops": 0.0}
    n = case["n"]
    if kind == "stats":
        return {"bytes": 16.0 * n, "flops": 0.0}
    if kind == "stages":  # the tree's build and two queries of it
        step = [case["wsize" + k] * (1 - case["overlap" + k]) for k in ("", "2")]
        windows = n / case["density"] / step[0] ** 2
        return {"bytes": 24.0 * n + 4.0 * windows, "flops": 0.0}
    if kind == "reader":  # the text, and the coordinates parsed from it
        return {"bytes": 28.0 * n + 24.0 * n, "flops": 0.0}
    return {"bytes": 24.0 * n, "flops": 0.0}


def exact(case, seed):
    """No case returns computed real numbers: ids and counts are compared as
    they are."""
    return None
