"""Whole runs by the column-grid chain (leaf_size 0) against the oracle, at the
sizes where it can go wrong: the edges of sort tiles, buckets of one cell row,
shares of large buckets, points on and within ulps of window and cell edges,
more points without a column than the chain's pool holds, and parameters it
hands to the tree chain.  Seeds are ids: equal or wrong."""
import numpy as np
import pytest

import pyoracle as O
from fastowm_amd import owm, synth

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def ctx():
    with owm.Context(0) as c:
        yield c


def _run(ctx, x, y, z, ws, bs, ov, phase=True):
    want, _, _ = O.run(x, y, z, ws, bs, ov, 32)
    ctx.profile(True)
    got = ctx.run_tile(x, y, z, ws, bs, ov)
    calls = ctx.profile_read()
    ctx.profile(False)
    assert (calls["grid_partition"]["calls"] > 0) == phase
    assert np.array_equal(got, want), (len(got), len(want))
    assert np.array_equal(ctx.run_tile(x, y, z, ws, bs, ov), want)  # again: nothing left over
    return want


@pytest.mark.parametrize("n", [1, 2, 63, 64, 4095, 4096, 4097, 8192, 12289, 70_001])
@pytest.mark.parametrize("ws,bs,ov", [(10, 20, 0.8), (7, 13, 0.5), (12, 20, 0.7), (8, 0, 0.0)])
def test_sizes(ctx, n, ws, bs, ov):
    say("grid chain", n, ws, bs, ov)
    t = synth.scaled(synth.config_c1(seed=n), max(n, 400))
    x, y, z = t.generate()
    x, y, z = x[:n].copy(), y[:n].copy(), z[:n].copy()
    if n < 3:  # a box of one or two points needs an extent
        x, y, z = np.append(x, x[0] + 30.0), np.append(y, y[0] + 25.0), np.append(z, z[0])
    _run(ctx, x, y, z, ws, bs, ov)


@pytest.mark.parametrize("ws,bs,ov", [(12, 20, 0.8), (20, 10, 0.5), (5, 30, 0.9), (15, 25, 0.6),
                                      (9, 17, 0.63), (6, 14, 0.97), (3, 1, 0.0), (1, 2, 0.5)])
@pytest.mark.parametrize("cm", [False, True])
def test_parameters(ctx, ws, bs, ov, cm):
    say("grid chain parameters", ws, bs, ov, cm)
    t = synth.scaled(synth.config_c2(seed=ws), 150_000)
    x, y, z = t.generate()
    if cm:  # centimetre coordinates put about one point in a hundred on an edge
        x, y, z = (np.round(a, 2) for a in (x, y, z))
    _run(ctx, x, y, z, ws, bs, ov)


@pytest.mark.parametrize("origin", [(0.0, 0.0), (612_345.0, 4_512_345.0), (-1234.56, 7.89)])
@pytest.mark.parametrize("ws,bs,ov", [(8, 20, 0.5), (10, 20, 0.8), (12, 9, 0.7), (10, 6, 0.0)])
def test_points_near_edges(ctx, origin, ws, bs, ov):
    """Points 0 to 3 ulps, 1e-9 and 1e-6 either side of window and cell edges
    and of their crossings, among random ones; z in whole steps (ties)."""
    say("grid chain, points near edges", origin, ws, bs, ov)
    rng = np.random.default_rng(int(ws * 100 + bs))
    side, out = 180.0, []
    for o in origin:
        d = round(ws * (1 - ov), 2)
        i = np.arange(int((side + 2 * ws * ov) / d) + 2)
        c = (o - ws // 2 + d) + i * d
        edges = np.concatenate([c - ws // 2, c + ws // 2])
        k = np.arange(int(side / bs) + 1)
        edges = np.concatenate([edges, (o + bs // 2 + k * bs) - bs // 2, (o + bs // 2 + k * bs) + bs // 2])
        edges = edges[(edges > o) & (edges < o + side)]
        v = rng.choice(edges, 9_000)
        step = rng.integers(-3, 4, 9_000)
        for _ in range(3):
            v = np.where(step > 0, np.nextafter(v, np.inf), np.where(step < 0, np.nextafter(v, -np.inf), v))
            step -= np.sign(step)
        v[::7] += rng.choice([-1e-6, -1e-9, 1e-9, 1e-6], len(v[::7]))
        out.append((v, o + side * rng.random(60_000)))
    (ex, rx), (ey, ry) = out
    x = np.concatenate([ex, ex, rx[:9_000], rx, [origin[0], origin[0] + side]])
    y = np.concatenate([ey, ry[:9_000], ey, ry, [origin[1], origin[1] + side]])
    z = np.round(rng.normal(50.0, 2.0, len(x)), 1)
    p = rng.permutation(len(x))
    _run(ctx, x[p], y[p], z[p], ws, bs, ov)


def test_special_values(ctx):
    """NaN and infinite coordinates and heights, the type's largest value, zeros of
    both signs; coordinates far from every edge."""
    say("grid chain, special values")
    t = synth.scaled(synth.config_c1(seed=5), 40_000)
    x, y, z = t.generate()
    box = synth.bbox(x, y)
    rng = np.random.default_rng(5)
    for a in (x, y, z):
        a[rng.integers(0, len(a), 300)] = np.nan
    for a, v in ((x, np.inf), (y, -np.inf), (z, np.inf), (z, -np.inf), (z, 1.7976931348623157e308),
                 (z, -0.0), (z, 0.0), (x, 1e300), (y, -1e300)):
        a[rng.integers(0, len(a), 60)] = v
    want = None
    for leaf in (32, 0):
        got = ctx.run_tile(x, y, z, 12, 20, 0.8, leaf, bbox=box)
        want = got if want is None else want
    assert np.array_equal(got, want) and len(want) > 50


def test_lattice_falls_back(ctx):
    """Every point on an edge: more than the pool holds, so the tree chain
    answers; with the same points moved off the edges the grid chain does."""
    say("grid chain, edge lattice")
    rng = np.random.default_rng(9)
    n = 400_000
    x, y = (rng.integers(0, 801, n).astype(np.float64) for _ in range(2))
    z = np.round(rng.normal(50.0, 3.0, n), 1)
    _run(ctx, x, y, z, 8, 20, 0.5)
    _run(ctx, x + 0.25, y + 0.25, z, 8, 20, 0.5)


def test_shares_of_large_buckets(ctx):
    """Few cells and many points: buckets read in shares, and cells beyond the
    first class of buckets in one batch with small tiles."""
    say("grid chain, shares")
    big = synth.Tile(seed=3, n=3_000_000, width=150.0, height=140.0)
    wide = synth.Tile(seed=4, n=300_000, width=1500.0, height=1300.0)
    small = synth.scaled(synth.config_c1(seed=6), 20_011)
    tiles = [(small, 10, 20, 0.8), (wide, 5, 12, 0.9), (big, 12, 20, 0.75), (small, 12, 20, 0.7)]
    arrs = [t.generate() for t, *_ in tiles]
    wants = [O.run(*a, ws, bs, ov, 32)[0] for a, (_, ws, bs, ov) in zip(arrs, tiles)]
    desc = [(len(a[0]), dict(wsize=ws, bsize=bs, overlap=ov)) for a, (_, ws, bs, ov) in zip(arrs, tiles)]
    xyz = [np.concatenate([a[k] for a in arrs]) for k in range(3)]
    for graph in (False, True, True, False, True):
        got = ctx.batch_run(*xyz, desc, graph=graph)
        for i, (g, w) in enumerate(zip(got, wants)):
            assert np.array_equal(g, w), f"tile {i}"


def _batch(ctx, clouds, params, graph=False):
    wants = [O.run(*c, *p, 32)[0] if len(c[0]) else np.empty(0, np.uint32) for c, p in zip(clouds, params)]
    box = (0.0, 50.0, 0.0, 40.0)
    desc = [(len(c[0]), dict(wsize=p[0], bsize=p[1], overlap=p[2], bbox=None if len(c[0]) else box))
            for c, p in zip(clouds, params)]
    got = ctx.batch_run(*(np.concatenate([c[k] for c in clouds]) for k in range(3)), desc, graph=graph)
    for i, (g, w) in enumerate(zip(got, wants)):
        assert np.array_equal(g, w), f"tile {i}"
    return wants


@pytest.mark.parametrize("order", ["front", "middle", "end", "all_between"])
def test_empty_tiles(ctx, order):
    """Tiles without points (their boxes given) in front, between, at the end: the
    other tiles' ranges stay theirs."""
    say("grid chain, empty tiles", order)
    tiles = [synth.scaled(synth.config_c1(seed=s), n).generate() for s, n in ((1, 5000), (2, 131_072), (3, 777))]
    e = (np.empty(0),) * 3
    clouds = {"front": [e, e] + tiles, "middle": tiles[:1] + [e, e, e] + tiles[1:], "end": tiles + [e, e],
              "all_between": [e, tiles[0], e, tiles[1], e, tiles[2], e]}[order]
    _batch(ctx, clouds, [(10, 20, 0.8)] * len(clouds))


def test_dense_seeds_over_many_tiles(ctx):
    """Nearly every point a seed (windows of a few points), so that a stretch of
    the bitmap holds many stages of indices, with tile starts at and off its
    boundaries; 70 tiles take the general box pass."""
    say("grid chain, dense seeds")
    rng = np.random.default_rng(3)
    for sizes in ([131_072, 4096, 60_001, 262_144, 5], [int(v) for v in rng.integers(40, 4000, 70)]):
        clouds = []
        for n in sizes:
            s = 3.0 * np.sqrt(n) + 5.0
            c = [rng.random(n) * s, rng.random(n) * s, np.round(rng.random(n) * 50.0, 1)]
            c[0][:2], c[1][:2] = (0.0, s), (0.0, s)
            clouds.append(c)
        wants = _batch(ctx, clouds, [(3, 4, 0.0)] * len(sizes))
        assert sum(len(w) for w in wants) > 0.3 * sum(sizes)


@pytest.mark.parametrize("n,leaf", [(3, 1), (64, 32), (4097, 8), (50_001, 32), (300_000, 16)])
@pytest.mark.parametrize("cm", [False, True])
def test_resident_tree(ctx, n, leaf, cm):
    """Minima and seeds of a resident tree (its points permuted) by the chain:
    several parameters, a box of the query's own, ties, points on edges."""
    say("grid chain, resident tree", n, leaf, cm)
    t = synth.scaled(synth.config_c1(seed=n), max(n, 400))
    x, y, z = (a[:n].copy() for a in t.generate())
    if n < 4:
        x, y = np.array([0.0, 40.5, 11.0]), np.array([1.0, 30.5, 12.0])
    z = np.round(z, 1)
    if cm:
        x, y = np.round(x, 2), np.round(y, 2)
    box = synth.bbox(x, y)
    tree = ctx.parallel_qtree(x, y, z, leaf_size=leaf)
    for ws, bs, ov, b in [(10, 20, 0.8, None), (7, 13, 0.5, None), (8, 0, 0.0, None), (3, 1, 0.0, None),
                          (12, 20, 0.75, (box[0] - 7.0, box[1] + 3.0, box[2] - 2.0, box[3] + 9.0)),
                          (9, 12, 0.7, (box[0] + 5.0, box[1] + 3.0, box[2] - 2.0, box[3] - 9.0))]:
        inside = b is None or (b[0] <= box[0] and box[1] <= b[1] and b[2] <= box[2] and box[3] <= b[3])
        p = O.params(ws, bs, ov, b or box, n, leaf)
        ctx.profile(True)
        gm, d = ctx.stage1(tree, ws, ov, bs, bbox=b)
        seeds = ctx.tree_run(tree, ws, bs, ov, bbox=b)
        calls = ctx.profile_read()
        ctx.profile(False)
        assert calls["grid_partition"]["calls"] == (2 if inside else 0)
        assert (d.ncols, d.nrows) == (p.ncols, p.nrows)
        assert np.array_equal(gm, O.Tree(x, y, z, p).stage1())
        assert np.array_equal(seeds, O.run(x, y, z, ws, bs, ov, leaf, b or box)[0])
    tree.free()


def test_resident_tree_falls_back(ctx):
    """More points on edges than the pool holds: the tree chain answers."""
    say("grid chain, resident tree falls back")
    rng = np.random.default_rng(10)
    n = 400_000
    x, y = (rng.integers(0, 801, n).astype(np.float64) for _ in range(2))
    z = np.round(rng.normal(50.0, 3.0, n), 1)
    box = synth.bbox(x, y)
    p = O.params(8, 20, 0.5, box, n, 32)
    tree = ctx.parallel_qtree(x, y, z)
    gm, _ = ctx.stage1(tree, 8, 0.5, 20)
    assert np.array_equal(gm, O.Tree(x, y, z, p).stage1())
    assert np.array_equal(ctx.tree_run(tree, 8, 20, 0.5), O.run(x, y, z, 8, 20, 0.5, 32)[0])
    tree.free()


@pytest.mark.parametrize("frac", [0.02, 0.3, 0.97])
def test_box_of_a_part(ctx, frac):
    """A box given that holds a part of the points: most lie before the first
    edges or behind the last ones; some not a number."""
    say("grid chain, box of a part", frac)
    t = synth.scaled(synth.config_c1(seed=3), 60_000)
    x, y, z = t.generate()
    x[::997], y[5::997] = np.nan, np.inf
    x0, x1, y0, y1 = synth.bbox(x[np.isfinite(x)], y[np.isfinite(y)])
    box = (x0 + 0.1 * frac * (x1 - x0), x0 + frac * (x1 - x0), y0, y0 + max(frac, 0.2) * (y1 - y0))
    for ws, bs, ov in ((10, 20, 0.8), (7, 13, 0.5), (8, 0, 0.0)):
        want, _, _ = O.run(x, y, z, ws, bs, ov, 32, box)
        ctx.profile(True)
        got = ctx.run_tile(x, y, z, ws, bs, ov, bbox=box)
        calls = ctx.profile_read()
        ctx.profile(False)
        assert calls["grid_partition"]["calls"] == 1
        assert np.array_equal(got, want)


@pytest.mark.parametrize("n,blobs", [(70_000, 1), (300_000, 1), (1_500_000, 1), (1_500_000, 3)])
@pytest.mark.parametrize("order", ["random", "sorted"])
def test_heavy_buckets(ctx, n, blobs, order):
    """Most points in a few square metres: stretches of one bucket's points binned
    by several workgroups and added up; ties, and points on edges (listed by
    several workgroups) among them.  As a whole run, in a batch, captured, and of
    a resident tree."""
    say("grid chain, heavy buckets", n, blobs, order)
    rng = np.random.default_rng(n + blobs)
    side = 400.0
    x, y = rng.random(n) * side, rng.random(n) * side
    k = int(n * 0.9)
    at = rng.random((blobs, 2)) * (side - 20.0) + 5.0
    b = rng.integers(0, blobs, k)
    x[:k], y[:k] = at[b, 0] + rng.random(k) * 6.0, at[b, 1] + rng.random(k) * 6.0
    x[: k // 50], y[: k // 70] = np.round(x[: k // 50]), np.round(y[: k // 70])
    z = np.round(rng.normal(50.0, 2.0, n), 1)
    z[::5003] = np.nan
    if order == "random":
        p = rng.permutation(n)
        x, y, z = x[p], y[p], z[p]
    want = _run(ctx, x, y, z, 10, 20, 0.8)
    _run(ctx, x, y, z, 7, 13, 0.5)
    tree = ctx.parallel_qtree(x, y, z)
    assert np.array_equal(ctx.tree_run(tree, 10, 20, 0.8), want)
    tree.free()
    for graph in (False, True, True, True):
        got = ctx.batch_run(*(np.concatenate([a, a]) for a in (x, y, z)),
                            [(n, dict(wsize=10, bsize=20, overlap=0.8)),
                             (n, dict(wsize=7, bsize=13, overlap=0.5))], graph=graph)
        assert np.array_equal(got[0], want)
        assert np.array_equal(got[1], O.run(x, y, z, 7, 13, 0.5, 32)[0])


@pytest.mark.parametrize("n", [1023, 1025, 131_072, 131_073, 132_097, 524_288, 524_289, 528_385])
def test_sort_tile_sizes(ctx, n):
    """Either side of the points at which sort tiles grow, and of their ends."""
    say("grid chain, sort tiles", n)
    x, y, z = (a[:n].copy() for a in synth.scaled(synth.config_c1(seed=n), n).generate())
    _run(ctx, x, y, z, 10, 20, 0.8)
    _run(ctx, np.round(x, 2), np.round(y, 2), z, 7, 13, 0.5)


@pytest.mark.parametrize("cm", [False, True])
def test_largest_sort_tiles(ctx, cm):
    """A sparse tile of 50M points takes the largest sort tiles; against the tree
    chain (an explicit leaf size), which is compared with the oracle elsewhere."""
    say("grid chain, largest sort tiles", cm)
    n = (48 << 20) + 8191
    rng = np.random.default_rng(48)
    side = np.sqrt(n / 3.0)
    x, y = rng.random(n) * side, rng.random(n) * side
    z = np.round(rng.normal(50.0, 3.0, n), 1)
    if cm:
        x, y = np.round(x, 2), np.round(y, 2)
    want = ctx.run_tile(x, y, z, 10, 20, 0.8, 32)
    ctx.profile(True)
    got = ctx.run_tile(x, y, z, 10, 20, 0.8)
    calls = ctx.profile_read()
    ctx.profile(False)
    assert calls["grid_partition"]["calls"] == 1
    assert np.array_equal(got, want) and len(want) > 300_000


@pytest.mark.parametrize("tiles,n,grid", [(64, 300, True), (65, 4095, False), (65, 4096, True), (300, 50, False)])
def test_many_small_tiles(ctx, tiles, n, grid):
    """Either side of the rule that leaves many tiles of few points to the tree chain."""
    say("grid chain, many small tiles", tiles, n)
    clouds = [synth.scaled(synth.config_c1(seed=s), n).generate() for s in range(tiles)]
    ctx.profile(True)
    _batch(ctx, clouds, [(10, 20, 0.8)] * tiles)
    calls = ctx.profile_read()
    ctx.profile(False)
    assert (calls["grid_partition"]["calls"] > 0) == grid
