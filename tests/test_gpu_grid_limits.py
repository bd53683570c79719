"""The column-grid chain at the limits of its scratch memory: calls it hands to the
tree chain, and calls that only just stay with it.  Which chain answered is read
from the phases' launches; seeds are ids, against the oracle equal or wrong."""
import numpy as np
import pytest
import torch

import pyoracle as O
from fastowm_amd import owm, synth

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


@pytest.fixture(scope="module")
def ctx():
    with owm.Context(0) as c:
        # scratch of a larger call, so that nothing below starts from cleared memory
        t = synth.scaled(synth.config_c2(seed=1), 2_000_003)
        c.run_tile(*t.generate(), 12, 20, 0.8)
        yield c


def profiled(ctx, f):
    ctx.profile(True)
    got = f()
    calls = {k: v["calls"] for k, v in ctx.profile_read().items()}
    ctx.profile(False)
    return got, calls


def raster(side, origin=0.0, seed=0):
    """side x side points one metre apart."""
    g = origin + np.arange(side, dtype=np.float64)
    x, y = (a.ravel() for a in np.meshgrid(g, g))
    return x, y, np.round(np.random.default_rng(seed).normal(50.0, 3.0, len(x)), 1)


@pytest.mark.parametrize("side,p", [(450, (10, 20, 0.9)), (450, (5, 20, 0.8)), (800, (5, 20, 0.8))])
def test_full_pool(ctx, side, p):
    """Rasters whose every point lies on an edge, in both sizes of sort tiles: as a
    tile, beside a plain tile in a batch, and as a resident tree."""
    say("grid limits, full pool", side, p)
    c = raster(side, 512_000.0)
    want = O.run(*c, *p, 32)[0]
    got, calls = profiled(ctx, lambda: ctx.run_tile(*c, *p))
    assert calls["grid_partition"] and calls["sort_tree_pass"] and np.array_equal(got, want)
    plain = synth.scaled(synth.config_c1(seed=2), 132_072).generate()
    q = dict(wsize=10, bsize=20, overlap=0.8)
    desc = [(len(plain[0]), q), (len(c[0]), dict(wsize=p[0], bsize=p[1], overlap=p[2]))]
    both = [np.concatenate(a) for a in zip(plain, c)]
    for graph in (False, True, True, True):
        a, b = ctx.batch_run(*both, desc, graph=graph)
        assert np.array_equal(a, O.run(*plain, 10, 20, 0.8, 32)[0]) and np.array_equal(b, want)
    tree = ctx.parallel_qtree(*c)
    (minima, _), calls = profiled(ctx, lambda: ctx.stage1(tree, p[0], p[2], p[1]))
    assert calls["grid_partition"] and calls["stage1"]
    box = synth.bbox(c[0], c[1])
    assert np.array_equal(minima, O.Tree(*c, O.params(*p, box, len(c[0]), 32)).stage1())
    assert np.array_equal(ctx.tree_run(tree, *p), want)
    tree.free()


@pytest.mark.parametrize("frac,grid", [(0.10, True), (0.30, False)])
def test_many_on_edges(ctx, frac, grid):
    """More than 4M points: beyond a sixth of them on edges the tree chain answers.
    Against the tree chain, which is compared with the oracle elsewhere."""
    say("grid limits, many on edges", frac)
    rng = np.random.default_rng(4)
    n = (4 << 20) + 5
    side = 900.0
    x, y = rng.random(n) * side, rng.random(n) * side
    x[:2], y[:2] = (0.0, side), (0.0, side)
    m = rng.random(n) < frac
    x[m] = np.floor(x[m])
    c = x, y, np.round(rng.normal(50.0, 3.0, n), 1)
    want = ctx.run_tile(*c, 5, 20, 0.8, 32)
    got, calls = profiled(ctx, lambda: ctx.run_tile(*c, 5, 20, 0.8))
    assert (calls["sort_tree_pass"] == 0) == grid and np.array_equal(got, want)


@pytest.mark.parametrize("frac", [0.05, 0.12, 0.24])
@pytest.mark.parametrize("order", ["random", "scan"])
def test_share_on_edges(ctx, frac, order):
    """A share of the points on edges, in one tile and in one of a batch: below a
    quarter the column grid answers, every window block meets listed points."""
    say("grid limits, share on edges", frac, order)
    rng = np.random.default_rng(int(100 * frac))
    n = 300_000
    x, y = rng.random(n) * 190.0, rng.random(n) * 190.0
    x[:2], y[:2] = (0.0, 190.0), (0.0, 190.0)
    m = rng.random(n) < frac / 2
    x[m], y[~m & (rng.random(n) < frac / 2)] = np.round(x[m]), 77.0
    if order == "scan":
        s = np.argsort(y, kind="stable")
        x, y = x[s], y[s]
    c = x, y, np.round(rng.normal(50.0, 3.0, n), 1)
    want = O.run(*c, 5, 20, 0.8, 32)[0]
    got, calls = profiled(ctx, lambda: ctx.run_tile(*c, 5, 20, 0.8))
    assert calls["grid_partition"] == 1 and calls["sort_tree_pass"] == 0
    assert np.array_equal(got, want)


def test_longest_lists(ctx):
    """More listed points in one bucket than a window block takes: the tree chain
    answers.  Against the tree chain, as above."""
    say("grid limits, longest lists")
    rng = np.random.default_rng(9)
    n = 2_000_000
    x, y = rng.random(n) * 500.0, rng.random(n) * 500.0
    m = rng.random(n) < 0.2
    x[m], y[m] = 100.0, 140.0 + rng.random(m.sum())
    x[:2], y[:2] = (0.0, 500.0), (0.0, 500.0)
    c = x, y, np.round(rng.normal(50.0, 3.0, n), 1)
    want = ctx.run_tile(*c, 10, 20, 0.8, 32)
    got, calls = profiled(ctx, lambda: ctx.run_tile(*c, 10, 20, 0.8))
    assert calls["sort_tree_pass"] > 0 and np.array_equal(got, want)


def test_handed_on_calls_replay(ctx):
    """A repeated call on device memory, handed on each time: its chains are replayed from
    the third call on; other calls lie between."""
    say("grid limits, replays of calls handed on")
    c, p = raster(450, 512_000.0), (5, 20, 0.8)
    d = [torch.from_numpy(a).cuda() for a in c]
    e = [torch.from_numpy(a).cuda() for a in raster(450, 512_000.0, seed=1)]
    wants = [O.run(*c, *p, 32)[0], O.run(*raster(450, 512_000.0, seed=1), *p, 32)[0]]
    for k in (0, 0, 0, 0, 1, 0, 1, 1, 1, 0):
        assert np.array_equal(ctx.run_tile(*(d, e)[k], *p), wants[k])
    d[2].copy_(e[2])  # the same memory, other heights
    assert np.array_equal(ctx.run_tile(*d, *p), wants[1])


@pytest.mark.parametrize("at", [0, 1, 4095, 4096, 8190, 8191])
def test_first_bad_id(ctx, at):
    """Ids that stage 2 refuses, by their place in the list; OWM_NONE is no such id."""
    say("grid limits, bad id", at)
    c = synth.scaled(synth.config_c1(seed=3), 5000).generate()
    tree = ctx.parallel_qtree(*c)
    ids = np.full(8192, owm.NONE, np.uint32)
    ids[::3] = np.arange(len(ids[::3]))
    ids[7] = 4999
    ids[8191] = 0xFFFFFFFE if at < 8191 else owm.NONE
    ids[at] = 5000
    with pytest.raises(owm.OWMError, match=rf"min_ids\[{at}\] = 5000 "):
        ctx.stage2(tree, ids, 10, 0.8)
    tree.free()


def _clouds():
    rng = np.random.default_rng(11)
    plain = synth.scaled(synth.config_c2(seed=5), 150_000).generate()
    yield "plain", plain, (10, 20, 0.8)
    yield "cm", tuple(np.round(a, 2) for a in plain), (7, 13, 0.5)
    yield "unpaired", plain, (12, 20, 0.7)
    yield "no cells", plain, (8, 0, 0.0)
    yield "one sort tile", tuple(a[:1023] for a in plain), (10, 20, 0.8)
    x, y, z = (a.copy() for a in synth.scaled(synth.config_c2(seed=6), 700_000).generate())
    yield "large sort tiles", (x, y, z), (10, 20, 0.8)
    h = 400.0 * rng.random((2, 300_000))
    h[:, :270_000] = 50.0 + 6.0 * rng.random((2, 270_000))
    h[0, :5000] = np.round(h[0, :5000])
    yield "heavy", (h[0], h[1], np.round(rng.normal(50.0, 2.0, 300_000), 1)), (10, 20, 0.8)


@pytest.mark.parametrize("name,c,p", [pytest.param(*v, id=v[0]) for v in _clouds()])
def test_grid_alone_answers(ctx, name, c, p):
    """The column grid's own answer: nothing of the tree chain runs behind it, neither for
    a whole run nor for a resident tree's queries."""
    say("grid limits, grid alone", name)
    want = O.run(*c, *p, 32)[0]
    got, calls = profiled(ctx, lambda: ctx.run_tile(*c, *p))
    assert calls["grid_partition"] == 1 and not calls["sort_tree_pass"] and not calls["stage1"]
    assert np.array_equal(got, want)
    tree = ctx.parallel_qtree(*c)
    (minima, _), calls = profiled(ctx, lambda: ctx.stage1(tree, p[0], p[2], p[1]))
    assert calls["grid_partition"] == 1 and not calls["stage1"] and not calls["stage1_join"]
    assert np.array_equal(minima, O.Tree(*c, O.params(*p, synth.bbox(c[0], c[1]), len(c[0]), 32)).stage1())
    got, calls = profiled(ctx, lambda: ctx.tree_run(tree, *p))
    assert calls["grid_partition"] == 1 and not calls["stage1"] and np.array_equal(got, want)
    tree.free()


@pytest.mark.parametrize("shift,grid", [(0.0, False), (0.25, True)])
def test_lattice_and_its_box(ctx, shift, grid):
    """Points on a lattice of the windows' step: all on edges where the box starts on the
    lattice, none where the points are shifted in the same box."""
    say("grid limits, lattice", shift)
    rng = np.random.default_rng(9)
    n = 400_000
    x, y = (rng.integers(1, 800, n) + shift for _ in range(2))
    z = np.round(rng.normal(50.0, 3.0, n), 1)
    box = (0.0, 801.0, 0.0, 801.0)
    want = O.run(x, y, z, 5, 20, 0.8, 32, box)[0]
    got, calls = profiled(ctx, lambda: ctx.run_tile(x, y, z, 5, 20, 0.8, bbox=box))
    assert calls["grid_partition"] == 1 and (calls["sort_tree_pass"] == 0) == grid
    assert np.array_equal(got, want) and len(want) > 1000
