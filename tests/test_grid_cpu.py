"""The column-grid chain's kernels and planning code on the CPU (tests/hipcpu):
what cannot be provoked on a device, or must not be before it is right.  Against
the oracle: seeds are ids, equal or wrong."""
import os
import subprocess

import numpy as np
import pytest

import pyoracle as O
from fastowm_amd import synth

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "fastowm_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    """The chain built for the CPU: LDS arrays whose size the launch gives are globals
    there, and the one inline wait has nothing to wait for."""
    d = tmp_path_factory.mktemp("grid_cpu")
    with open(os.path.join(CSRC, "grid.hip")) as f:
        text = f.read()
    text = text.replace("extern __shared__", "extern").replace(
        'asm volatile("s_waitcnt vmcnt(0)" ::: "memory");', "")
    assert "asm" not in text
    src, out = str(d / "grid_source.h"), str(d / "grid_cpu")
    with open(src, "w") as f:
        f.write(text)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-D__HIPCC__", f'-DGRID_SOURCE="{src}"',
                    "-I", os.path.join(HERE, "hipcpu"), "-I", CSRC, "-Wl,--unresolved-symbols=ignore-all", "-o", out,
                    os.path.join(HERE, "hipcpu", "grid_cpu.cpp"), os.path.join(CSRC, "owm_grid.cpp"),
                    os.path.join(CSRC, "owm_host.cpp")], check=True)
    return out


def chain(exe, clouds, params, mode=0, poke=0, calls=1, boxes=None):
    """(taken, flags, ids per tile) of the chain for these tiles."""
    head = [mode, poke, calls, len(clouds)]
    for k, (c, p) in enumerate(zip(clouds, params)):
        box = boxes[k] if boxes else None
        head += [len(c[0]), *p, 1 if box else 0, *(box or (0, 0, 0, 0))]
    paths = exe + ".in", exe + ".out"
    with open(paths[0], "wb") as f:
        np.array(head, np.float64).tofile(f)
        for k in range(3):
            np.concatenate([c[k] for c in clouds]).astype(np.float64).tofile(f)
    r = subprocess.run([exe, *paths], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stderr)
    with open(paths[1], "rb") as f:
        status, taken, flags, count, stray, *work = np.fromfile(f, np.int64, 11)
        off = np.fromfile(f, np.int64, len(clouds) + 1)
        ids = np.fromfile(f, np.uint32, count)
    assert status == 0 and stray == 0
    chain.after, chain.part, chain.groups, chain.replays, chain.repeats, chain.largest = work
    return bool(taken), int(flags), [ids[a:b] for a, b in zip(off, off[1:])] if taken else None


def oracle(c, p, box=None):
    return O.run(*c, *p, 32, box)[0]


def raster(side, step=1.0, seed=0):
    """side x side points on a lattice."""
    g = np.arange(side) * step
    x, y = (a.ravel().astype(np.float64) for a in np.meshgrid(g, g))
    z = np.round(np.random.default_rng(seed).normal(50.0, 3.0, len(x)), 1)
    return x, y, z


def test_answers(exe):
    """The chain on the CPU equals the oracle: plain tiles, centimetres, a resident
    tree's seeds and minima, heavy stretches."""
    t = synth.scaled(synth.config_c1(seed=3), 9_001).generate()
    cm = tuple(np.round(a, 2) for a in synth.scaled(synth.config_c1(seed=4), 20_000).generate())
    p = (10, 20, 0.8)
    taken, flags, got = chain(exe, [t, cm], [p, (7, 13, 0.5)])
    assert taken and flags == 0
    assert np.array_equal(got[0], oracle(t, p)) and np.array_equal(got[1], oracle(cm, (7, 13, 0.5)))
    taken, _, got = chain(exe, [cm], [p], mode=1)
    assert taken and np.array_equal(got[0], oracle(cm, p))
    taken, _, got = chain(exe, [cm], [p], mode=2)
    assert taken and np.array_equal(
        got[0], O.Tree(*cm, O.params(*p, synth.bbox(cm[0], cm[1]), len(cm[0]), 32)).stage1())


@pytest.mark.parametrize("side,p", [(450, (10, 20, 0.9)), (800, (5, 20, 0.8))])
def test_full_pool(exe, side, p):
    """A raster whose every point lies on an edge: more than the pool holds.  The chain
    hands the call on, and no kernel took a place that was never written for a point
    (grid_cpu's device memory starts with points whose ids lie far out of range)."""
    c = raster(side)
    for mode in (0, 1, 2):
        taken, flags, _ = chain(exe, [c], [p], mode=mode)
        assert not taken and flags & 32


@pytest.mark.parametrize("side,ok", [(247, True), (560, False)])
def test_raster_beside_a_plain_tile(exe, side, ok):
    """The first shares of the pool are the plain tile's, which has no use for them."""
    tiles = synth.scaled(synth.config_c1(seed=3), 132_072).generate(), raster(side)
    params = (10, 20, 0.8), (5, 20, 0.8)
    taken, flags, got = chain(exe, tiles, params)
    assert taken == ok and bool(flags & 32) != ok
    for k in range(2 if ok else 0):
        assert np.array_equal(got[k], oracle(tiles[k], params[k]))


def heavy_cloud(n=160_000, seed=5, on_edges=0):
    """Most points in a few square metres; about half of the first `on_edges` on the
    edges of windows (the corner points place the box)."""
    rng = np.random.default_rng(seed)
    x, y = rng.random(n) * 400.0, rng.random(n) * 400.0
    k = int(n * 0.95)
    x[:k], y[:k] = 101.0 + rng.random(k) * 6.0, 203.0 + rng.random(k) * 6.0
    m = on_edges
    x[:m], y[:m] = np.round(x[:m]), np.round(y[:m])
    x[-2:], y[-2:] = (0.0, 400.0), (0.0, 400.0)
    s = rng.permutation(n)
    return x[s], y[s], np.round(rng.normal(50.0, 2.0, n), 1)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("edges", [0, 3000])
def test_heavy_stretches(exe, mode, edges):
    c, p = heavy_cloud(on_edges=edges), (10, 20, 0.8)
    taken, flags, got = chain(exe, [c], [p], mode=mode)
    assert taken and flags == 0 and np.array_equal(got[0], oracle(c, p))


def test_flag_raised_during_the_heavy_launch(exe):
    """Another workgroup of the launch finds its list full while waves of this one
    start: a workgroup's waves go on or stop together."""
    c, p = heavy_cloud(on_edges=3000), (10, 20, 0.8)
    taken, _, _ = chain(exe, [c], [p], poke=1)
    assert not taken


def test_full_queue(exe):
    """More heavy stretches than the queue holds: entries that were never written are
    not taken for stretches."""
    c, p = heavy_cloud(on_edges=3000), (10, 20, 0.8)
    taken, flags, _ = chain(exe, [c], [p], poke=2)
    assert not taken and flags & 32


def test_handed_on_early(exe):
    """A raster whose every point lies on an edge: once the pool is full no further
    sort tile is partitioned, and the launches behind it do nothing."""
    taken, flags, _ = chain(exe, [raster(800)], [(5, 20, 0.8)])
    assert not taken and flags & 32
    whole = chain.part
    chain(exe, [tuple(a * 0.93 for a in raster(800))], [(5, 20, 0.8)])  # (off the edges: every sort tile)
    per_tile = chain.part / chain.groups
    assert chain.after == 0 and whole < 0.6 * per_tile * chain.groups


@pytest.mark.parametrize("frac,ok", [(0.10, True), (0.25, False)])
def test_many_on_edges(exe, frac, ok):
    """Beyond 4M points a sixth of the points on edges in a quarter of the sort tiles
    decides; a few sort tiles full of them do not."""
    n = (4 << 20) + 4096
    rng = np.random.default_rng(3)
    side = 400.0
    x, y = rng.random(n) * side, rng.random(n) * side
    x[:2], y[:2] = (0.0, side), (0.0, side)
    x[rng.random(n) < frac] //= 1.0
    x[200_000:260_000] //= 1.0
    z = np.round(rng.normal(50.0, 3.0, n), 1)
    taken, flags, got = chain(exe, [(x, y, z)], [(5, 20, 0.8)])
    assert taken == ok and (flags == 0) == ok and chain.after == 0
    # (a taken cloud passes 11 barriers a sort tile)
    assert ok or chain.part < 0.4 * 11 * chain.groups


@pytest.mark.parametrize("place", ["sort tiles", "bucket"])
def test_places_of_other_shares(exe, place):
    """Points on edges in few sort tiles, or in one bucket: the pool's and the lists'
    shares lend each other room."""
    rng = np.random.default_rng(8)
    n = 300_000
    x, y = rng.random(n) * 300.0, rng.random(n) * 300.0
    if place == "sort tiles":  # every 64th of 2048 points, whose share is the same
        m = (np.arange(n) // 2048) % 64 == 5
        x[m] = np.floor(x[m])
    else:
        m = rng.random(n) < 0.03
        x[m], y[m] = 100.0 + np.floor(rng.random(m.sum()) * 3.0), 140.0 + rng.random(m.sum()) * 3.0
    x[:2], y[:2] = (0.0, 300.0), (0.0, 300.0)
    c, p = (x, y, np.round(rng.normal(50.0, 3.0, n), 1)), (5, 20, 0.8)
    for mode in (0, 1):
        taken, flags, got = chain(exe, [c], [p], mode=mode)
        assert taken and flags == 0 and np.array_equal(got[0], oracle(c, p))


def test_longest_lists(exe):
    """More listed points in one bucket than a window block takes: handed on."""
    rng = np.random.default_rng(9)
    n = 1_900_000
    x, y = rng.random(n) * 500.0, rng.random(n) * 500.0
    m = rng.random(n) < 0.2
    x[m], y[m] = 100.0, 140.0 + rng.random(m.sum())
    x[:2], y[:2] = (0.0, 500.0), (0.0, 500.0)
    taken, flags, _ = chain(exe, [(x, y, np.round(rng.normal(50.0, 3.0, n), 1))], [(10, 20, 0.8)])
    assert not taken and flags & 32


def test_handed_on_calls_replay(exe):
    """A repeated call that the chain hands on: both chains find their last key again."""
    taken, _, _ = chain(exe, [raster(450)], [(5, 20, 0.8)], mode=3, calls=4)
    assert not taken and chain.replays == 3 and chain.repeats == 3


def test_no_memory_for_the_chain(exe):
    """The tree chain's memory is not this chain's: without room for its scratch the
    call is handed on, not refused."""
    t = synth.scaled(synth.config_c1(seed=3), 9_001).generate()
    for mode in (0, 1, 2):
        taken, _, _ = chain(exe, [t], [(10, 20, 0.8)], mode=mode, poke=3)
        assert not taken


@pytest.mark.parametrize("origin,ok", [(1e9, True), (1e15, False)])
def test_far_coordinates(exe, origin, ok):
    """Coordinates that a window step is lost in: the tree chain's from the start."""
    rng = np.random.default_rng(2)
    n = 3000
    x, y = origin + np.floor(rng.random(n) * 320.0) / 4.0, origin + rng.random(n) * 70.0
    taken, flags, _ = chain(exe, [(x, y, rng.normal(50.0, 3.0, n))], [(10, 20, 0.8)])
    assert taken == ok and flags == 0 and (chain.groups > 0) == ok


@pytest.mark.parametrize("tiles,planned", [(31, True), (33, False)])
def test_too_many_windows(exe, tiles, planned):
    """A batch of 2^31 windows and more, which the tree chain refuses, is not this
    chain's either (seen by the scratch it asks for; the device has 2 MB)."""
    c = np.array([1.0, 40_000.0]), np.array([1.0, 40_000.0]), np.array([1.0, 2.0])
    boxes = [(0.0, 40_900.0, 0.0, 40_900.0)] * tiles  # 8181 x 8181 windows
    taken, _, _ = chain(exe, [c] * tiles, [(10, 0, 0.5)] * tiles, poke=3, boxes=boxes)
    assert not taken and (chain.largest > 1 << 30) == planned


@pytest.mark.parametrize("poke", [4, 5])
def test_full_lists(exe, poke):
    """Shares of the lists that one block nearly fills, for the bins and for the heavy
    stretches alone: handed on, and the launches behind do nothing."""
    c, p = heavy_cloud(on_edges=100_000), (10, 20, 0.8)
    taken, flags, _ = chain(exe, [c], [p], poke=poke)
    assert not taken and flags & 32 and chain.after == 0
