"""Rays aimed at a small cluster of daughters from far away, against the
oracle.  The navigator searches a ray in growing stretches from where it
enters the box of all daughters; at the far end of a long way the first
stretch can be shorter than the spacing of floats there, and the search must
go on all the same.  The navigator runs in a child process with a time limit,
so that a search without end fails the test instead of stopping it."""
import math
import multiprocessing as mp

import numpy as np
import pytest

import pyoracle as po
from conftest import same
from test_nav_hostcheck import _HostNav
from vecgeom_amd import geometry as G
from vecgeom_amd import workloads as W

KINDS = (0, 1, 3)


def cluster(n, size, half, centre=(0.0, 0.0, 0.0)):
    """A world box of half-width `half` with n boxes, orbs and tubes of
    half-width about `size` on a grid around `centre`; returns the geometry
    and half the cluster's side."""
    gm = G.GeoManager()
    world = G.LogicalVolume("world", G.UnplacedBox(half, half, half), gm)
    shapes = [G.LogicalVolume("box", G.UnplacedBox(size, size, size), gm),
              G.LogicalVolume("orb", G.UnplacedOrb(size), gm),
              G.LogicalVolume("tube", G.UnplacedTube(0.3 * size, size, size, 0.0, 2 * math.pi), gm)]
    m = math.ceil(n ** (1 / 3))
    for i in range(n):
        at = [c + 2.5 * size * (k - (m - 1) / 2) for c, k in zip(centre, (i % m, i // m % m, i // (m * m)))]
        world.PlaceDaughter(f"d{i}", shapes[i % 3], G.Transformation3D(*at))
    gm.SetWorld(world.Place("world"))
    return gm.CloseGeometry(), 1.25 * size * m


def aimed(n, reach, centre, distance, seed):
    """n tracks at about `distance` from the cluster, aimed at points of a box
    around it somewhat larger than it is; a third of them along an axis."""
    rng = np.random.Generator(np.random.Philox(seed))
    c = np.array(centre)[:, None]
    target = c + rng.uniform(-1.3 * reach, 1.3 * reach, (3, n))
    away = W.isotropic(n, rng)
    k = n // 3
    away[:, :k] = 0.0
    away[rng.integers(0, 3, k), np.arange(k)] = rng.choice((-1.0, 1.0), k)
    p = target + away * distance * rng.uniform(0.5, 1.0, n)
    d = target - p
    return p, d / np.sqrt((d * d).sum(0))


def _answers(lib, flat, p, d):
    nav = po.Nav(lib, flat)
    level, path = nav.locate(p, nthreads=4)
    out = [level, path, nav.safety(p, level, path, nthreads=4)]
    for kind in KINDS:
        out += nav.step(p, d, level, path, kind=kind, nthreads=4)
    for kind in (0, 1):
        out += nav.trace(p, d, kind=kind, max_steps=64, nthreads=4)
    return out


def _child(pipe, flat, p, d):
    pipe.send(_answers(_HostNav(), flat, p, d))


def within(seconds, flat, p, d):
    """The host build's answers, or None after `seconds`."""
    mine, other = mp.Pipe(duplex=False)
    child = mp.get_context("fork").Process(target=_child, args=(other, flat, p, d))
    child.start()
    other.close()
    out = None
    try:
        if mine.poll(seconds):
            out = mine.recv()
    except EOFError:
        pass
    child.kill()
    child.join()
    return out


# Half-width of the daughters (mm) and distance in cluster widths.
SCALES = [1e-3, 1.0, 1e3]
RATIOS = [1.0, 30.0, 1e3, 1e4, 3e4, 1e5, 1e6, 1e7]


@pytest.mark.parametrize("n", [3, 64, 65])
@pytest.mark.parametrize("size", SCALES)
@pytest.mark.parametrize("off", [False, True])
def test_far_rays(oracle, n, size, off):
    for i, ratio in enumerate(RATIOS):
        width = 2.5 * size * math.ceil(n ** (1 / 3))
        distance = ratio * width
        centre = (0.4 * distance, -0.2 * distance, 0.1 * distance) if off else (0.0, 0.0, 0.0)
        flat, reach = cluster(n, size, 2.0 * distance + 4 * width, centre)
        p, d = aimed(200, reach, centre, distance, seed=W.SEED_BASE + 300 + i)
        got = within(20, flat, p, d)
        assert got is not None, f"no answer in 20 s: {n} daughters of {size} mm from {distance} mm"
        for k, (x, y) in enumerate(zip(_answers(oracle, flat, p, d), got)):
            assert same(x, y).all(), (n, size, ratio, off, k, int((~same(x, y)).sum()))


@pytest.mark.gpu
@pytest.mark.parametrize("size,ratio", [(1.0, 3e4), (1e-3, 1e6), (1e3, 1e7)])
def test_far_rays_on_the_device(oracle, size, ratio):
    import torch

    from vecgeom_amd import nav as N
    from vecgeom_amd import queries as Q
    Q.init(0)
    width = 10.0 * size
    distance = ratio * width
    flat, reach = cluster(65, size, 2.0 * distance + 4 * width)
    p, d = aimed(500, reach, (0.0, 0.0, 0.0), distance, seed=W.SEED_BASE + 320)
    want = _answers(oracle, flat, p, d)
    assert within(20, flat, p, d) is not None  # the same code ends on the host
    geom = G.DeviceGeometry(flat)
    t = lambda a: tuple(torch.from_numpy(np.ascontiguousarray(a[i])).to("cuda:0") for i in range(3))
    tp, td = t(p), t(d)
    cur = N.locate_points(geom, tp)
    got = [cur.level, cur.path, N.get_safety(geom, tp, cur)]
    for kind in KINDS:
        new, step = N.find_next_boundary_and_step(geom, tp, td, cur, navigator=kind)
        got += [new.level, new.path, new.boundary, step]
    for kind in (0, 1):
        r = N.trace_tracks(geom, tp, td, navigator=kind, max_steps=64)
        got += [r.nsteps, torch.stack(r.final), r.travelled, r.hash]
    torch.cuda.synchronize()
    for k, (x, y) in enumerate(zip(want, got)):
        y = y.cpu().numpy()
        assert same(x, y.view(np.uint64) if x.dtype == np.uint64 else y).all(), k  # torch holds the hash signed
    geom.free()
