"""Rays aimed at daughters of all twelve shapes: the navigators that look only
at the daughters their index names, against the oracle and against the same
code without indexes.  The Parallelepiped's DistanceToIn compares a sheared
safety with the step limit, so its answer can depend on the limit, and the
limit on the order of the walk."""
import ctypes
import math

import numpy as np
import pytest

import pyoracle as po
from conftest import same
from test_nav_hostcheck import _HostNav
from vecgeom_amd import geometry as G
from vecgeom_amd import workloads as W

SHAPES = dict(W.zoo_shapes())
KINDS = (0, 1, 3)
SETS = {
    "sheared": ["Box", "Parallelepiped"],
    "planar": ["Box", "Parallelepiped", "Trd", "Trapezoid", "Polyhedron"],
    # (the Torus's and the Sphere's distances differ from the oracle's in the
    # last places; they are compared with the walk without indexes only)
    "exact": [k for k in SHAPES if k not in ("Torus", "Sphere")],
    "all": list(SHAPES),
}


def world_of(names, n, half, seed):
    """n daughters of the shapes in turn at random places (overlaps and all)
    and rotations in a world box of half-width `half`."""
    rng = np.random.Generator(np.random.Philox(seed))
    gm = G.GeoManager()
    world = G.LogicalVolume("world", G.UnplacedBox(half, half, half), gm)
    lv = {k: G.LogicalVolume(k, SHAPES[k], gm) for k in names}
    at = rng.uniform(-0.8 * half, 0.8 * half, (n, 3))
    for i in range(n):
        k = names[i % len(names)]
        world.PlaceDaughter(f"{k}{i}", lv[k], G.Transformation3D(*at[i], *W.random_rotation(rng)))
    gm.SetWorld(world.Place("world"))
    return gm.CloseGeometry(), at.T


def aimed(n, half, centres, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    p = rng.uniform(-half, half, (3, n))
    to = centres[:, rng.integers(0, centres.shape[1], n)] + rng.normal(0.0, 20.0, (3, n))
    p[:, : n // 4] = to[:, : n // 4] + rng.normal(0.0, 40.0, (3, n // 4))  # near them, or inside
    d = to - p
    return p, d / np.sqrt((d * d).sum(0))


@pytest.fixture(scope="module")
def hostnav():
    return _HostNav()


@pytest.mark.parametrize("names", sorted(SETS))
@pytest.mark.parametrize("n,half", [(8, 500.0), (24, 600.0), (24, 3000.0), (80, 1500.0)])
def test_aimed_rays(oracle, hostnav, names, n, half):
    flat, centres = world_of(SETS[names], n, half, W.SEED_BASE + 400 + n)
    H = po.Nav(hostnav, flat)
    if names == "all":
        want = po.Nav(hostnav, flat)
        hostnav.lib.navhost_drop_indexes(ctypes.c_void_p(want.h))
    else:
        want = po.Nav(oracle, flat)
    p, d = aimed(20000, half, centres, 17 + n)
    world_only = want.locate(p, nthreads=8)[0] == 1
    level = np.ones(p.shape[1], np.int32)  # in the world, as the tracks that a step has left there
    path = np.full((want.depth, p.shape[1]), -1, np.int32)
    path[0] = flat.world
    for kind in KINDS:
        for pstep in (math.inf, 40.0):
            a = want.step(p, d, level, path, pstep=pstep, kind=kind, nthreads=8)
            b = H.step(p, d, level, path, pstep=pstep, kind=kind, nthreads=8)
            for x, y in zip(a, b):
                bad = ~same(x, y)
                bad = bad.any(0) if bad.ndim > 1 else bad
                assert not bad.any(), (names, kind, pstep, int(bad.sum()), int((bad & world_only).sum()))
    assert same(want.safety(p, level, path, nthreads=8), H.safety(p, level, path, nthreads=8)).all()
    for kind in (0, 1):
        for x, y in zip(want.trace(p, d, kind=kind, nthreads=8), H.trace(p, d, kind=kind, nthreads=8)):
            assert same(x, y).all(), (names, kind)


@pytest.mark.parametrize("names,n", [("exact", 30), ("all", 80), ("grazed", 70)])
@pytest.mark.parametrize("how", ["float", 1.0 + 4.9e-7, 1.0 - 4.9e-7, 1.0 + 1e-3, 1.0 + 1e-9])
def test_directions_near_unit_length(hostnav, names, n, how):
    """Directions that were stored as float, or a little longer or shorter
    than a unit vector, up to the length where the index is left aside and
    beyond: the index changes nothing.  "grazed": rays along an axis that pass
    round shapes of half-width 50 mm at a distance to which such a direction
    shifts their tangents (from 10^5 mm, 10^10 * 1e-6 / 100 = 100 mm)."""
    half = 100000.0 if names == "grazed" else 2000.0
    round_ones = ["Orb", "Tube", "Cone", "Paraboloid", "Torus", "Polycone"]
    flat, centres = world_of(round_ones if names == "grazed" else SETS[names], n, half, W.SEED_BASE + 460)
    H, want = po.Nav(hostnav, flat), po.Nav(hostnav, flat)
    hostnav.lib.navhost_drop_indexes(ctypes.c_void_p(want.h))
    p, d = aimed(60000, half, centres, 23)
    if names == "grazed":  # along an axis, so that one coordinate decides
        rng = np.random.Generator(np.random.Philox(29))
        n = p.shape[1]
        axis, sign = rng.integers(0, 3, n), rng.choice((-1.0, 1.0), n)
        c = centres[:, rng.integers(0, centres.shape[1], n)]
        d = np.zeros((3, n))
        d[axis, np.arange(n)] = sign
        p = c.copy()
        p[axis, np.arange(n)] = -sign * 0.99 * half
        p[(axis + 1) % 3, np.arange(n)] += (50.0 + rng.uniform(-1.0, 40.0, n)) * rng.choice((-1.0, 1.0), n)
    d = d.astype(np.float32).astype(np.float64) if how == "float" else d * how
    level, path = want.locate(p, nthreads=8)
    for kind in KINDS[:2]:
        for x, y in zip(want.step(p, d, level, path, kind=kind, nthreads=8),
                        H.step(p, d, level, path, kind=kind, nthreads=8)):
            assert same(x, y).all(), (kind, int((~same(x, y)).sum()))
        for x, y in zip(want.trace(p, d, kind=kind, nthreads=8), H.trace(p, d, kind=kind, nthreads=8)):
            assert same(x, y).all(), (kind, int((~same(x, y)).sum()))


@pytest.mark.parametrize("n", [31, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("scale", [1e-3, 1.0, 1e4])
def test_safety_among_safe_daughters(oracle, hostnav, n, scale):
    """Orbs and boxes turned about z, from the number of daughters where the
    safety takes the index on: points near them, in them, and beyond."""
    rng = np.random.Generator(np.random.Philox(W.SEED_BASE + 470 + n))
    gm = G.GeoManager()
    half = 400.0 * scale
    world = G.LogicalVolume("world", G.UnplacedBox(half, half, half), gm)
    lv = [G.LogicalVolume("box", G.UnplacedBox(10 * scale, 30 * scale, 5 * scale), gm),
          G.LogicalVolume("orb", G.UnplacedOrb(12 * scale), gm)]
    for i in range(n):
        f = rng.uniform(0, 2 * math.pi)
        c, s = math.cos(f), math.sin(f)
        at = rng.uniform(-0.6, 0.6, 3) * half
        turn = [c, -s, 0.0, s, c, 0.0, 0.0, 0.0, 1.0] if i % 2 == 0 else []
        world.PlaceDaughter(f"d{i}", lv[i % 2], G.Transformation3D(*at, *turn))
    gm.SetWorld(world.Place("world"))
    flat = gm.CloseGeometry()
    O, H = po.Nav(oracle, flat), po.Nav(hostnav, flat)
    p = rng.uniform(-1.0, 1.0, (3, 8000)) * half
    p[:, :1000] *= 1e3  # outside the world
    p[0, 1000:1200] = half * (1 - rng.uniform(0, 1e-9, 200))  # at its wall
    level = np.ones(p.shape[1], np.int32)
    path = np.full((O.depth, p.shape[1]), -1, np.int32)
    path[0] = flat.world
    assert same(O.safety(p, level, path, nthreads=8), H.safety(p, level, path, nthreads=8)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("names,n", [("planar", 4), ("planar", 33), ("exact", 20), ("exact", 101), ("boxes", 65)])
def test_steps_on_the_device(oracle, names, n):
    """Launches on both sides of the sizes and numbers of daughters where a
    step takes the index, the loop, and full waves."""
    import torch

    from vecgeom_amd import nav as N
    from vecgeom_amd import queries as Q
    Q.init(0)
    flat, centres = world_of(["Box"] if names == "boxes" else SETS[names], n, 1200.0, W.SEED_BASE + 480 + n)
    O, geom = po.Nav(oracle, flat), G.DeviceGeometry(flat)
    host = lambda a: a.cpu().numpy()
    for tracks in (200, 32767, 32768):
        p, d = aimed(tracks, 1200.0, centres, 31)
        t = lambda a: tuple(torch.from_numpy(np.ascontiguousarray(a[i])).to("cuda:0") for i in range(3))
        tp, td = t(p), t(d)
        level, path = O.locate(p, nthreads=8)
        cur = N.locate_points(geom, tp)
        assert (host(cur.level) == level).all() and (host(cur.path) == path).all()
        assert same(host(N.get_safety(geom, tp, cur)), O.safety(p, level, path, nthreads=8)).all()
        for kind in KINDS:
            new, step = N.find_next_boundary_and_step(geom, tp, td, cur, navigator=kind)
            want = O.step(p, d, level, path, kind=kind, nthreads=8)
            for x, y in zip(want, (new.level, new.path, new.boundary, step)):
                assert same(x, host(y)).all(), (tracks, kind)
    geom.free()
