"""The navigator's daughter index (csrc/vg_daughter_index.hpp): the host build
of the navigation code, which looks only at the daughters the index names,
against the oracle, which looks at all of them.  The geometries have more
daughters than a mask word holds, extents that the index must not take too
tight (phi sections, sheared and turned shapes), and a volume whose
daughters' matrices are no rotations; the tracks include directions that
are not unit vectors, axis-parallel ones, and points far outside the
daughters."""
import math

import numpy as np
import pytest

import pyoracle as po
from conftest import same
from test_nav_hostcheck import _HostNav
from vecgeom_amd import geometry as G
from vecgeom_amd import workloads as W

SHAPES = dict(W.zoo_shapes())


def _grid(n, pitch):
    m = int(math.ceil(n ** (1 / 3)))
    at = [((i % m) - (m - 1) / 2, (i // m % m) - (m - 1) / 2, i // (m * m) - (m - 1) / 2) for i in range(n)]
    return [tuple(pitch * v for v in a) for a in at]


def many_geometry(n, kind):
    """A world of n daughters on a grid, each holding an Orb: "boxes" turned
    about z, "mixed" shapes at any rotation, "tubes" with phi sections in
    upright placements, "skewed" ones whose matrix is no rotation."""
    rng = np.random.Generator(np.random.Philox(W.SEED_BASE + 200 + n))
    gm = G.GeoManager()
    pitch = 130.0
    half = pitch * (math.ceil(n ** (1 / 3)) / 2 + 1)
    world = G.LogicalVolume("world", G.UnplacedBox(half, half, half), gm)
    orb = G.LogicalVolume("orb", G.UnplacedOrb(2.0), gm)
    names = ["Box", "Tube", "Trd", "Orb", "Cone", "Parallelepiped", "Trapezoid", "Paraboloid", "Polycone"]
    lv = {}
    for k in names:
        lv[k] = G.LogicalVolume(k, SHAPES[k], gm)
    for j in range(4):  # enough daughters for an index of their own
        lv["Box"].PlaceDaughter(f"orb{j}", orb, G.Transformation3D(-15.0 + 10 * j, 3.0, 0.0))
    for k, t in enumerate(_grid(n, pitch)):
        f = rng.uniform(0, 2 * math.pi)
        c, s = math.cos(f), math.sin(f)
        about_z = [c, -s, 0.0, s, c, 0.0, 0.0, 0.0, 1.0]
        name, r = "Box", about_z
        if kind == "mixed":
            name, r = names[k % len(names)], W.random_rotation(rng)
        elif kind == "tubes":
            name, r = ("Tube", about_z) if k % 3 else ("Trd", [])
        elif kind == "skewed":
            r = [0.9 * v for v in about_z] if k % 2 else about_z
        world.PlaceDaughter(f"{name}{k}", lv[name], G.Transformation3D(*t, *r))
    gm.SetWorld(world.Place("world"))
    return gm.CloseGeometry(), half


def tracks(n, half, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    p = rng.uniform(-half, half, (3, n))
    p[:, : n // 8] *= 0.1
    d = W.isotropic(n, rng)
    k = n // 5
    d[:, :k] = 0.0  # along an axis
    d[rng.integers(0, 3, k), np.arange(k)] = rng.choice((-1.0, 1.0), k)
    return p, d


@pytest.fixture(scope="module")
def hostnav():
    return _HostNav()


@pytest.mark.parametrize("n,kind", [(3, "boxes"), (63, "tubes"), (64, "boxes"), (65, "mixed"), (128, "tubes"),
                                    (150, "mixed"), (70, "skewed")])
def test_index_matches_full_scan(oracle, hostnav, n, kind):
    flat, half = many_geometry(n, kind)
    O, H = po.Nav(oracle, flat), po.Nav(hostnav, flat)
    p, d = tracks(1500, half, 77 + n)
    lo, pa = O.locate(p, nthreads=8)
    lh, ph = H.locate(p, nthreads=8)
    assert (lo == lh).all() and (pa == ph).all()
    assert same(O.safety(p, lo, pa, nthreads=8), H.safety(p, lo, pa, nthreads=8)).all()
    # Directions of other lengths; at 3 some shapes' walks (their skipped
    # sections) take the direction for a unit vector where the oracle does not.
    for scale in (1.0, 1.0 + 1e-7) + ((3.0,) if kind != "mixed" else ()):
        for kind_ in (0, 1):
            for x, y in zip(O.step(p, d * scale, lo, pa, kind=kind_, nthreads=8),
                            H.step(p, d * scale, lo, pa, kind=kind_, nthreads=8)):
                assert same(x, y).all(), (scale, kind_)
    for kind_ in (0, 1):
        for x, y in zip(O.trace(p, d, kind=kind_, nthreads=8), H.trace(p, d, kind=kind_, nthreads=8)):
            assert same(x, y).all(), kind_


def test_safety_and_step_outside_the_daughters(oracle, hostnav):
    """Points of the world far beyond its daughters, and states whose point
    lies outside their volume."""
    flat, half = many_geometry(64, "boxes")
    O, H = po.Nav(oracle, flat), po.Nav(hostnav, flat)
    p, d = tracks(1000, half, 5)
    lo, pa = O.locate(p)
    far = p * np.array([[1e3], [1.0], [-1e4]])
    for q in (far, p + 1e-9, p * 1e9):
        assert same(O.safety(q, lo, pa), H.safety(q, lo, pa)).all()
        for x, y in zip(O.step(q, d, lo, pa, kind=0), H.step(q, d, lo, pa, kind=0)):
            assert same(x, y).all()
