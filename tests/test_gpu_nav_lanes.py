"""Navigation launches at the sizes where the tracks per wave change
(LanesShift: 1 track a wave up to 2,048 tracks, then 2, 4, ...), over a
volume with more daughters than one mask word holds, against the oracle."""
import numpy as np
import pytest

import pyoracle as po
from conftest import same
from test_daughter_index import many_geometry, tracks
from vecgeom_amd import geometry as G
from vecgeom_amd import nav as N

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[(64, "boxes"), (65, "tubes"), (150, "mixed")], ids=lambda p: f"{p[1]}{p[0]}")
def world(request, oracle):
    from vecgeom_amd import queries as Q
    Q.init(0)
    flat, half = many_geometry(*request.param)
    geom = G.DeviceGeometry(flat)
    yield geom, po.Nav(oracle, flat), half
    geom.free()


@pytest.mark.parametrize("n", [1, 65, 2048, 2049, 8193])
def test_step_trace_safety(world, n):
    import torch
    geom, O, half = world
    p, d = tracks(n, half, 900 + n)
    t = lambda a: tuple(torch.from_numpy(np.ascontiguousarray(a[i])).to("cuda:0") for i in range(3))
    host = lambda a: a.cpu().numpy()
    tp, td = t(p), t(d)
    lo, pa = O.locate(p, nthreads=8)
    cur = N.locate_points(geom, tp)
    assert (host(cur.level) == lo).all() and (host(cur.path) == pa).all()
    assert same(host(N.get_safety(geom, tp, cur)), O.safety(p, lo, pa, nthreads=8)).all()
    for kind in (N.ABBOX, N.SIMPLE):
        new, step = N.find_next_boundary_and_step(geom, tp, td, cur, navigator=kind)
        ol, op, ob, os_ = O.step(p, d, lo, pa, kind=kind, nthreads=8)
        assert (host(new.level) == ol).all() and (host(new.path) == op).all() and (host(new.boundary) == ob).all()
        assert same(host(step), os_).all()
        r = N.trace_tracks(geom, tp, td, navigator=kind)
        ns, fin, trav, hs = O.trace(p, d, kind=kind, nthreads=8)
        assert (host(r.nsteps) == ns).all() and (r.hash_u64() == hs).all()
        assert same(host(r.travelled), trav).all()
        assert all(same(host(r.final[i]), fin[i]).all() for i in range(3))
