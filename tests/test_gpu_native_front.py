"""The native front of queries.py (csrc/py_queries.cpp) against the same
queries through the Python checks and ctypes: outputs, given outputs, optional
arguments, lists for tuples, empty baskets, another stream, and the
refusals."""
import os

import numpy as np
import pytest

from vecgeom_amd import geometry as G
from vecgeom_amd import queries as Q
from vecgeom_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def world():
    Q.init(0)
    if not os.path.exists(Q._FRONT_PATH):
        pytest.skip("the native front is not built here")
    assert Q._load_front(), "the native front is built and does not load"
    xf = W.random_placement(np.random.Generator(np.random.Philox(88)))
    geom, ids, _ = G.single_shape_geometry([dict(W.zoo_shapes())["Tube"]], [xf])
    yield geom, ids[0], xf
    geom.free()


def inputs(world, n):
    import torch
    geom, pid, xf = world
    inp = W.shape_inputs(geom.placed_extent(pid), xf, n, seed=5)
    t = lambda k: tuple(torch.from_numpy(np.ascontiguousarray(inp[k][i])).to("cuda:0") for i in range(3))
    sm = torch.rand(n, dtype=torch.float64, device="cuda:0") * 100
    return t("p"), t("d"), t("lp"), t("ld"), sm


def everything(geom, pid, p, d, lp, ld, sm):
    import torch
    n = p[0].numel()
    nxt = torch.full((n,), 9, dtype=torch.int32, device="cuda:0")
    out = [Q.contains(geom, pid, p), Q.inside(geom, pid, p), Q.unplaced_contains(geom, pid, lp),
           Q.distance_to_in(geom, pid, p, d), Q.distance_to_in(geom, pid, p, d, sm),
           Q.distance_to_out(geom, pid, lp, ld, sm, next_node=nxt), nxt, Q.placed_distance_to_out(geom, pid, p, d),
           Q.safety_to_in(geom, pid, p), Q.safety_to_out(geom, pid, lp),
           Q.safety_to_out(geom, pid, lp, out=torch.zeros(n, dtype=torch.float64, device="cuda:0"))]
    nrm, valid = Q.normal(geom, pid, lp)
    t, nrm2, valid2, convex = Q.distance_to_out_normal(geom, pid, lp, ld, sm)
    return out + list(nrm) + [valid, t] + list(nrm2) + [valid2, convex]


@pytest.mark.parametrize("n", [0, 1, 1000])
@pytest.mark.parametrize("as_list", [False, True])
def test_same_as_python_path(world, monkeypatch, n, as_list):
    import torch
    geom, pid, _ = world
    args = [list(a) if as_list and isinstance(a, tuple) else a for a in inputs(world, n)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = everything(geom, pid, *args)
    side.synchronize()
    monkeypatch.setattr(Q, "_native", lambda *a, **k: None)
    want = everything(geom, pid, *args)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape and a.device == b.device
        assert torch.equal(a.view(torch.uint8) if n else a, b.view(torch.uint8) if n else b)


def test_refusals(world):
    import torch
    geom, pid, _ = world
    p, d, lp, ld, sm = inputs(world, 64)
    out = torch.empty(64, dtype=torch.uint8, device="cuda:0")
    assert Q.contains(geom, pid, p, out=out) is out
    strided = tuple(torch.zeros(128, dtype=torch.float64, device="cuda:0")[::2] for _ in range(3))
    for call in (lambda: Q.contains(geom, pid, strided), lambda: Q.contains(geom, pid, tuple(a.cpu() for a in p)),
                 lambda: Q.contains(geom, pid, tuple(a.float() for a in p)), lambda: Q.contains(geom, pid, p[:2]),
                 lambda: Q.contains(geom, pid, p, out=out[:63]), lambda: Q.inside(geom, pid, p, out=out),
                 lambda: Q.distance_to_in(geom, pid, p, tuple(a[:32] for a in d)),
                 lambda: Q.distance_to_in(geom, pid, p, d, sm[:3]),
                 lambda: Q.distance_to_out(geom, pid, lp, ld, next_node=out)):
        with pytest.raises(ValueError):
            call()
    with pytest.raises(RuntimeError, match="vg_contains failed"):
        Q.contains(geom, 10 ** 6, p)
