"""Batches at the sizes where the heavy classes' items per lane and the
Polyhedron walks' tiles change, against the per-query kernels (bit for bit,
for every launch shape and for the no-allocation entry)."""
import ctypes

import numpy as np
import pytest

from vecgeom_amd import batch as B
from vecgeom_amd import geometry as G
from vecgeom_amd import queries as Q
from vecgeom_amd import workloads as W

pytestmark = pytest.mark.gpu

NAMES = ("Polyhedron", "Polycone", "Cone")


@pytest.mark.parametrize("n", [1, 257, 65535, 131073, 530001])
def test_batch_tiles(n):
    import torch
    Q.init(0)
    rng = np.random.Generator(np.random.Philox(4242))
    zoo = dict(W.zoo_shapes())
    xfs = [W.random_placement(rng) for _ in NAMES]
    geom, ids, _ = G.single_shape_geometry([zoo[k] for k in NAMES], xfs)
    tasks, want = [], []
    for k, (pid, xf) in enumerate(zip(ids, xfs)):
        inp = W.shape_inputs(geom.placed_extent(pid), xf, n, seed=31 + k)
        t = lambda a: tuple(torch.from_numpy(np.ascontiguousarray(a[i])).to("cuda:0") for i in range(3))
        p, d, lp, ld = t(inp["p"]), t(inp["d"]), t(inp["lp"]), t(inp["ld"])
        tasks += [B.Task(pid, B.DISTANCE_TO_IN, p, d), B.Task(pid, B.DISTANCE_TO_OUT, lp, ld),
                  B.Task(pid, B.PLACED_DISTANCE_TO_OUT, p, d), B.Task(pid, B.INSIDE, p)]
        want += [Q.distance_to_in(geom, pid, p, d), Q.distance_to_out(geom, pid, lp, ld),
                 Q.placed_distance_to_out(geom, pid, p, d), Q.inside(geom, pid, p)]
    same = lambda: all(torch.equal(a.out.view(torch.int64) if a.out.dtype == torch.float64 else a.out,
                                   b.view(torch.int64) if b.dtype == torch.float64 else b)
                       for a, b in zip(tasks, want))
    batch = B.Batch(geom, tasks)
    for it, blocks in ((1, 0), (2, 0), (4, 256)):
        batch.set_launch(it, blocks)
        for t in tasks:
            t.out.fill_(77)
        batch.run()
        torch.cuda.synchronize()
        assert same(), (it, blocks)
    for t in tasks:
        t.out.fill_(77)
    arr = (B.CQueryTask * len(tasks))(*[t.c() for t in tasks])
    from vecgeom_amd import capi
    capi.register({"vg_batch_run_noalloc": [B.c_vp, ctypes.POINTER(B.CQueryTask), ctypes.c_int32, B.c_vp]})
    capi.call("vg_batch_run_noalloc", geom.handle, arr, len(tasks), B._stream())
    torch.cuda.synchronize()
    assert same(), "no-allocation entry"
    batch.free()
    geom.free()
