"""Boolean volumes with a Torus operand, which run in kernels of their own:
the union of a Torus with a disjoint operand answers as the two placed shapes
do by themselves."""
import numpy as np
import pytest

from vecgeom_amd import geometry as G
from vecgeom_amd import queries as Q
from vecgeom_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other", ["Box", "Polycone"])
@pytest.mark.parametrize("torus_first", [True, False])
def test_union_with_torus(other, torus_first):
    import torch
    Q.init(0)
    zoo = dict(W.zoo_shapes())
    ident, away = G.Transformation3D(), G.Transformation3D(150.0, 20.0, -30.0)
    # (The left operand sits at the origin, as DistanceToOut takes it.)
    a, b = (zoo["Torus"], zoo[other]) if torus_first else (zoo[other], zoo["Torus"])
    union = G.UnplacedBooleanVolume(G.kUnion, a, ident, b, away)
    geom, ids, _ = G.single_shape_geometry([union, a, b], [ident, ident, away])
    rng = np.random.Generator(np.random.Philox(17))
    n = 4099
    p = rng.uniform(-80.0, 80.0, (3, n))
    p[0, n // 2:] += 150.0
    d = W.isotropic(n, rng)
    t = lambda v: tuple(torch.from_numpy(np.ascontiguousarray(v[i])).to("cuda:0") for i in range(3))
    tp, td = t(p), t(d)
    one = [f(geom, i, *x) for f, x in ((Q.contains, (tp,)), (Q.distance_to_in, (tp, td)), (Q.safety_to_in, (tp,)))
           for i in ids]
    assert torch.equal(one[0], one[1] | one[2])
    assert int(one[1].sum()) > 0 and int(one[2].sum()) > 0
    out = one[0] == 0
    assert torch.equal(one[3][out], torch.minimum(one[4], one[5])[out])
    assert torch.equal(one[6][out], torch.minimum(one[7], one[8])[out])
    # From inside one operand, the exit of the union is that operand's.
    for k, (xf, i) in enumerate(((ident, ids[1]), (away, ids[2]))):
        held = one[1 + k] != 0
        local = t(W.master_to_local(xf, p)) if k else tp
        whole = Q.distance_to_out(geom, ids[0], tp, td)[held]
        alone = Q.distance_to_out(geom, i, local, td)[held]
        assert torch.allclose(whole, alone, rtol=0, atol=1e-7)  # a union advances by 1e-8 mm pushes
    geom.free()
