"""The one-launch D2Q9 Shan-Chen step (tiles of 4 x 16 sites) against the
oracle, bit for bit: lattices smaller than a tile, whole tiles, tiles over the
end of an axis, one to four components, with and without solids."""
import numpy as np
import pytest


@pytest.fixture(scope="module")
def D():
    import dlbc_amd
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    return dlbc_amd


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(2, 2), (3, 17), (4, 16), (5, 15), (8, 33), (33, 70), (64, 64),
                               (61, 257)], ids=str)
@pytest.mark.parametrize("nc,form", [(1, "BDist2"), (2, "SecondOrder"), (2, "BDist2"),
                                     (3, "ThirdOrder"), (4, "BDist2")])
@pytest.mark.parametrize("solid", [False, True])
def test_tile_step_equals_oracle(D, n, nc, form, solid):
    from oracle.oracle import Oracle
    rng = np.random.default_rng(100 * nc + n[0])
    g = rng.uniform(0.5, 2.0, (nc, nc))
    p = dict(d=2, q=9, gn=list(n), components=nc, tau=list(rng.uniform(0.8, 1.3, nc)),
             eqDistForm=form, gcc=((g + g.T) / 2).tolist(), gwc=list(rng.uniform(-0.2, 0.2, nc)),
             enableShanChen=True, psiForm="Exponential", globalAcc=[1e-5, 0.0],
             bodyForce=[[0.0, 1e-6]] * nc, fluidInit=["EqDistPerturb"] * nc,
             fluidDensities=[[v] for v in rng.uniform(0.2, 0.8, nc)], fluidPerturb=[0.02] * nc,
             randomReseed=[True] * nc, randomSeed=list(range(31, 31 + nc)))
    if solid:
        p["maskArray"] = (rng.random(n) < 0.15).astype(np.int32)
    a, o = D.Lattice.from_params(p), Oracle.from_params(p)
    o.set_body_force(p["bodyForce"])
    a.step(3)
    a.step(33, graph=True)
    o.run(36)
    for f in range(nc):
        x, y = a.population(f), o.population(f)
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), f
