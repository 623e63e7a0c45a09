"""The single-component step without Shan-Chen force against the oracle, bit
for bit: one site short of and past a wave, rows shorter and longer than a
wave, solid lines, and a lattice past the cached size."""
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
@pytest.mark.parametrize("dq,n", [((3, 19), (2, 2, 2)), ((3, 19), (3, 3, 7)), ((3, 19), (5, 13, 1000)),
                                  ((3, 19), (9, 8, 64)), ((3, 19), (33, 20, 41)),
                                  ((3, 19), (96, 97, 98)), ((2, 9), (2, 2)), ((2, 9), (13, 5)),
                                  ((2, 9), (64, 64)), ((2, 9), (3, 700)), ((1, 3), (63,)),
                                  ((1, 3), (513,)), ((1, 5), (65,))], ids=str)
@pytest.mark.parametrize("form", ["SecondOrder", "ThirdOrder", "BDist2"])
@pytest.mark.parametrize("solid", [False, True])
def test_single_component_equals_oracle(D, dq, n, form, solid):
    from oracle.oracle import Oracle
    d, q = dq
    rng = np.random.default_rng(sum(n))
    p = dict(d=d, q=q, gn=list(n), components=1, tau=[0.8], eqDistForm=form,
             globalAcc=[1e-5] + [0.0] * (d - 1), fluidInit=["EqDistPerturb"],
             fluidDensities=[[1.0]], fluidPerturb=[0.02], randomReseed=[True], randomSeed=[11])
    if solid:
        p["maskArray"] = (rng.random(n) < 0.3).astype(np.int32)
        p["maskArray"].reshape(-1)[: p["maskArray"].size // 3] = 1  # lines of solid sites
    a, o = D.Lattice.from_params(p), Oracle.from_params(p)
    a.step(4)
    o.run(4)
    x, y = a.population(0), o.population(0)
    assert np.array_equal(x.view(np.uint64), y.view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(2, 2), (5, 3), (8, 8), (23, 9), (24, 25), (64, 64), (128, 128),
                               (129, 121), (256, 250), (300, 300), (2000, 3)], ids=str)
@pytest.mark.parametrize("form", ["SecondOrder", "BDist2"])
@pytest.mark.parametrize("solid", [False, True])
def test_several_steps_in_one_launch_equal_oracle(D, n, form, solid):
    """Step counts below, at and past a launch's eight or four steps, eager and
    from a graph, on lattices smaller than a workgroup's 24 x 24 sites, of whole
    tiles, and with tiles over the end of an axis."""
    from oracle.oracle import Oracle
    rng = np.random.default_rng(n[0])
    p = dict(d=2, q=9, gn=list(n), components=1, tau=[0.9], eqDistForm=form,
             globalAcc=[0.0, 1e-5], fluidInit=["EqDistPerturb"], fluidDensities=[[1.0]],
             fluidPerturb=[0.02], randomReseed=[True], randomSeed=[12])
    if solid:
        p["maskArray"] = (rng.random(n) < 0.1).astype(np.int32)
    a, o = D.Lattice.from_params(p), Oracle.from_params(p)
    done = 0
    for k, graph in ((3, False), (8, False), (13, False), (39, True)):
        a.step(k, graph=graph)
        done += k
    o.run(done)
    x, y = a.population(0), o.population(0)
    assert np.array_equal(x.view(np.uint64), y.view(np.uint64))
