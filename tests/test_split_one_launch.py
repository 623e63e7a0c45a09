"""The split schedule's one-launch step (psi and collide workgroups in one
launch, in the order of a table): the order on the CPU; on the GPU the same
bits as the oracle and as two launches, at the smallest lattices that take it
and with planes cut into strips."""
import numpy as np
import pytest


@pytest.mark.parametrize("n", [(2, 2, 2), (2, 3, 4), (3, 3, 3), (5, 7, 9), (100, 4, 4), (1000, 2, 2),
                               (4, 4, 1000), (64, 64, 64), (12, 10, 128), (6, 40, 256),
                               (31, 97, 65), (17, 64, 512), (9, 260, 127), (9, 300, 301),
                               (2, 5000, 7), (3, 700, 129), (7, 5, 3000), (4, 256, 256)])
@pytest.mark.parametrize("sites", [128, 256])
def test_order_visits_every_block_and_never_waits_for_a_later_one(n, sites):
    import dlbc_amd as D
    assert D.lib().dlbc_selftest_split_order(*n, sites) == 0


@pytest.fixture(scope="module")
def D():
    import dlbc_amd
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible")
    return dlbc_amd


def _params(n, form, solid):
    rng = np.random.default_rng(sum(n))
    p = dict(d=3, q=19, gn=list(n), components=2, tau=[1.0, 0.9], eqDistForm=form,
             gcc=[[0.0, 3.6], [3.6, 0.0]], enableShanChen=True, psiForm="Exponential",
             fluidInit=["EqDistPerturb"] * 2, fluidDensities=[[0.7], [0.6]],
             fluidPerturb=[0.02, 0.02], randomReseed=[True] * 2, randomSeed=[5, 6])
    if solid:
        p["gwc"] = [0.1, -0.1]
        p["maskArray"] = (rng.random(n) < 0.1).astype(np.int32)
    return p


def _same(a, b, what):
    for f in range(2):
        x, y = a.population(f), b.population(f)
        assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), (what, f)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(70, 90, 61), (2, 1250, 131), (16, 200, 128), (15, 211, 131),
                               (41, 3, 2620)], ids=str)
@pytest.mark.parametrize("form,solid", [("BDist2", True), ("SecondOrder", False)])
def test_f64_equals_oracle(D, n, form, solid):
    from oracle.oracle import Oracle
    p = _params(n, form, solid)
    g, o = D.Lattice.from_params(p, schedule="split"), Oracle.from_params(p)
    g.step(3)
    o.run(3)
    _same(g, o, n)


@pytest.mark.gpu
@pytest.mark.parametrize("storage,n", [("f64", (15, 211, 131)), ("f32_shift", (70, 150, 149)),
                                       ("f32_shift", (13, 470, 256)), ("f16_shift", (24, 256, 256))],
                         ids=str)
@pytest.mark.parametrize("solid", [True, False])
def test_equals_two_launches(D, storage, n, solid):
    """Any block order keeps two launches per step; both give the same bits,
    also in turn, over odd step counts, from a graph and where no collide wave
    waits for the psi it reads (each computes it)."""
    p = _params(n, "BDist2", solid)
    a, b = (D.Lattice.from_params(p, storage=storage, schedule="split") for _ in range(2))
    b.set_block_order(8)
    for k in (3, 1, 4):
        a.step(k)
        b.step(k)
    _same(a, b, "steps")
    a.set_block_order(8)
    a.step(1)
    a.set_block_order(0)
    a.step(33, graph=True)
    b.step(34)
    _same(a, b, "block order, then a graph")
    a._check(D.lib().dlbc_selftest_set_psi_polls(a.h, 0), "polls")
    a.step(1)
    b.step(1)
    _same(a, b, "no waiting")


@pytest.mark.gpu
@pytest.mark.parametrize("storage,solid", [("f32_shift", False), ("f32_shift", True),
                                           ("f16_shift", False)])
def test_batch_in_one_launch_equals_lattices_alone(D, storage, solid):
    """A batch large enough for one launch per step: eager, graph and odd step
    counts, and a member whose Shan-Chen force goes off and on in between."""
    sizes = [(70, 83, 91), (4, 4, 4), (64, 96, 128), (33, 70, 31)]
    ps = [_params(n, "BDist2", solid) for n in sizes]
    alone, members = ([D.Lattice.from_params(p, storage=storage) for p in ps] for _ in range(2))
    batch = D.Batch(members)
    batch.set_config(8, 64, 512, 2)

    def params(lat, p, on):
        lat.set_params(p["tau"], p["gcc"], p.get("gwc"), None, None, p["eqDistForm"], "Exponential",
                       on)

    for k, graph, on in ((4, True, True), (3, False, True), (2, True, False), (1, False, False),
                         (6, True, True), (1, True, True)):
        for lats in (alone, members):
            params(lats[2], ps[2], on)
        batch.step(k, graph=graph)
        for lat in alone:
            lat.step(k)
        batch.synchronize()
    for a, b, n in zip(alone, members, sizes):
        _same(a, b, n)


@pytest.mark.gpu
@pytest.mark.parametrize("n,kernels", [((21000, 4, 4), 2), ((5, 13, 16385), 2), ((2600, 8, 16), 1),
                                       ((6, 9, 16384), 2), ((5, 13, 16384), 1)], ids=str)
def test_thin_planes_and_long_rows_equal_oracle(D, n, kernels):
    """Planes of fewer sites than a block and rows of more than 128 blocks take
    two launches; planes of one block and, in a large lattice, rows of 128 are
    the smallest and the longest that take one."""
    from oracle.oracle import Oracle
    p = _params(n, "BDist2", False)
    g, o = D.Lattice.from_params(p, schedule="split"), Oracle.from_params(p)
    assert len(g.step_timed(2)[1]) == kernels
    g.step(1)
    o.run(3)
    _same(g, o, n)


# 6,187 blocks of 256 sites: past the 6,000 from which a batch takes one launch
# (that it does is counted in test_host_calls.py), with a member of one block
BATCH = [(70, 83, 91), (4, 4, 4), (64, 96, 160), (33, 70, 31)]


@pytest.mark.gpu
@pytest.mark.parametrize("storage,solid", [("f32_shift", False), ("f32_shift", True),
                                           ("f16_shift", False)])
def test_large_batch_equals_lattices_alone(D, storage, solid):
    """One launch per step over all members: eager, graph and odd step counts, a
    member whose Shan-Chen force goes off and on in between, one with
    self-coupling, and one of other solids than its neighbours."""
    ps = [_params(n, ("BDist2", "SecondOrder")[k % 2], solid and k != 3)
          for k, n in enumerate(BATCH)]
    ps[0]["gcc"] = [[0.4, 3.0], [3.0, -0.3]]
    alone, members = ([D.Lattice.from_params(p, storage=storage) for p in ps] for _ in range(2))
    for lat in alone:
        lat.set_block_order(8)  # two launches
    batch = D.Batch(members)
    batch.set_config(8, 64, 512, 2)
    for k, graph, on in ((4, True, True), (3, False, True), (2, True, False), (1, False, False),
                         (7, True, True), (5, True, True), (1, True, True)):
        for lats in (alone, members):
            p = ps[2]
            lats[2].set_params(p["tau"], p["gcc"], p.get("gwc"), None, None, p["eqDistForm"],
                               "Exponential", on)
        batch.step(k, graph=graph)
        for lat in alone:
            lat.step(k)
        batch.synchronize()
        for a, b, n in zip(alone, members, BATCH):
            _same(a, b, (n, k))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(70, 90, 61), (16, 200, 128)], ids=str)
@pytest.mark.parametrize("solid", [True, False])
def test_f64_self_coupling_equals_oracle(D, n, solid):
    from oracle.oracle import Oracle
    p = dict(_params(n, "BDist2", solid), gcc=[[0.4, 3.0], [3.0, -0.3]])
    g, o = D.Lattice.from_params(p, schedule="split"), Oracle.from_params(p)
    assert list(g.step_timed(1)[1]) == ["split_one_launch"]
    g.step(2)
    o.run(3)
    _same(g, o, n)
