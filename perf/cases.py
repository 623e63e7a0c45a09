"""What a user of this framework has it do, as cases that can be timed.

A DLBC run is a time loop between outputs: some steps, then the fields of the
output files (or of a checkpoint) on the host.  A pass of a case is one such
stretch through the public entry points: `Lattice.step` (or `Batch.step`) and
the fields of that output.  The state lives on from pass to pass, as in a run.

Lattices, parameters and initial states are those of the reference's input
files, of the tests and of bench.py: droplets, spinodal noise, two-fluid
channels with solid spheres, plates; D2Q9 and D3Q19; one, two and three
components; FP64 and the FP32- and FP16-shifted storages; single lattices and
ensembles.
"""
import math

import numpy as np
import torch

import dlbc_amd

LIGHT, DENSE = 0.05, 1.0

# D3Q19 and D2Q9 in the reference's order of velocities.
C3 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0),
      (-1, 1, 0), (0, 1, 1), (0, -1, 1), (1, 0, 1), (1, 0, -1), (1, -1, 0), (-1, -1, 0),
      (0, 1, -1), (0, -1, -1), (-1, 0, 1), (-1, 0, -1)]
W3 = [1 / 3] + [1 / 18] * 6 + [1 / 36] * 12
C2 = [(0, 0), (1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (1, -1), (-1, 1), (-1, -1)]
W2 = [4 / 9] + [1 / 9] * 4 + [1 / 36] * 4


def _case(name, n, components, init, steps, out="density", **more):
    c = {"name": name, "nx": n[0], "ny": n[1], "nz": n[2] if len(n) == 3 else 0,
         "components": components, "storage": "f64", "form": "BDist2", "shan_chen": True,
         "tau": 1.0, "init": init, "solid": "none", "wall_coupling": 0.0, "acceleration": 0.0,
         "steps": steps, "graph": False, "out": out, "lattices": 1}
    c.update(more)
    return c


def listed():
    return [
        # A host program that looks at the mixture after every step (a coupling
        # hook, a live plot): the smallest call, where latency is all.
        _case("hook_2d", (64, 64), 2, "droplet", 1, "colour"),
        # The plain single-fluid D2Q9 run of 64x64 sites with seeded noise, small
        # enough to be replayed from a graph.
        _case("bgk_2d", (64, 64), 1, "noise", 200, "velocity", form="SecondOrder",
              shan_chen=False, graph=True),
        # A two-fluid D2Q9 droplet on a larger, odd lattice: the reference's
        # Laplace and merging-droplet runs at a production size.
        _case("droplet_2d", (321, 257), 2, "droplet", 200),
        # Three immiscible fluids in two dimensions with the default equilibrium's
        # third-order form.
        _case("three_fluids_2d", (192, 192), 3, "noise", 100, form="ThirdOrder"),
        # Flow of one fluid between plates under a body acceleration (Poiseuille),
        # D3Q19, ragged.
        _case("plates_3d", (70, 45, 98), 1, "noise", 100, "velocity", form="SecondOrder",
              shan_chen=False, solid="plates", acceleration=1e-5),
        # The reference's small three-dimensional droplet lattice, replayed from a
        # graph between outputs.
        _case("droplet_3d_small", (32, 32, 32), 2, "droplet", 200, graph=True),
        # Spinodal decomposition from noise, 128^3, the default equilibrium.
        _case("spinodal_3d", (128, 128, 128), 2, "noise", 200, form="SecondOrder"),
        # The two-fluid channel with walls and solid spheres in FP64: the headline
        # workload, between two outputs.
        _case("channel_f64", (256, 256, 256), 2, "halves", 200, solid="spheres",
              acceleration=1e-6),
        # A channel of odd extents with wetting walls, FP32-shifted populations.
        _case("channel_f32_odd", (190, 151, 117), 2, "halves", 200, storage="f32_shift",
              solid="spheres", acceleration=1e-6, wall_coupling=0.2),
        # A large droplet, FP16-shifted populations.
        _case("droplet_f16_large", (384, 384, 384), 2, "droplet", 200, storage="f16_shift"),
        # A parameter study: droplet lattices of 32 to 96 sites edge length with
        # their own tau, coupling and radius, FP32-shifted, advanced as one batch.
        _case("ensemble_f32", (96, 96, 96), 2, "droplet", 100, storage="f32_shift", graph=True,
              lattices=40),
        # Restart: populations and mask of a checkpoint up, some steps, the next
        # checkpoint's populations down.
        _case("restart", (96, 80, 75), 2, "checkpoint", 50, "populations", solid="spheres"),
    ]


# ---- drawn cases -----------------------------------------------------------------


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["2d", "2d", "one_3d", "two_f64", "two_f64", "two_shift", "two_shift",
                       "ensemble", "restart"])
    if kind == "2d":
        n = (_log_int(rng, 16, 700), _log_int(rng, 16, 700))
        comps = rng.choice([1, 2, 2, 3])
        form = rng.choice(["BDist2", "SecondOrder", "ThirdOrder"])
        return _unnamed(n, comps, "droplet" if comps == 2 and form == "BDist2" else "noise",
                        _log_int(rng, 1, 300), rng.choice(["density", "velocity"]), form=form,
                        shan_chen=comps > 1, graph=rng.random() < 0.5)
    if kind == "one_3d":
        n = tuple(_log_int(rng, 16, 160) for _ in range(3))
        return _unnamed(n, 1, "noise", _log_int(rng, 10, 150), "velocity", form="SecondOrder",
                        shan_chen=False, solid=rng.choice(["none", "plates"]),
                        acceleration=1e-5)
    if kind == "restart":
        n = tuple(_log_int(rng, 24, 110) for _ in range(3))
        return _unnamed(n, 2, "checkpoint", _log_int(rng, 5, 60), "populations",
                        solid=rng.choice(["none", "spheres"]))
    if kind == "ensemble":
        edge = _log_int(rng, 40, 96)
        return _unnamed((edge, edge, edge), 2, "droplet", _log_int(rng, 20, 120),
                        storage=rng.choice(["f32_shift", "f32_shift", "f16_shift"]), graph=True,
                        lattices=rng.randint(4, 40))
    storage = "f64" if kind == "two_f64" else rng.choice(["f32_shift", "f16_shift"])
    # the extent along z is the one that decides alignment: powers of two, multiples
    # of 32 and odd ones
    top = 256 if storage == "f64" else 320
    nz = rng.choice([rng.choice([32, 64, 128, 256]), 32 * rng.randint(1, top // 32),
                     _log_int(rng, 17, top)])
    n = (_log_int(rng, 24, top), _log_int(rng, 24, top), nz)
    init = rng.choice(["droplet", "halves", "noise"])
    sites = n[0] * n[1] * n[2]
    steps = max(20, min(300, int(2.5e9 / sites), _log_int(rng, 20, 300)))
    return _unnamed(n, 2, init, steps, storage=storage,
                    solid="none" if init == "noise" else rng.choice(["none", "plates", "spheres"]),
                    wall_coupling=rng.choice([0.0, 0.0, 0.2]), acceleration=1e-6,
                    graph=sites < 40000)


def _unnamed(*a, **k):
    c = _case("", *a, **k)
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------------


def _extent(case):
    return [case["nx"], case["ny"]] + ([case["nz"]] if case["nz"] else [])


def _spheres(n, fraction, rng):
    """Walls at both ends of the last axis and random solid spheres, periodic
    along the others, up to a solid fraction."""
    m = np.zeros(n, np.int32)
    m[:, :, 0] = 1
    m[:, :, -1] = 1
    solid, total = int(m.sum()), m.size
    top = max(2, min(12, min(n) // 6))
    while solid < fraction * total:
        r = int(rng.integers(max(1, top // 3), top + 1))
        d = np.arange(-r, r + 1)
        centre = [int(rng.integers(0, v)) for v in n]
        ball = (d[:, None, None] ** 2 + d[:, None] ** 2 + d ** 2 <= r * r).astype(np.int32)
        z = centre[2] + d
        keep = (z >= 0) & (z < n[2])
        at = np.ix_((centre[0] + d) % n[0], (centre[1] + d) % n[1], z[keep])
        new = m[at] | ball[:, :, keep]
        solid += int(new.sum() - m[at].sum())
        m[at] = new
    return m


def _mask(case, n, rng):
    if case["solid"] == "none":
        return None
    if case["solid"] == "spheres":
        return _spheres(n, 0.2, rng)
    m = np.zeros(n, np.int32)
    m[..., 0] = 1
    m[..., -1] = 1
    return m


def _edges(case):
    """Edge lengths of an ensemble's cubic lattices, 32 to the case's extent."""
    rng = np.random.default_rng([case["nx"], case["lattices"]])
    return [int(v) for v in rng.integers(min(32, case["nx"]), case["nx"] + 1, case["lattices"])]


def _member(case, seed, k):
    """Parameters and initial state of lattice k of a case, from the seed alone."""
    rng = np.random.default_rng([int(seed), k])
    n = _extent(case)
    nc = case["components"]
    tau, g = [case["tau"]] * nc, 3.6
    if case["lattices"] > 1:  # a member of a parameter study
        n = [_edges(case)[k]] * 3
        tau, g = [float(rng.uniform(1.0, 1.5))] * nc, float(rng.uniform(3.0, 4.5))
    p = {"n": n, "nc": nc, "tau": tau, "form": case["form"], "seed": int(rng.integers(1 << 31)),
         "mask": _mask(case, n, rng)}
    if nc == 3:
        g = 2.4
    p["gcc"] = [[0.0 if i == j else g for j in range(nc)] for i in range(nc)]
    p["gwc"] = [case["wall_coupling"] * (1 - 2 * (f % 2)) for f in range(nc)]
    p["acc"] = [0.0] * len(n)
    p["body"] = None
    if case["acceleration"] and nc == 1:
        p["acc"][0] = case["acceleration"]
    elif case["acceleration"]:  # on the second fluid alone
        p["body"] = [[0.0] * len(n) for _ in range(nc)]
        p["body"][1][0] = case["acceleration"]
    small = min(n)
    if case["init"] == "droplet":
        p["radius"] = float(rng.uniform(0.2, 0.35))
        p["offset"] = [float(v) for v in rng.uniform(-0.1, 0.1, len(n))]
        big, low = float(rng.uniform(0.66, 0.74)), float(rng.uniform(0.035, 0.045))
        p["dens"] = [[big, low], [low, big]]
        p["thickness"] = min(5.0, small / 6)
    elif case["init"] == "halves":
        cut = int(rng.integers(2 * n[0] // 5, 3 * n[0] // 5 + 1))
        p["widths"] = [float(cut), float(n[0] - cut)]
        big = float(rng.uniform(0.95, 1.0))
        p["dens"] = [[big, LIGHT], [LIGHT, big]]
    elif case["init"] == "noise":
        p["dens"] = [0.7 if nc > 1 else 1.0] * nc
        p["noise"] = 0.01 if nc > 1 else 1e-3
    else:  # the populations of a checkpoint
        p["pops"] = [_checkpoint(n, f, rng, p["mask"]) for f in range(nc)]
    return p


def _checkpoint(n, f, rng, mask):
    """Populations of a running two-fluid mixture: a smooth density profile,
    off equilibrium by a little everywhere; the rest state inside walls."""
    x = [np.arange(v) / v for v in n]
    phase = rng.uniform(0, 2 * np.pi, 3)
    s = (np.sin(2 * np.pi * x[0] + phase[0])[:, None, None]
         + np.sin(2 * np.pi * x[1] + phase[1])[:, None]
         + np.sin(2 * np.pi * x[2] + phase[2])) / 3
    rho = 0.4 + (0.3 if f == 0 else -0.3) * s
    pop = rho[..., None] * np.asarray(W3)
    pop *= 1.0 + 0.02 * (rng.random(pop.shape, np.float32) - np.float32(0.5))
    if mask is not None:
        pop[mask != 0] = [1.0] + [0.0] * 18
    return pop


def _rho0(storage):
    """The reference densities bench.py stores deviations from."""
    if storage == "f16_shift":
        return [2 * LIGHT * DENSE / (LIGHT + DENSE)] * 2
    return [0.5 * (LIGHT + DENSE)] * 2


def _lattice(case, p):
    d, q = (3, 19) if len(p["n"]) == 3 else (2, 9)
    lat = dlbc_amd.Lattice(d, q, p["nc"], p["n"], storage=case["storage"])
    lat.set_params(p["tau"], p["gcc"], p["gwc"], p["acc"], p["body"], p["form"], "Exponential",
                   case["shan_chen"], _rho0(case["storage"]) if case["storage"] != "f64" else None)
    if "pops" in p:
        return lat
    if p["mask"] is not None:
        lat.upload_mask(p["mask"])
    rng = dlbc_amd.Rng(p["seed"])
    for f in range(p["nc"]):
        if case["init"] == "droplet":
            lat.init_fluid(f, "EqDistSphereFrac", p["dens"][f], p["form"], radius=p["radius"],
                           offset=p["offset"], thickness=p["thickness"])
        elif case["init"] == "halves":
            lat.init_fluid(f, "EqDistLamellae", p["dens"][f], p["form"], widths=p["widths"])
        else:
            lat.init_fluid(f, "EqDistPerturb", [p["dens"][f]], p["form"], perturb=p["noise"],
                           rng=rng)
        lat.init_eq_dist_wall(f)
    return lat


def prepare(case, seed):
    members = [_member(case, seed, k) for k in range(case["lattices"])]
    state = {"case": case, "lats": [_lattice(case, p) for p in members]}
    if case["lattices"] > 1:
        state["batch"] = dlbc_amd.Batch(state["lats"])
        state["batch"].autotune()
    if "pops" in members[0]:
        state["mask"] = members[0]["mask"]
        if state["mask"] is None:
            state["mask"] = np.zeros(members[0]["n"], np.int32)
        state["pops"] = members[0]["pops"]
    return state


# ---- one pass ----------------------------------------------------------------------


def run(state):
    case, lats = state["case"], state["lats"]
    if "batch" in state:
        state["batch"].step(case["steps"], graph=case["graph"])
        return [lat.density(0) for lat in lats]
    lat = lats[0]
    if "pops" in state:
        lat.upload_mask(state["mask"])
        for f, pop in enumerate(state["pops"]):
            lat.upload_population(f, pop)
    lat.step(case["steps"], graph=case["graph"])
    if case["out"] == "populations":
        return [lat.population(f) for f in range(lat.nc)]
    if case["out"] == "colour":
        return lat.colour(0, 1)
    if case["out"] == "velocity":
        return [lat.density(0), lat.velocity(0)]
    # the largest output of a long FP16 run is the first fluid's field alone
    if lat.sites > 1 << 25:
        return lat.density(0)
    return [lat.density(f) for f in range(lat.nc)]


def work(case):
    """Every population read once and written once per step (BGK and the force
    from its neighbours), and the fields of the output written once."""
    n = _extent(case)
    q = 19 if len(n) == 3 else 9
    sites = float(np.prod(n))
    if case["lattices"] > 1:
        sites = float(sum(e ** 3 for e in _edges(case)))
    fluid = sites * (0.8 if case["solid"] == "spheres" else 1.0)
    elem = {"f64": 8, "f32_shift": 4, "f16_shift": 2}[case["storage"]]
    nc = case["components"]
    moved = case["steps"] * fluid * 2 * nc * q * elem
    field = {"density": nc, "colour": 1, "velocity": 1 + len(n), "populations": 2 * nc * q}
    fields = 1 if case["lattices"] > 1 or sites > 1 << 25 else field[case["out"]]
    # per population and component: streaming, moments, force, equilibrium, relaxation
    flops = case["steps"] * fluid * nc * q * (24.0 if case["shan_chen"] else 16.0)
    return {"bytes": moved + 8.0 * sites * fields, "flops": flops}


# ---- the same in 64 bits, with torch alone ---------------------------------------------


def _unity(d, form):
    """Equilibrium of unit density at rest."""
    if d == 2 and form == "BDist2":
        return [1 / 2] + [1 / 12] * 4 + [1 / 24] * 4
    return W3 if d == 3 else W2


def _transition(pos, width, neg, posv):
    """Linear from neg to posv over [-width / 2, width / 2]."""
    t = (pos / width).clamp(-0.5, 0.5)
    return neg * (0.5 - t) + posv * (0.5 + t)


def _density_0(case, p, f, dev, draws):
    n = p["n"]
    x = [torch.arange(v, dtype=torch.float64, device=dev) for v in n]
    if case["init"] == "droplet":
        r2 = torch.zeros(n, dtype=torch.float64, device=dev)
        for i, v in enumerate(n):
            shape = [1] * len(n)
            shape[i] = v
            r2 += ((x[i] - (v * 0.5 + p["offset"][i] * v) + 0.5) ** 2).reshape(shape)
        return _transition(r2.sqrt() - p["radius"] * min(n), p["thickness"], *p["dens"][f])
    if case["init"] == "halves":
        rho = torch.full_like(x[0], p["dens"][f][1])
        rho[: int(p["widths"][0])] = p["dens"][f][0]
        return rho[:, None, None].expand(n)
    pad = [v + 4 for v in n]  # drawn over the field with its halo of two
    u = draws.randint(0, 1 << 32, int(np.prod(pad)), dtype=np.uint32) / (2.0 ** 32 - 1)
    u = u.reshape(pad)[tuple(slice(2, -2) for _ in n)]
    return torch.from_numpy(p["dens"][f] - p["noise"] + 2 * p["noise"] * u).to(dev)


def _equilibrium(d, form, rho, v, i, c, w, uu):
    """Population i of the equilibrium; uu: v.v."""
    cu = sum(v[a] * c[i][a] for a in range(d) if c[i][a])
    if not torch.is_tensor(cu):
        cu = torch.zeros_like(rho)
    if form != "BDist2":
        e = 1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * uu
        if form == "ThirdOrder":
            e = e + 4.5 * cu ** 3 - 4.5 * uu * cu
        return rho * w[i] * e
    cst = 1.0 - 1.5 * uu
    a1 = 1 / 36 if d == 3 else 1 / 24
    if i == 0:
        return rho * cst * (1 / 3 if d == 3 else 1 / 2)
    t = 3.0 * cu
    e = a1 * (cst + 0.5 * t * t + cst * t + t ** 3 / 6)
    return rho * e * (2.0 if sum(abs(a) for a in c[i]) == 1 else 1.0)


def _advance(case, p, f_in, solid, steps):
    n, nc, form = p["n"], p["nc"], p["form"]
    d = len(n)
    c, w = (C3, W3) if d == 3 else (C2, W2)
    q = len(c)
    back = [c.index(tuple(-a for a in v)) for v in c]
    dims = tuple(range(d))
    f = f_in
    wall_rho = [None] * nc
    if solid is not None:
        near = [torch.roll(solid, c[i], dims) for i in range(q)]  # x - c_i is solid
        wall_rho = [torch.where(solid, sum(f[k]), 0.0) for k in range(nc)]
    for _ in range(steps):
        s, rho, psi = [], [], []
        for k in range(nc):
            new = []
            for i in range(q):
                v = torch.roll(f[k][i], c[i], dims) if i else f[k][0]
                if solid is not None and i:
                    v = torch.where(near[i], f[k][back[i]], v)
                if solid is not None:
                    v = torch.where(solid, f[k][i], v)
                new.append(v)
            s.append(new)
            rho.append(sum(new[1:], new[0].clone()))
        f = None
        if case["shan_chen"]:
            psi = [-torch.expm1(-r) for r in rho]
        mom = [[sum(s[k][i] * c[i][a] for i in range(q) if c[i][a]) for a in range(d)]
               for k in range(nc)]
        if form == "BDist2":
            total = sum(rho)
            common = [sum(mom[k][a] / p["tau"][k] for k in range(nc)) / total for a in range(d)]
        grad = []
        if case["shan_chen"]:
            for k in range(nc):
                g = [torch.zeros_like(rho[0]) for _ in range(d)]
                for i in range(1, q):
                    v = torch.roll(psi[k], [-a for a in c[i]], dims)
                    if solid is not None:
                        v = torch.where(near[back[i]], psi[k], v)
                    for a in range(d):
                        if c[i][a]:
                            g[a].add_(v, alpha=w[i] * c[i][a])
                grad.append(g)
        f = []
        for k in range(nc):
            dv = []
            for a in range(d):
                force = torch.zeros_like(rho[k])
                for o in range(nc):
                    if case["shan_chen"] and p["gcc"][k][o]:
                        force -= psi[k] * grad[o][a] * p["gcc"][k][o]
                if solid is not None and case["shan_chen"] and p["gwc"][k]:
                    for i in range(1, q):
                        if c[i][a]:
                            v = torch.roll(wall_rho[k], [-b for b in c[i]], dims)
                            force -= psi[k] * v * (w[i] * c[i][a] * p["gwc"][k])
                if p["body"]:
                    force += p["body"][k][a]
                shift = p["tau"][k] * (p["acc"][a] + force / rho[k])
                dv.append(shift + (common[a] if form == "BDist2" else mom[k][a] / rho[k]))
            uu = sum(v * v for v in dv)
            om = 1.0 / p["tau"][k]
            for i in range(q):
                e = _equilibrium(d, form, rho[k], dv, i, c, w, uu)
                v = s[k][i] + om * (e - s[k][i])
                s[k][i] = v if solid is None else torch.where(solid, s[k][i], v)
            f.append(s[k])
    return f


def exact(case, seed):
    n = _extent(case)
    sites = float(np.prod(n))
    if case["lattices"] > 1:
        sites = float(sum(e ** 3 for e in _edges(case)))
    if sites * case["steps"] * case["components"] * (19 if len(n) == 3 else 9) > 1.4e11:
        return None  # too long in plain torch
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    outs = []
    for k in range(case["lattices"]):
        p = _member(case, seed, k)
        n = p["n"]
        d = len(n)
        solid = None if p["mask"] is None else torch.from_numpy(p["mask"] != 0).to(dev)
        draws = np.random.RandomState(p["seed"])
        f = []
        for comp in range(p["nc"]):
            if "pops" in p:
                a = torch.from_numpy(p["pops"][comp]).to(dev)
                f.append([a[..., i].contiguous() for i in range(a.shape[-1])])
                continue
            rho = _density_0(case, p, comp, dev, draws)
            f.append([(rho * u).contiguous() for u in _unity(d, p["form"])])
            if solid is not None:
                for i, v in enumerate(f[comp]):
                    v[solid] = 1.0 if i == 0 else 0.0
        f = _advance(case, p, f, solid, case["steps"])
        if case["lattices"] > 1:
            outs.append(sum(f[0]).cpu().numpy())
            continue
        if case["out"] == "populations":
            return [torch.stack(v, -1).cpu().numpy() for v in f]
        rho = [sum(v) for v in f]
        if case["out"] == "colour":
            col = rho[0] - rho[1]
            return (col if solid is None else torch.where(solid, 0.0, col)).cpu().numpy()
        if case["out"] == "velocity":
            c = C3 if d == 3 else C2
            u = torch.stack([sum(f[0][i] * c[i][a] for i in range(len(c)) if c[i][a])
                             for a in range(d)], -1) / rho[0][..., None]
            if solid is not None:
                u[solid] = 0.0
            return [rho[0].cpu().numpy(), u.cpu().numpy()]
        if sites > 1 << 25:
            return rho[0].cpu().numpy()
        return [r.cpu().numpy() for r in rho]
    return outs
