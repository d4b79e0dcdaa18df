"""The work that a user of this framework has it do, as cases to be timed.

A case is one pass of a simulation program between two of its outputs, through
the package's public calls.  The sizes are those of this repository's
benchmark workloads and tests (the 1-D Couette flows, the two-gas box, the
batched 0-D cells, the BKW boxes with merging), cut down where a single pass
over the whole batch would only repeat the same work on more cells, and the
range around them that draw() covers.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the store a program holds before the pass
    run(state)          one pass and its outputs
    work(case)          bytes and flops that a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   what run() returns, from plain numpy in 64 bits

Where the number of particles is fixed, the particle state is returned up to
STATE_MAX particles, as a program that writes a particle dump does.  Elsewhere
a program keeps the particles on the GPU and reads the computed properties and
collision factors, so those are returned: every particle's weight and velocity
goes into its cell's, at the full 64 bits, and the counts are whole numbers.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "merzbild.jl_amd")
K_B = 1.380649e-23
MASS = {"Ar": 66.3e-27, "He": 6.65e-27}
VHS = {"Ar,Ar": (4.11e-10, 0.81, 273.0), "Ar,He": (3.25e-10, 0.735, 273.0), "He,He": (2.33e-10, 0.66, 273.0)}
STATE_MAX = 200_000
DATA = os.path.join(PACKAGE, "data")

# The Couette flow: argon, walls at 300 K moving at -/+500 m/s, 5e-4 m wide.
L, T_WALL, V_WALL = 5e-4, 300.0, 500.0
# The 0-D boxes: pseudo-Maxwell argon, BKW velocities at 273 K, V = 1, 1e23 m^-3.
T_BKW, NDENS_BKW = 273.0, 1e23



def load_package():
    """The package, whose folder's name is not a Python identifier."""
    name = "merzbild_jl_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(PACKAGE, "__init__.py"),
                                                      submodule_search_locations=[PACKAGE])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # test_2species: a single box of 400 Ar and 4,000 He particles, a step
        # at a time with the properties after it: the smallest calls there are
        dict(name="two_gas_box", kind="two_gas", n_ar=400, n_he=4000, steps=4),
        # test_1D_couette: 50 cells of 1,000, the properties written every 200 steps
        dict(name="couette_50x1000", kind="couette", cells=50, ppc=1000, dt=2.59e-9, ndens=5e22, steps=200,
             mode="slab"),
        # the headline flow, 500 cells of 200, all steps in one call
        dict(name="couette_500x200", kind="couette", cells=500, ppc=200, dt=2e-10, ndens=1e23, steps=2000,
             mode="slab"),
        # the same flow from a program that calls the operators one by one
        dict(name="operators_500x200", kind="operators", cells=500, ppc=200, dt=2e-10, ndens=1e23, steps=4,
             equal_weight=True, flux=False),
        # a large flow, operator by operator with the heat fluxes: memory-bound
        dict(name="operators_16000x250", kind="operators", cells=16000, ppc=250, dt=2e-10, ndens=1e23, steps=2,
             equal_weight=False, flux=True),
        # couette_with_surface_quantities: 2,000 cells of 250, the averaging phase
        dict(name="wall_averages_2000x250", kind="averages", cells=2000, ppc=250, dt=2.59e-9, ndens=5e22, steps=50),
        # test_1D_couette_varweight at the headline size: splitting, octree merges
        dict(name="varweight_500x200", kind="varweight", cells=500, threshold=400, target=64, dt=2e-10, ndens=1e23,
             steps=10),
        # uneven 0-D cells, log-uniform 20..20000 particles, no splitting
        dict(name="batched_0d_2048", kind="batched", cells=2048, nmin=20, nmax=20000, steps=50),
        # the same cells with splitting and octree merging back to each cell's count
        dict(name="batched_split_1024", kind="split", cells=1024, nmin=20, nmax=20000, steps=2),
        # test_bkw_varweight_octree_swpm over many boxes
        dict(name="swpm_octree_4096", kind="boxes", cells=4096, target=1000, threshold=1250, merge="octree", steps=2),
        # the same loop with the merge on a velocity grid
        dict(name="swpm_grid_2048", kind="boxes", cells=2048, target=140, threshold=1000, merge="grid", steps=2),
        # test_bkw_varweight_nnls over many boxes: moment-preserving merges
        # (35 moments), octree merges where NNLS finds no solution
        dict(name="ntc_nnls_8192", kind="nnls", cells=8192, threshold=200, method="wave", steps=2),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["two_gas", "couette", "couette", "operators", "operators", "averages", "varweight",
                       "varweight", "batched", "batched", "split", "split", "boxes", "boxes", "nnls"])
    if kind == "two_gas":
        return dict(kind=kind, n_ar=_log_int(rng, 50, 4000), n_he=_log_int(rng, 50, 8000), steps=rng.randint(1, 5))
    if kind == "couette":
        # dt keeps particles within about a cell a step (slab-resident steps)
        # or lets them cross several (the step graph)
        cells, ppc = _log_int(rng, 20, 700), _log_int(rng, 20, 1000)
        while cells * ppc > 150_000:
            ppc = max(20, ppc // 2)
        return dict(kind=kind, cells=cells, ppc=ppc, dt=rng.uniform(0.05, 0.3) * (L / cells) / 1000.0,
                    ndens=rng.choice([5e22, 1e23]), steps=_log_int(rng, 50, 1000),
                    mode=rng.choice(["slab", "slab", "graph"]))
    if kind == "operators":
        cells, ppc = _log_int(rng, 20, 20000), _log_int(rng, 20, 1000)
        while cells * ppc > 4_000_000:
            ppc = max(20, ppc // 2)
        return dict(kind=kind, cells=cells, ppc=ppc, dt=2e-10, ndens=1e23, steps=rng.randint(1, 2),
                    equal_weight=rng.random() < 0.5, flux=rng.random() < 0.5)
    if kind == "averages":
        return dict(kind=kind, cells=_log_int(rng, 100, 2000), ppc=_log_int(rng, 20, 250), dt=2.59e-9, ndens=5e22,
                    steps=rng.randint(10, 50))
    if kind == "varweight":
        target = rng.randint(32, 100)
        return dict(kind=kind, cells=_log_int(rng, 50, 2000), threshold=target * rng.randint(3, 6), target=target,
                    dt=2e-10, ndens=1e23, steps=rng.randint(2, 10))
    if kind == "batched":
        return dict(kind=kind, cells=_log_int(rng, 64, 2048), nmin=20, nmax=_log_int(rng, 200, 20000),
                    steps=rng.randint(5, 50))
    if kind == "split":
        return dict(kind=kind, cells=_log_int(rng, 64, 1024), nmin=20, nmax=_log_int(rng, 500, 20000),
                    steps=rng.randint(1, 2))
    if kind == "boxes":
        merge = rng.choice(["octree", "octree", "grid", "roulette"])
        # a 4 x 4 x 4 velocity grid leaves at most 144 particles
        target = 140 if merge == "grid" else _log_int(rng, 100, 1000)
        threshold = _log_int(rng, 300, 1200) if merge == "grid" else target * 5 // 4 + 50
        return dict(kind=kind, cells=_log_int(rng, 128, 4096), target=target, threshold=threshold, merge=merge,
                    steps=rng.randint(1, 2))
    return dict(kind="nnls", cells=_log_int(rng, 256, 8192), threshold=rng.randint(160, 230),
                method=rng.choice(["wave", "wave", "lds", "reference"]), steps=rng.randint(1, 2))


# ---------------------------------------------------------------------------
# inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _int_log_uniform(g, n, lo, hi):
    return torch.exp(math.log(lo) + _rand(g, n) * (math.log(hi) - math.log(lo))).floor().long()


def _inputs(case, seed):
    """The particles of a case, in cell order, as host arrays: x, v [n, 3], w
    [n] and the particles per cell; per species for the two-gas box."""
    g, kind = _generator(seed), case["kind"]
    if kind == "two_gas":
        out = []
        for name, n, temp in (("Ar", case["n_ar"], 3000.0), ("He", case["n_he"], 360.0)):
            v = math.sqrt(K_B * temp / MASS[name]) * _randn(g, n, 3)
            out.append(dict(x=_rand(g, n, 3).cpu().numpy(), v=v.cpu().numpy(), w=np.full(n, 5e12),
                            counts=np.array([n])))
        return out
    nc = case["cells"]
    if kind in ("couette", "operators", "averages"):
        counts = torch.full((nc,), case["ppc"], device="cuda")
    elif kind == "varweight":
        # anywhere between a merge's result and the next merge
        counts = _int_log_uniform(g, nc, case["target"], case["threshold"])
    elif kind == "batched":
        counts = _int_log_uniform(g, nc, case["nmin"], case["nmax"])
    elif kind == "split":
        counts = (_targets(case, g).double() * (1.0 + 0.5 * _rand(g, nc))).long()
    elif kind == "boxes" and case["merge"] == "grid":
        counts = _int_log_uniform(g, nc, case["target"], case["threshold"])
    elif kind == "boxes":
        counts = (case["target"] + _rand(g, nc) * (case["threshold"] - case["target"])).long()
    else:
        counts = _int_log_uniform(g, nc, 35, case["threshold"] * 5 // 4)
    cell = torch.repeat_interleave(torch.arange(nc, device="cuda"), counts)
    n = cell.numel()
    if kind in ("couette", "operators", "averages", "varweight"):
        dx = L / nc
        x = torch.cat([((cell + _rand(g, n)) * dx)[:, None], _rand(g, n, 2)], 1)
        v = math.sqrt(K_B * T_WALL / MASS["Ar"]) * _randn(g, n, 3)
        w = (case["ndens"] * dx / counts.double())[cell]
    else:
        x = torch.full((n, 3), 0.5, device="cuda", dtype=torch.float64)
        x[:, 0] += cell
        speed = math.sqrt(2 * K_B * T_BKW / MASS["Ar"]) * math.sqrt(0.3) * _randn(g, n, 5).norm(dim=1)
        th, ph = math.pi * _rand(g, n), 2 * math.pi * _rand(g, n)
        v = speed[:, None] * torch.stack([th.sin() * ph.cos(), th.sin() * ph.sin(), th.cos()], 1)
        w = (NDENS_BKW / counts.double())[cell]
    if kind in ("varweight", "nnls"):
        w = w * torch.exp(_randn(g, n)) / math.exp(0.5)
    elif kind in ("batched", "split"):
        w = w * (0.5 + 1.5 * _rand(g, n))
    return dict(x=x.cpu().numpy(), v=v.cpu().numpy(), w=w.cpu().numpy(), counts=counts.cpu().numpy())


def _targets(case, g):
    """The particles a splitting cell is merged back to."""
    return _int_log_uniform(g, case["cells"], case["nmin"], case["nmax"])


def _upload(st, species, p):
    counts, n = p["counts"].astype(np.int64), len(p["w"])
    first = np.cumsum(counts) - counts
    pia = np.zeros((len(counts), 7), dtype=np.int64)
    pia[:, 0] = pia[:, 3] = counts
    pia[:, 1], pia[:, 2], pia[:, 5] = first + 1, first + counts, -1
    st.upload_species(species, p["x"], p["v"], p["w"], np.arange(1, n + 1), pia, n, True, None, n)


def prepare(case, seed):
    pkg, kind = load_package(), case["kind"]
    p = _inputs(case, seed)
    flow = kind in ("couette", "operators", "averages", "varweight")
    names = ["Ar", "He"] if kind == "two_gas" else ["Ar"]
    sp = pkg.load_species_data(os.path.join(DATA, "particles.toml"), names)
    table = "vhs.toml" if flow or kind == "two_gas" else "pseudo_maxwell.toml"
    it = pkg.load_interaction_data(os.path.join(DATA, table), sp)
    nc = case.get("cells", 1)
    if kind == "two_gas":
        st = pkg.DeviceStore(1, 2, [case["n_ar"] + 256, case["n_he"] + 256])
        for s, q in enumerate(p):
            _upload(st, s + 1, q)
        st.set_grid(pkg.Grid1DUniform(1.0, 1))
    else:
        n = len(p["w"])
        # room for the particles that splits and SWPM collisions create
        # between merges
        cap = n + 4096
        if kind == "varweight":
            cap = nc * (3 * case["threshold"] // 2) + 4096
        elif kind == "split":
            cap = 2 * n + 65536
        elif kind == "boxes":
            cap = 2 * nc * case["threshold"] + 4096
        elif kind == "nnls":
            cap = nc * 500 + 4096
        st = pkg.DeviceStore(nc, 1, cap)
        _upload(st, 1, p)
        st.set_grid(pkg.Grid1DUniform(L if flow else float(nc), nc))
    if flow:
        st.set_walls(pkg.MaxwellWalls1D(sp, T_WALL, T_WALL, -V_WALL, V_WALL, 1.0, 1.0))
    st.set_interactions(it)
    st.set_species_data(sp)
    st.set_seed(seed)
    s = dict(pkg=pkg, st=st, sp=sp, case=case, step=1)
    if kind == "two_gas":
        temp = (3000.0, 360.0)
        for i in range(2):
            for k in range(2):
                st.set_sigma_g_w_max(i + 1, k + 1, pkg.estimate_sigma_g_w_max(
                    it[i][k], sp[i].mass, sp[k].mass, temp[i], temp[k], 5e12))
        return s
    m, temp = sp[0].mass, T_WALL if flow else T_BKW
    fnum = (case["ndens"] * (L / nc) if flow else NDENS_BKW) / np.maximum(p["counts"], 1)
    if kind == "boxes":
        fnum = np.ones(nc)     # swpm keeps (sigma g)_max, without a weight
    st.set_sigma_g_w_max(1, 1, pkg.estimate_sigma_g_w_max(it[0][0], m, m, temp, temp, fnum))
    if not flow:
        t_ref = 1.0 / (NDENS_BKW * math.pi * it[0][0].vhs_d ** 2) / math.sqrt(2 * K_B * T_BKW / m)
        s["dt"] = (0.1 if kind == "nnls" else 0.025) * t_ref
    if kind == "split":
        targets = _targets(case, _generator(seed)).cpu().numpy()
        s["targets"], s["thresholds"] = targets.astype(np.int32), (3 * targets // 2).astype(np.int32)
    elif kind == "averages":
        s["surf"] = pkg.SurfProps.grid1d(1)
        st.surf_clear(1)
        st.props_avg_clear()
    elif kind == "boxes" and case["merge"] == "grid":
        s["grid"] = pkg.GridN2Merge(4, extent_multiplier=3.5)
    elif kind == "nnls":
        s["moments"] = [t for order in range(1, 5) for t in pkg.multi_index_moments(order)]
    return s


# ---------------------------------------------------------------------------
# one pass

def _props(pp):
    return dict(lpa=pp.lpa, np=pp.np, n=pp.n, v=pp.v, T=pp.T)


def _particles(s):
    """The particle state as a dump reads it, where a program takes one."""
    if sum(s["st"].scalars(k + 1)["n_total"] for k in range(s["st"].n_species)) > STATE_MAX:
        return []
    out = []
    for k in range(s["st"].n_species):
        d = s["st"].download_species(k + 1)
        out.append({f: d[f] for f in ("x", "v", "w", "index", "pia")})
    return out


def _collisions(s, pairs=((1, 1),)):
    return [s["st"].collision_factors(i, k) for i, k in pairs]


def run(s):
    pkg, st, sp, case, k = s["pkg"], s["st"], s["sp"], s["case"], s["case"]["kind"]
    steps, t0 = case["steps"], s["step"]
    s["step"] = t0 + steps
    return {"two_gas": _run_two_gas, "couette": _run_couette, "operators": _run_operators,
            "averages": _run_averages, "varweight": _run_varweight, "batched": _run_batched, "split": _run_split,
            "boxes": _run_boxes, "nnls": _run_nnls}[k](s, pkg, st, sp, case, range(t0, t0 + steps))


def _run_two_gas(s, pkg, st, sp, case, steps):
    series = []
    for t in steps:
        # one tag per call: each call of a step draws streams of its own
        for j, (a, b) in enumerate(((1, 1), (2, 2), (1, 2))):
            pkg.ntc(st, a, b, 2.5e-3, V=1.0, tag=(t << 4) | (j + 1))
        series.append(_props(pkg.compute_props(st, sp)))
    return dict(series=series, collisions=_collisions(s, ((1, 1), (2, 2), (1, 2))), particles=_particles(s))


def _run_couette(s, pkg, st, sp, case, steps):
    pkg.couette_steps(st, len(steps), steps[0], case["dt"], sp, mode=case["mode"])
    pp = pkg.PhysProps(case["cells"], 1).fetch(st)
    return dict(props=_props(pp), collisions=_collisions(s), particles=_particles(s))


def _run_operators(s, pkg, st, sp, case, steps):
    out = []
    for t in steps:
        pkg.ntc(st, 1, 1, case["dt"], equal_weight=case["equal_weight"], tag=(t << 4) | 1)
        pkg.convect_particles(st, 1, case["dt"], tag=(t << 4) | 2)
        pkg.sort_particles(st, 1)
        r = _props(pkg.compute_props_sorted(st, sp))
        if case["flux"]:
            f = pkg.compute_flux_props_sorted(st, sp)
            r.update(energy_flux=f.kinetic_energy_flux, diagonal=f.diagonal_momentum_flux,
                     off_diagonal=f.off_diagonal_momentum_flux)
        out.append(r)
    return dict(series=out, collisions=_collisions(s), particles=_particles(s))


def _run_averages(s, pkg, st, sp, case, steps):
    pkg.couette_avg_steps(st, len(steps), steps[0], case["dt"], len(steps), sp, surf_props=s["surf"], mode="graph")
    surf = s["surf"].fetch(st, 1)
    pp = pkg.PhysProps(case["cells"], 1).fetch_avg(st)
    out = dict(props=_props(pp), surf={f: getattr(surf, f).copy() for f in surf.FIELDS}, collisions=_collisions(s),
               particles=_particles(s))
    st.surf_clear(1)
    st.props_avg_clear()
    return out


def _run_varweight(s, pkg, st, sp, case, steps):
    merged = 0
    for t in steps:
        pkg.ntc(st, 1, 1, case["dt"], tag=(t << 4) | 1)
        merged += pkg.merge_octree_N2_based(st, 1, case["threshold"], case["target"], max_depth=8, grid_clamp=True,
                                            tag=(t << 4) | 3)
        pkg.convect_particles(st, 1, case["dt"], tag=(t << 4) | 2)
        pkg.sort_particles(st, 1)
        pkg.compute_props_sorted(st, sp, fetch=False)
    return dict(merged=merged, props=_props(pkg.PhysProps(case["cells"], 1).fetch(st)), collisions=_collisions(s))


def _moments(pkg, s):
    pp = pkg.PhysProps(s["case"]["cells"], 1, [4, 6, 8], Tref=T_BKW)
    pkg.compute_props_with_total_moments(s["st"], s["sp"], pp)
    return dict(_props(pp), moments=pp.moments)


def _run_batched(s, pkg, st, sp, case, steps):
    pkg.batch0d_steps(st, len(steps), steps[0], s["dt"], sp)
    return dict(props=_props(pkg.PhysProps(case["cells"], 1).fetch(st)), collisions=_collisions(s))


def _run_split(s, pkg, st, sp, case, steps):
    merged, series = 0, []
    for t in steps:
        pkg.ntc(st, 1, 1, s["dt"], V=1.0, tag=(t << 4) | 1)
        pkg.sort_particles(st, 1)
        merged += pkg.merge_octree_targets(st, 1, s["thresholds"], s["targets"], max_Nbins=1 << 20,
                                           tag=(t << 4) | 3)
        series.append(_moments(pkg, s))
    return dict(merged=merged, series=series, collisions=_collisions(s))


def _run_boxes(s, pkg, st, sp, case, steps):
    merged, series = 0, []
    for t in steps:
        pkg.swpm(st, 1, 1.0, s["dt"], V=1.0, tag=(t << 4) | 1)
        if case["merge"] == "octree":
            merged += pkg.merge_octree_N2_based(st, 1, case["threshold"], case["target"], max_Nbins=512,
                                                tag=(t << 4) | 3)
        elif case["merge"] == "grid":
            pkg.compute_props(st, sp)      # the velocity grid's extents
            merged += pkg.merge_grid_based(st, 1, case["threshold"], s["grid"], sp, tag=(t << 4) | 3)
        else:
            merged += pkg.merge_roulette(st, 1, case["threshold"], case["target"], conservative=True,
                                         tag=(t << 4) | 3)
        pkg.sort_particles(st, 1)
        series.append(_moments(pkg, s))
    return dict(merged=merged, series=series, collisions=_collisions(s))


def _run_nnls(s, pkg, st, sp, case, steps):
    status, series = [], []
    for t in steps:
        pkg.ntc(st, 1, 1, s["dt"], V=1.0, tag=(t << 4) | 1)
        status.append(pkg.merge_nnls_candidates(st, 1, case["threshold"], s["moments"], 239, method=case["method"],
                                                tag=(t << 4) | 3))
        # the octree where NNLS found no solution
        pkg.merge_octree_N2_based(st, 1, 400, case["threshold"], tag=(t << 4) | 5)
        pkg.sort_particles(st, 1)
        series.append(_moments(pkg, s))
    return dict(status=status, series=series, collisions=_collisions(s))


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _mean_particles(case):
    kind, nc = case["kind"], case.get("cells", 1)
    if kind == "two_gas":
        return case["n_ar"] + case["n_he"]
    if kind in ("couette", "operators", "averages"):
        return nc * case["ppc"]
    if kind == "boxes":
        return nc * (case["target"] + case["threshold"]) / 2
    lo, hi = {"varweight": (case.get("target"), case.get("threshold")), "nnls": (35, case.get("threshold", 0) * 1.25),
              "batched": (case.get("nmin"), case.get("nmax")), "split": (case.get("nmin"), case.get("nmax"))}[kind]
    return nc * (hi - lo) / math.log(hi / lo) * (1.25 if kind == "split" else 1.0)


def work(case):
    """The particles (x, v, w: 56 B, id: 4 B) read and written once, the cell
    table and the properties written once; per particle and step 30 flops of
    flight, cell and property sums, and 60 per collision candidate of the
    few-per-cent that a step picks."""
    n, nc = _mean_particles(case), case.get("cells", 1)
    return {"bytes": 120.0 * n + 100.0 * nc, "flops": 32.0 * n * case["steps"]}


def tolerance(case):
    """Every sum and every particle is in 64 bits; two implementations differ
    by the order of sums and by an ulp or two of pow, log, sin and cos, which
    collisions carry on without growing them (the scattering direction comes
    from the draws).  Against plain numpy the properties are up to 1.4e-14 off
    (SWPM and merges over 4,096 boxes) and the particles of four Couette steps
    6e-18; the bound leaves room for thousands of steps.  An NNLS merge may end
    anywhere its moments are met to 1e-11.  Whole numbers are the same."""
    return {"rel": 1e-10, "max": 1e-8} if case["kind"] == "nnls" else {"rel": 1e-12, "max": 1e-10}


# ---------------------------------------------------------------------------
# plain numpy

def _cell_props(w, v, cell, nc, mass):
    n = np.bincount(cell, w, nc)
    vm = np.stack([np.bincount(cell, w * v[:, d], nc) for d in range(3)], 1) / n[:, None]
    c = v - vm[cell]
    e = np.bincount(cell, w * (c * c).sum(1), nc)
    return n, vm, e * mass / (3.0 * n * K_B)


def exact(case, seed):
    """0-D boxes: collisions and merges keep each cell's weight, momentum and
    energy, so after any number of steps n, v and T are the initial
    particles'; which particles carry them follows from the random streams and
    has no value apart from them.  The flows' walls draw from those streams
    too; their first step is worked out whole (with its draws) up to a million
    particles."""
    kind = case["kind"]
    if kind == "operators":
        return _exact_operators(case, seed) if case["cells"] * case["ppc"] * case["steps"] <= 1_000_000 else None
    if kind in ("couette", "averages", "varweight"):
        return None
    if kind == "two_gas":
        # the gases exchange momentum and energy: only their densities stay
        p = _inputs(case, seed)
        n = np.array([[q["w"].sum()] for q in p])
        return dict(series=[dict(lpa=None, np=None, n=n, v=None, T=None)] * case["steps"], collisions=None,
                    particles=None)
    p, nc = _inputs(case, seed), case["cells"]
    cell = np.repeat(np.arange(nc), p["counts"])
    n, v, temp = _cell_props(p["w"], p["v"], cell, nc, MASS["Ar"])
    keep = dict(lpa=None, np=None, n=n[None], v=v[None], T=temp[None])
    if kind == "batched":
        # ntc_equal_weight! on unequal weights keeps the weight alone
        return dict(props=dict(keep, v=None, T=None))
    return dict(series=[keep] * case["steps"])


def _philox(stream, k, tag, key):
    """Draw k of each stream: Philox4x32-10 on (k / 2, stream, tag) under the
    key, 53 bits of the block's half k % 2."""
    u32, mask = np.uint64(32), np.uint64(0xFFFFFFFF)
    stream, k = np.broadcast_arrays(np.asarray(stream, np.uint64), np.asarray(k, np.uint64))
    c0, c1 = k >> np.uint64(1), stream & mask
    c2, c3 = np.full(c0.shape, tag & 0xFFFFFFFF, np.uint64), np.full(c0.shape, tag >> 32, np.uint64)
    k0, k1 = np.uint64(key & 0xFFFFFFFF), np.uint64(key >> 32)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c0, np.uint64(0xCD9E8D57) * c2
        c0, c1, c2, c3 = (p1 >> u32) ^ c1 ^ k0, p1 & mask, (p0 >> u32) ^ c3 ^ k1, p0 & mask
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & mask, (k1 + np.uint64(0xBB67AE85)) & mask
    odd = (k & np.uint64(1)) == 1
    bits = (np.where(odd, c3, c1) << u32) | np.where(odd, c2, c0)
    return (bits >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _collide(x, v, w, cell_first, count, sgwm, dt, dx, tag, seed):
    """One NTC step of every cell (equal weights): per candidate the pair, the
    acceptance and, if accepted, an isotropic scatter."""
    d, omega, tref = VHS["Ar,Ar"]
    m = MASS["Ar"]
    factor = math.pi * d ** 2 * (4 * K_B * tref / m) ** (omega - 0.5) / math.gamma(2.5 - omega)
    nc = len(count)
    stream, at = np.arange(nc), np.ones(nc, np.int64)
    n_coll = np.floor(0.5 * dt * count * (count - 1.0) * sgwm / dx + _philox(stream, 0, tag, seed)).astype(int)
    done = np.zeros(nc, np.int64)
    for j in range(int(n_coll.max(initial=0))):
        c = np.flatnonzero(n_coll > j)

        def next_draw(c):
            r = _philox(c, at[c], tag, seed)
            at[c] += 1
            return r

        i = np.floor(next_draw(c) * count[c]).astype(int)
        k = np.floor(next_draw(c) * count[c]).astype(int)
        while (i == k).any():
            same = np.flatnonzero(i == k)
            k[same] = np.floor(next_draw(c[same]) * count[c[same]]).astype(int)
        i, k = cell_first[c] + i, cell_first[c] + k
        g = np.linalg.norm(v[i] - v[k], axis=1)
        c, i, k, g = (a[g > 2.2e-16] for a in (c, i, k, g))
        sgw = factor * g ** (2.0 - 2.0 * omega) * np.maximum(w[i], w[k])
        sgwm[c] = np.maximum(sgwm[c], sgw)
        hit = next_draw(c) < sgw / sgwm[c]
        c, i, k, g = (a[hit] for a in (c, i, k, g))
        done[c] += 1
        phi, ct = 2 * math.pi * next_draw(c), 2.0 * next_draw(c) - 1.0
        stt = np.sqrt(1.0 - ct * ct)
        com = 0.5 * (v[i] + v[k])
        half = 0.5 * g[:, None] * np.stack([stt * np.cos(phi), stt * np.sin(phi), ct], 1)
        v[i], v[k] = com + half, com - half
    return n_coll, done


def _fly(x, v, ids, dt, dx, tag, seed):
    """Free flight with diffuse walls."""
    t, old = np.full(len(x), dt), x[:, 0].copy()
    new, at = old + v[:, 0] * dt, np.zeros(len(x), np.int64)
    vsq = 2 * K_B * T_WALL / MASS["Ar"]
    while True:
        out = np.flatnonzero((new >= L) | (new <= 0))
        if not len(out):
            break
        right = new[out] >= L
        wall = np.where(right, L, 0.0)
        t[out] -= np.abs((wall - old[out]) / v[out, 0])
        r = [_philox(ids[out] - 1, at[out] + j, tag, seed) for j in range(3)]
        at[out] += 3
        vn, vt = (np.sqrt(-vsq * np.log(np.maximum(1e-50, q))) for q in r[:2])
        v[out, 0] = np.where(right, -vn, vn)
        v[out, 1] = vt * np.sin(2 * math.pi * r[2]) + np.where(right, V_WALL, -V_WALL)
        v[out, 2] = vt * np.cos(2 * math.pi * r[2])
        old[out] = wall
        new[out] = wall + v[out, 0] * t[out]
    x[:, 0] = np.clip(new, 1e-12 * dx, L - 1e-12 * dx)


def _exact_operators(case, seed):
    p, nc, m = _inputs(case, seed), case["cells"], MASS["Ar"]
    x, v, w, count, dx = p["x"], p["v"], p["w"], p["counts"].astype(np.int64), L / case["cells"]
    ids = np.arange(1, len(w) + 1)
    d, omega, tref = VHS["Ar,Ar"]
    factor = math.pi * d ** 2 * (4 * K_B * tref / m) ** (omega - 0.5) / math.gamma(2.5 - omega)
    sgwm = factor * math.sqrt(2 * T_WALL * K_B / m) ** (2.0 - 2.0 * omega) * case["ndens"] * dx / count
    series = []
    for t in range(1, 1 + case["steps"]):
        _collide(x, v, w, np.cumsum(count) - count, count, sgwm, case["dt"], dx, (t << 4) | 1, seed)
        _fly(x, v, ids, case["dt"], dx, (t << 4) | 2, seed)
        cell = np.floor(x[:, 0] / dx).astype(int)
        order = np.argsort(cell, kind="stable")
        x, v, w, ids, cell = x[order], v[order], w[order], ids[order], cell[order]
        count = np.bincount(cell, minlength=nc)
        n, vm, temp = _cell_props(w, v, cell, nc, m)
        r = dict(lpa=None, np=count[None].astype(float), n=n[None], v=vm[None], T=temp[None])
        if case["flux"]:
            c = v - vm[cell]

            def per_cell(a):
                return np.stack([np.bincount(cell, w * a[:, j], nc) for j in range(3)], 1)[None] * (m / dx)

            r.update(energy_flux=0.5 * per_cell(c * (c * c).sum(1)[:, None]), diagonal=per_cell(c * c),
                     off_diagonal=per_cell(np.stack([c[:, 0] * c[:, 1], c[:, 0] * c[:, 2], c[:, 1] * c[:, 2]], 1)))
        series.append(r)
    out = dict(series=series, collisions=[dict(sigma_g_w_max=sgwm)])
    if len(w) <= STATE_MAX:
        out["particles"] = [dict(x=x, v=v, w=w)]
    return out
