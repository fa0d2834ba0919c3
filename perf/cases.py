"""The work that users of the library have it do, as cases for timing.

A case is one run of a simulation from a stored state to its next output:
the state is uploaded, the time loop runs on the device and the state comes
back to the host, the way the reference's main program drives its solver
module.  ``prepare`` holds what such a program has in hand before the run
(the context with its grid, bed, source and erodible layer, and the initial
state on the host); ``run`` is one pass through the public entry points.
Every pass starts from the same initial state at t = 0.

Kinds:
  grid      one grid through ``Solver.advance`` (the device-resident time loop)
  calls     one grid through the solver module's procedures one at a time
            (check_solve, timestep, imex_RK_solver, ...), as a host program
            with its own time loop calls them
  ensemble  many member grids through ``Ensemble.advance``

Nothing here says what a step costs the library; ``work`` counts the values
that a step has to read and write and the FP64 operations of the scheme.
"""
import math

import numpy as np

from imex_sflow2d_v2_amd import decks, learned
from imex_sflow2d_v2_amd.params import make_params
from imex_sflow2d_v2_amd.solver import Ensemble, Solver


def listed():
    return [
        # the smallest run: the 1-D dam break of the tests, all launch latency
        dict(name="dam_break_1d", kind="grid", deck="dambreak", nx=400, ny=1, steps=400),
        # the size of the reference's own 2-D test deck, with its rheology
        # (turbulent drag, model 6, the tableau-driven path)
        dict(name="pile_drag_100x68", kind="grid", deck="small", nx=100, ny=68, solids=1, n_rk=2,
             model=6, terrain=False, erosion=False, source=False, steps=200),
        # a host program with its own time loop, one procedure per call:
        # erosion, deposition and a changing bed
        dict(name="calls_200x151", kind="calls", deck="small", nx=200, ny=151, solids=2, n_rk=2,
             model=1, terrain=False, erosion=True, source=False, steps=60),
        # a pulsed vent on a small grid: few wet cells, erosion
        dict(name="vent_257x190", kind="grid", deck="small", nx=257, ny=190, solids=3, n_rk=2,
             model=1, terrain=False, erosion=True, source=True, steps=400),
        # the second-order scheme (IMEX-SSP(3,3,2)) with slope correction and
        # curvature, ragged sizes
        dict(name="ssp3_301x203", kind="grid", deck="small", nx=301, ny=203, solids=2, n_rk=3,
             model=1, terrain=True, erosion=False, source=False, steps=60),
        # a collapse on an incline, wet everywhere
        dict(name="incline_512", kind="grid", deck="incline", nx=512, ny=512, steps=80,
             start="plain"),
        # the same with the learned start of the Newton solves
        dict(name="incline_256_learned", kind="grid", deck="incline", nx=256, ny=256, steps=80,
             start="learned"),
        # the headline run: a vent on a large volcanic DEM, nearly all dry
        dict(name="volcano_2048", kind="grid", deck="volcano", nx=2048, ny=2048, steps=1000),
        # a large grid, wet everywhere, three classes
        dict(name="wet_1000", kind="grid", deck="wet", nx=1000, ny=1000, steps=40),
        # vertical profiles and the closed-form friction (model 8)
        dict(name="profiles_500x386", kind="grid", deck="profiles", nx=500, ny=386, n_rk=2,
             solids=2, quad=20, steps=20),
        # a parameter sweep: members of different sizes advanced together
        dict(name="ensemble_24", kind="ensemble", members=24, n_min=128, n_max=512, steps=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["dambreak", "small", "small", "calls", "vent", "incline", "volcano", "wet",
                       "profiles", "ensemble"])
    if what == "dambreak":
        return dict(kind="grid", deck="dambreak", nx=_log_int(rng, 100, 3000), ny=1,
                    steps=rng.randrange(200, 400))
    if what in ("small", "calls", "vent"):
        nx, ny = _log_int(rng, 60, 360), _log_int(rng, 60, 360)
        c = dict(kind="calls" if what == "calls" else "grid", deck="small", nx=nx, ny=ny,
                 solids=rng.choice([1, 2, 3]), n_rk=2, model=1, terrain=False,
                 erosion=what != "small", source=what == "vent", steps=rng.randrange(30, 60))
        if what == "small":
            c["n_rk"] = rng.choice([2, 3, 4])
            c["model"] = rng.choice([1, 1, 6])
            c["terrain"] = rng.choice([False, True])
        elif what == "vent":
            c["steps"] = rng.randrange(200, 400)
        return c
    if what == "incline":
        n = _log_int(rng, 150, 620)
        return dict(kind="grid", deck="incline", nx=n, ny=n, steps=rng.randrange(30, 60),
                    start=rng.choice(["plain", "plain", "closed"]))
    if what == "volcano":
        n = _log_int(rng, 600, 1900)
        return dict(kind="grid", deck="volcano", nx=n, ny=n, steps=rng.randrange(300, 600))
    if what == "wet":
        n = _log_int(rng, 300, 1000)
        return dict(kind="grid", deck="wet", nx=n, ny=n, steps=rng.randrange(15, 40))
    if what == "profiles":
        return dict(kind="grid", deck="profiles", nx=_log_int(rng, 100, 500),
                    ny=_log_int(rng, 80, 380), n_rk=rng.choice([2, 3]),
                    solids=rng.choice([1, 2, 3]), quad=rng.choice([10, 20]),
                    steps=rng.randrange(8, 16))
    return dict(kind="ensemble", members=rng.randrange(6, 24), n_min=100,
                n_max=_log_int(rng, 200, 520), steps=rng.randrange(25, 60))


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _depth_field(nx, ny, rng, amount=0.2):
    """A smooth positive factor around 1 (random phases and wave numbers)."""
    f = np.ones((nx, ny))
    x = np.arange(nx) / max(nx, 2)
    y = np.arange(ny) / max(ny, 2)
    for _ in range(4):
        a, b = rng.integers(1, 7, 2)
        f += (amount / 4) * np.outer(np.cos(2 * np.pi * (a * x + rng.random())),
                                     np.cos(2 * np.pi * (b * y + rng.random())))
    return f


def _volcano(n, rng):
    """A vent at the summit of a 1500 m cone (3 km radius) with bumps and
    rough ground on a 10.24 km square: dry at first; three classes, erosion,
    deposition and a changing bed."""
    dx = 10240.0 / n
    L = n * dx
    xc = (np.arange(n) + 0.5) * dx
    r2 = ((xc - 0.5 * L) ** 2)[:, None] + ((xc - 0.5 * L) ** 2)[None, :]
    B = 1500.0 * np.clip(1.0 - np.sqrt(r2) / 3000.0, 0.0, None)
    for _ in range(32):
        a, s = rng.uniform(10.0, 80.0), rng.uniform(50.0, 300.0)
        x0, y0 = rng.uniform(0.0, L, 2)
        B += np.outer(a * np.exp(-(xc - x0) ** 2 / (2 * s * s)),
                      np.exp(-(xc - y0) ** 2 / (2 * s * s)))
    for m, rms in ((16, 15.0), (64, 5.0), (256, 1.5)):
        # rough ground: a coarse random grid, interpolated
        g = rng.standard_normal((m + 2, m + 2)) * rms
        u = np.arange(n) * (m / n)
        i, w = u.astype(int), u - u.astype(int)
        g = g[i] * (1 - w)[:, None] + g[i + 1] * w[:, None]
        B += g[:, i] * (1 - w)[None, :] + g[:, i + 1] * w[None, :]
    B = np.maximum(B, 0.0)
    kw = dict(energy_flag=True, cfl=0.24, max_dt=1.0, rho_s=(2500.0,) * 3,
              diam_s=(0.1e-3, 1.0e-3, 4.0e-3), sp_heat_s=(1617.0,) * 3, settling=True,
              erosion_coeff=1.0e-5, erodible_porosity=0.3, erodible_fract=(0.4, 0.4, 0.2),
              T_erodible=300.0, topo_change=True, radial_source=True, T_ambient=300.0)
    alphas = [0.02, 0.02, 0.01]
    hs = decks.h_source_from_mfr(make_params(n, n, dx, 3, **kw), 1.0e6, 10.0, 800.0, alphas, 50.0)
    src = dict(x=0.5 * L, y=0.5 * L, r=50.0, h=hs, vel=10.0, T=800.0, alphas=alphas,
               time_param=(1e9, 1e9, 0.0, 1e9))
    p = make_params(n, n, dx, 3, source=src, **kw)
    # the ring on a window around the vent (the rest of the grid has none)
    w = int(math.ceil(50.0 / dx)) + 4
    j0 = n // 2 - w
    pw = make_params(2 * w, 2 * w, dx, 3, x0=j0 * dx, y0=j0 * dx, source=src, **kw)
    ring = decks.init_source_np(pw)
    sc = np.zeros((n, n), np.int32, order="F")
    bits = np.zeros((n, n), np.uint8, order="F")
    vect = np.zeros((8, n, n), order="F")
    win = slice(j0, j0 + 2 * w)
    sc[win, win], bits[win, win], vect[:, win, win] = ring
    q = np.zeros((p.n_vars, n, n), order="F")
    er = np.ones((3, n, n), order="F")
    return p, np.asfortranarray(B), q, er, (sc, bits, vect), 1e-3


def _inputs(case, rng, seed):
    """params, bed, initial state, erodible layer, source ring and first dt."""
    nx, ny = case["nx"], case["ny"]
    if case["deck"] == "volcano":
        return _volcano(nx, rng)
    if case["deck"] == "dambreak":
        d = decks.dambreak_1d(nx=nx)
    elif case["deck"] == "incline":
        d = decks.incline_2d(n=nx)
    elif case["deck"] == "wet":
        d = decks.wet_2048(n=nx)
    elif case["deck"] == "profiles":
        def convert(p, qp):
            s = Solver(p)
            q = s.qp_to_qc(qp)
            s.close()
            return q
        d = decks.profile_channel(nx=nx, ny=ny, n_rk=case["n_rk"], n_solid=case["solids"],
                                  n_quad=case["quad"], seed=seed % (1 << 31), convert=convert)
        return (d.params, d.B_cent, d.q, None, None, d.dt0)
    else:
        d = decks.small_2d(n=nx, ny=ny, seed=seed % (1 << 31), n_solid=case["solids"],
                           n_rk=case["n_rk"], rheology_model=case["model"],
                           friction_factor=1e-3 if case["model"] == 6 else -1.0,
                           slope_correction=case["terrain"], curvature=case["terrain"],
                           erosion=case["erosion"], topo_change=case["erosion"],
                           source=case["source"], source_time=(20.0, 12.0, 2.0, 1e9))
        if case["source"]:
            # a vent on a dry bed
            d.q[:] = 0.0
    # every conserved variable is proportional to the depth
    d.q *= _depth_field(nx, ny, rng)[None]
    ring = decks.init_source_np(d.params) if d.params.radial_source_flag else None
    er = d.erodible if d.params.erosion_coeff > 0.0 else None
    if er is not None:
        er = np.asfortranarray(er * _depth_field(nx, ny, rng)[None])
    return d.params, d.B_cent, np.asfortranarray(d.q), er, ring, d.dt0


def _loaded(p, B, q, er, ring):
    """A context set up in the order of the reference's main program."""
    s = Solver(p)
    s.set_topography(B)
    if ring is not None:
        s.set_source(*ring)
    s.upload_q(q)
    if er is not None:
        s.upload_erosion(er)
    s.check_solve(True)
    s.post_step(sums=False)
    return s


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "ensemble":
        n = case["members"]
        # the sizes are the case's, the terrain, materials and states the seed's
        sizes = np.exp(np.linspace(math.log(case["n_min"]), math.log(case["n_max"]), n))
        ds = decks.ensemble_members(count=n, seed=int(rng.integers(1 << 31)),
                                    sizes=np.rint(sizes).astype(int))
        ens = Ensemble([d.params for d in ds]).load(ds)
        return dict(case=case, ens=ens, q=[d.q for d in ds], dt0=ds[0].dt0)
    p, B, q, er, ring, dt0 = _inputs(case, rng, seed)
    s = _loaded(p, B, q, er, ring)
    st = dict(case=case, solver=s, q=q, dt0=dt0, erosion=er is not None)
    if case.get("start") == "closed":
        s.set_closed_form_start(True)
    elif case.get("start") == "learned":
        # pairs harvested from the run's own first steps, one short training
        learned.start_harvest(s, 1 << 20)
        s.advance(4, dt0=dt0)
        pairs, _ = learned.harvested(s)
        learned.stop_harvest(s)
        st["mlp"] = learned.Mlp(seed=1)
        st["mlp"].train(pairs, epochs=1, batch=8192, lr=1e-3, seed=2)
        learned.set_warm_start(s, st["mlp"])
    return st


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def _run_calls(s, steps, dt0):
    """The reference main program's time loop (src/IMEX_SfloW2D.f90:337-483)
    on the host, without an output time."""
    t, dt_old, dt_old_old = 0.0, dt0, dt0
    cells, sums = 0, None
    for _ in range(steps):
        cells += s.check_solve(False, t=t)
        dt = s.timestep()
        dt = min(dt, 1.1 * 0.5 * (dt_old + dt_old_old))
        dt_old_old, dt_old = dt_old, dt
        s.imex_RK_solver(dt, t=t)
        s.update_erosion_deposition_cell(dt)
        s.topography_reconstruction()
        t += dt
        sums = s.post_step(sums=True)
    return t, cells, sums


def run(state):
    case = state["case"]
    if case["kind"] == "ensemble":
        ens = state["ens"]
        for m, q in zip(ens.members, state["q"]):
            m.upload_q(q)
        ens.t[:] = 0.0
        ens.advance(case["steps"], dt0=state["dt0"])
        return {"q": [m.q() for m in ens.members], "t": ens.t.copy()}
    s = state["solver"]
    s.upload_q(state["q"])
    s.t = 0.0
    out = {}
    if case["kind"] == "calls":
        out["t"], out["cells"], out["sums"] = _run_calls(s, case["steps"], state["dt0"])
    else:
        out["steps"] = s.advance(case["steps"], dt0=state["dt0"])
        out["t"] = s.t
    out["q"] = s.q()
    if state["erosion"] and case["nx"] * case["ny"] < 1 << 20:
        # the hazard maxima and the deposit go out with the state
        out["hmax"], out["pdyn"], out["speed"], out["vuln"] = s.post()
        out["erodible"], out["deposit"], out["erosion"], out["bed"] = s.erosion_state()
    return out


def exact(case, seed):
    """None: a pass is tens to a thousand dependent steps of the whole scheme
    (limited reconstruction, Newton solves, settling fixed points), in 64
    bits already; in plain numpy a 2-D pass takes minutes."""
    return None


def work(case):
    if case["kind"] == "ensemble":
        sizes = np.exp(np.linspace(math.log(case["n_min"]), math.log(case["n_max"]),
                                   case["members"]))
        cells, ns = float(np.sum(np.rint(sizes) ** 2)), 2
        # a member's column covers about a fifth of its grid, with its margin
        wet = 0.25 * cells
    else:
        cells = float(case["nx"] * case["ny"])
        ns = {"dambreak": 1, "incline": 2, "wet": 3, "volcano": 3}.get(case["deck"],
                                                                     case.get("solids"))
        wet = cells
        if case["deck"] == "small":
            wet = 0.3 * cells
        if case.get("source") or case["deck"] == "volcano":
            # the current spreads from the vent: some ten rings of cells
            wet = min(0.2 * cells, 2000.0)
    nv = 4 + ns
    # per wet cell and step: the state in and out, two bed slopes, the
    # erodible, deposit and erosion layers and the bed in and out, three maxima
    fields = 2 * nv + 2 + 6 * ns + 2 + 6
    stages = {1: 1, 2: 1, 3: 3, 4: 3}[case.get("n_rk", 2)]
    # a step's FP64 operations for one wet cell: reconstruction, fluxes, the
    # implicit solve and the settling speeds; with profiles the depth sums
    flops = 3000.0 * stages
    if case.get("deck") == "profiles":
        flops += 600.0 * case["quad"] * stages
    return {"bytes": 8.0 * (case["steps"] * wet * fields + 2 * cells * nv),
            "flops": flops * case["steps"] * wet}
