"""The work that users of this package have it do, as cases to be timed: whole simulations from initial
conditions to their end time, resident simulations advanced between two outputs, the engine loop driven by
the host step by step, an ensemble in one batch, and a server that takes jobs.

A case is a dict of plain values.  "mode" says which of these it is:

  whole      a new device simulation from the problem (mesh and initial conditions), run to t_end, state fetched
  resident   a simulation that stays on the device: `steps` engine steps, state fetched
  host       the same with the host in charge of the time line: one hfv_step call a step (the drop-in runner)
  ensemble   independent 1D and 2D Riemann problems in one Batch: `steps` launches, every state fetched
  serve      a Server that is handed `count` jobs at once and serves them to their end

and "problem" the initial conditions: the presets of hydro_rs_amd.ics, their jitter drawn from the seed.
"""
import math

import numpy as np

from hydro_rs_amd import ensemble, fvs, ics, serve

PRECISION = {"fp64": fvs.FP64, "fp32": fvs.FP32_FLUX}
# a resident simulation is never meant to end: its time line is far longer than any run
LONG = 1000.0


def listed():
    return [
        # the reference's first example: a short shock tube, moving mesh, exact solver.  1000 cells: the time
        # is the latency of each step's kernels
        dict(name="sod1d_1000_fluid_fp64", mode="whole", problem="sod1d", size=1000, motion="fluid", precision="fp64",
             t_end=0.05),
        # a small fixed-mesh tube (parameter studies run many like it), odd size, FP32 flux
        dict(name="tube1d_333_fp32", mode="whole", problem="tube1d", size=333, motion="fixed", precision="fp32",
             t_end=0.1),
        # a blast on a fixed 2D mesh from start to end: most cells wait, a step moves few of them
        dict(name="sedov2d_256_fp32", mode="whole", problem="sedov2d", size=256, motion="fixed", precision="fp32",
             t_end=0.02),
        # the same blast on the reference's default moving mesh: each step rebuilds the cells it moves
        dict(name="sedov2d_256_steer_fp64", mode="whole", problem="sedov2d", size=256, motion="steer",
             precision="fp64", t_end=0.004),
        # an engine outside this library that calls the step itself, small 2D mesh of odd side
        dict(name="vortex2d_61_host_fp64", mode="host", problem="vortex2d", size=61, motion="fixed",
             precision="fp64", steps=50),
        # the largest served 2D size (an odd side near it), smooth flow, every cell active
        dict(name="vortex2d_509_fp64", mode="resident", problem="vortex2d", size=509, motion="fixed",
             precision="fp64", steps=100),
        # a smooth flow on a moving 2D mesh: nearly every cell is rebuilt in every step
        dict(name="vortex2d_125_steer_fp32", mode="resident", problem="vortex2d", size=125, motion="steer",
             precision="fp32", steps=40),
        # a moving 3D mesh
        dict(name="kh3d_48_steer_fp64", mode="resident", problem="kh3d", size=48, motion="steer", precision="fp64",
             steps=8),
        # fixed 3D meshes, ordinary and large, both precisions
        dict(name="kh3d_96_fp64", mode="resident", problem="kh3d", size=96, motion="fixed", precision="fp64", steps=24),
        dict(name="kh3d_128_fp32", mode="resident", problem="kh3d", size=128, motion="fixed", precision="fp32",
             steps=24),
        # an ensemble of Riemann problems of 200 to 65536 cells in one batch
        dict(name="ensemble_60_fp32", mode="ensemble", count=60, n_min=200, n_max=65536, precision="fp32", steps=128),
        # a server that is handed twelve 2D jobs at once
        dict(name="serve_12_fp32", mode="serve", count=12, side_min=32, side_max=128, precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sod1d", "tube1d", "sedov2d", "sedov2d", "vortex2d", "vortex2d", "kh3d", "kh3d", "ensemble", "serve"])
    precision = rng.choice(["fp64", "fp32"])
    if kind == "sod1d":
        n = _log_int(rng, 200, 2000)
        return dict(mode="whole", problem=kind, size=n, motion="fluid", precision=precision, t_end=40.0 / n)
    if kind == "tube1d":
        n = _log_int(rng, 200, 20000)
        return dict(mode="whole", problem=kind, size=n, motion="fixed", precision=precision, t_end=25.0 / n)
    if kind == "sedov2d":
        side = _log_int(rng, 48, 256)
        if rng.random() < 0.5:
            return dict(mode="whole", problem=kind, size=side, motion="fixed", precision=precision, t_end=5.0 / side)
        return dict(mode="whole", problem=kind, size=side, motion="steer", precision=precision, t_end=1.0 / side)
    if kind == "vortex2d":
        mode = rng.choice(["resident", "resident", "host"])
        motion = rng.choice(["fixed", "steer"]) if mode == "resident" else "fixed"
        side = _log_int(rng, 48, 180 if motion != "fixed" else 512)
        return dict(mode=mode, problem=kind, size=side, motion=motion, precision=precision,
                    steps=40 if motion != "fixed" or mode == "host" else 80)
    if kind == "kh3d":
        if rng.random() < 0.5:
            return dict(mode="resident", problem=kind, size=rng.randint(40, 54), motion="steer", precision=precision,
                        steps=8)
        return dict(mode="resident", problem=kind, size=rng.randint(72, 120), motion="fixed", precision=precision,
                    steps=24)
    if kind == "ensemble":
        return dict(mode="ensemble", count=rng.randint(8, 60), n_min=200, n_max=_log_int(rng, 2000, 65536),
                    precision=precision, steps=128)
    return dict(mode="serve", count=rng.randint(4, 16), side_min=32, side_max=rng.randint(64, 160), precision=precision)


def _problem(case, seed):
    precision = PRECISION[case["precision"]]
    kind, size = case["problem"], case["size"]
    t_end = case.get("t_end", LONG)
    if kind == "sod1d":
        p = ics.sod_1d(size, seed=seed, t_end=t_end, precision=precision)
    elif kind == "tube1d":
        p = ics.riemann_tube_1d(size, 1.0, 1.0, 0.0, 0.125, 0.1, 0.0, 1.4, seed=seed, t_end=t_end, precision=precision)
    elif kind == "sedov2d":
        p = ics.sedov_2d(size, seed=seed, t_end=t_end, precision=precision)
    elif kind == "vortex2d":
        # (a weak vortex, and a slow shear in 3D: a resident simulation has to stay smooth for as many passes as
        # anyone makes, and after thousands of steps the presets' own strengths reach states the scheme refuses)
        p = ics.isentropic_vortex_2d(size, seed=seed, t_end=t_end, beta=1.0, precision=precision)
    else:
        p = ics.kelvin_helmholtz_3d(size, seed=seed, t_end=t_end, precision=precision)
        p.vel *= 0.2
    p.cfg.motion = fvs.MOTIONS[case["motion"]]
    return p


def _sizes(lo, hi, count):
    """`count` sizes spread over the logarithm of [lo, hi], both among them, in no order."""
    sizes = [int(round(math.exp(math.log(lo) + (math.log(hi) - math.log(lo)) * k / max(1, count - 1))))
             for k in range(count)]
    order = np.random.default_rng(0).permutation(count)
    return [sizes[k] for k in order]


def _members(case, seed):
    """ensemble.ensemble_problems' distribution of states at sizes that are the case's own."""
    rng = np.random.default_rng(seed)
    out = []
    for k, n in enumerate(_sizes(case["n_min"], case["n_max"], case["count"])):
        rho = np.exp(rng.uniform(np.log(0.1), np.log(10.0), 2))
        p = np.exp(rng.uniform(np.log(0.01), np.log(10.0), 2))
        v = rng.uniform(-1.0, 1.0, 2)
        gamma = 1.4 if rng.random() < 0.5 else 5.0 / 3.0
        sub = int(rng.integers(0, 1 << 30))
        tube, size = (ics.riemann_tube_1d, n) if k % 2 == 0 else (ensemble.riemann_tube_2d, max(4, round(math.sqrt(n))))
        out.append(tube(size, rho[0], p[0], v[0], rho[1], p[1], v[1], gamma, seed=sub, t_end=LONG,
                        precision=PRECISION[case["precision"]]))
    return out


def _jobs(case, seed):
    """serve.served_jobs' two kinds in turn, at sides that are the case's own, all waiting at the start."""
    rng = np.random.default_rng(seed)
    out = []
    for k, side in enumerate(_sizes(case["side_min"], case["side_max"], case["count"])):
        sub, precision = int(rng.integers(0, 1 << 30)), PRECISION[case["precision"]]
        if k % 2 == 0:
            out.append(("sedov", ics.sedov_2d(side, seed=sub, t_end=0.01, gamma=1.4, precision=precision)))
        else:
            out.append(("vortex", ics.isentropic_vortex_2d(side, seed=sub, t_end=0.2, gamma=1.4, precision=precision)))
    return out


def prepare(case, seed):
    mode = case["mode"]
    if mode == "ensemble":
        return {"mode": mode, "steps": case["steps"], "batch": fvs.Batch.for_problems(_members(case, seed))}
    if mode == "serve":
        return {"mode": mode, "jobs": _jobs(case, seed), "server": serve.Server(2 << 30)}
    prob = _problem(case, seed)
    if mode == "whole":
        return {"mode": mode, "problem": prob}
    state = {"mode": mode, "steps": case["steps"], "sim": ics.build_device_sim(prob)}
    if mode == "host":
        state["time_base"] = state["sim"].engine_info()["time_base"]
        state["ti"] = (0, 0)
    return state


def _counts(info):
    return np.array([info[k] for k in ("step_count", "cell_updates", "face_fluxes", "ti_current", "ti_next")],
                    dtype=np.int64)


def run(state):
    mode = state["mode"]
    if mode == "ensemble":
        b = state["batch"]
        b.run(state["steps"])
        return {"prim": [b.get_state(s, ["prim"])["prim"] for s in range(b.nslots)],
                "counts": np.stack([_counts(b.engine_info(s)) for s in range(b.nslots)])}
    if mode == "serve":
        jobs = [serve.Job(k, 0.0, prob, kind) for k, (kind, prob) in enumerate(state["jobs"])]
        done = sorted(state["server"].serve(jobs), key=lambda j: j.jid)
        return {"prim": [j.result["prim"] for j in done],
                "counts": np.array([[j.steps, j.cell_updates, j.error_code] for j in done], dtype=np.int64)}
    if mode == "whole":
        sim = ics.build_device_sim(state["problem"])
        sim.run()
        out = sim.get_state(["prim", "grad", "cons", "loc", "timebin"])
        out["counts"] = _counts(sim.engine_info())
        sim.close()
        return out
    sim = state["sim"]
    if mode == "host":
        old, now = state["ti"]
        for _ in range(state["steps"]):
            old, now = now, sim.step(sim.timestep_info(old, now, state["time_base"]))
        state["ti"] = (old, now)
        out = sim.get_state(["prim", "grad", "cons", "timebin"])
        out["ti_next"] = now
        return out
    sim.run(state["steps"])
    out = sim.get_state(["prim", "timebin"])
    out["counts"] = _counts(sim.engine_info())
    return out


# ---- the least that a pass has to move and compute: per update of a cell its state, gradients, extrapolations
# and geometry once in and once out, and per face of it the face's geometry and index pair
FACES = {1: 1.0, 2: 3.0, 3: 7.8}  # faces a cell: of a 2D or 3D Voronoi mesh each face has two cells


def _update(dim, precision):
    real = 4 if precision == "fp32" else 8
    return {"bytes": 2 * (10 * 8 + 20 * real) + 64 + FACES[dim] * 64, "flops": 350.0 * FACES[dim] + 120.0 * FACES[dim] + 300}


def _updates(case):
    """(dimension, about how many cell updates a pass makes)."""
    if case["mode"] == "ensemble":
        cells = sum(_sizes(case["n_min"], case["n_max"], case["count"]))
        return 2, 0.7 * cells * case["steps"]
    if case["mode"] == "serve":
        sides = _sizes(case["side_min"], case["side_max"], case["count"])
        return 2, sum(s * s * s * (0.3 if k % 2 == 0 else 1.0) for k, s in enumerate(sides))
    n = case["size"]
    if case["problem"] == "sod1d":
        return 1, 0.57 * n * 41 * case["t_end"] * n
    if case["problem"] == "tube1d":
        return 1, 0.75 * n * 31 * case["t_end"] * n
    if case["problem"] == "sedov2d":  # the blast's cells grow as its radius does
        return 2, 25.0 * n ** 1.75 * case["t_end"] * 20 * n ** 0.5
    if case["problem"] == "vortex2d":
        return 2, 1.0 * n * n * case["steps"]
    return 3, 0.8 * n ** 3 * case["steps"]


def work(case):
    dim, updates = _updates(case)
    return {k: v * updates for k, v in _update(dim, case["precision"]).items()}


def exact(case, seed):
    """None: a pass is tens to thousands of steps of a nonlinear scheme with a time step of its own for every
    cell, on a mesh that this package tessellates; its outputs have no value apart from the scheme itself."""
    return None
