"""The work that is timed: what programs have this library do, through its
public entry points (the ctypes binding of the C ABI).

Kinds of case

* ``steps``: time steps of a mesh resident on the GPU (Gpu.run), a regrid
  interval's ten or near that, then the instances' times.  A solver spends
  most of its time here.  Sizes run from one small uniform forest, where
  launches count, over single adaptive problems to batches of 64 adaptive
  problems and meshes far larger than the caches; patches of 2x2 to 16x16
  cells; every time scheme; periodic, transmissive, slip and no-slip walls.
* ``seam``: one interval of a host-resident solver (physics_go_gpu): the
  reference-format arrays go in, its steps run, the solution comes back.
* ``rhs``: the residual and the CFL time step of host arrays
  (physics_rhs_structured_gpu, physics_time_step_gpu), the entry points of a
  solver that keeps its own time integration.
* ``evolve``: an adaptive run from its initial condition to a physical time
  (amr_evolve_device; with several instances amr_evolve_batch).
* ``train``: one epoch of the learned tagger's training over a labelled set.
* ``tag``: what a regrid asks of a resident state: the density-gradient
  indicator, the feature rows and classes of the learned tagger, and the
  reference's density thresholds.

The data are synthetic: seeded four-state fronts, waves and vortices with
densities and pressures of order one, on meshes refined along the fronts.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "amr-demo_amd"))
import amrhip  # noqa: E402

STEPS = 10                  # steps between regrids, the benchmark's interval, where a case names no other
STAGES = {1: 1, 2: 2, 3: 3, 4: 4, 5: 5}
# state vectors read and written per cell by one step of each scheme (32 B
# each): a stage reads its state and, where the scheme has one, the base
# state or the accumulator, and writes its state (and the accumulator)
VECTORS = {1: 2, 2: 2 + 3, 3: 2 + 3 + 3, 4: 3 + 5 + 5 + 4, 5: 3 + 4 * 4}
FACE_FLOPS = 110            # one upwind face flux with its two primitive states
DT_OVER_H = 0.12            # step limit, in finest cells, of the scheme that takes no CFL minimum
NIN, NH, NOUT = 384, 64, 3  # the tagger's layers


def listed():
    return [
        # a small uniform forest: launches and waits count
        {"name": "steps small vortex", "kind": "steps", "mesh": "vortex", "n": 8, "scheme": 3, "lmin": 4, "lmax": 4,
         "inst": 1, "bc": 0},
        # one adaptive problem: a mesh that fits the last-level cache
        {"name": "steps one problem", "kind": "steps", "mesh": "fronts", "n": 8, "scheme": 3, "lmin": 3, "lmax": 7,
         "inst": 1, "bc": 0},
        # the benchmark's workload: 64 adaptive problems in the same launches
        {"name": "steps batch of 64", "kind": "steps", "mesh": "fronts", "n": 8, "scheme": 3, "lmin": 3, "lmax": 8,
         "inst": 64, "bc": 0},
        # the largest: a uniform mesh several times the last-level cache
        {"name": "steps large vortex", "kind": "steps", "mesh": "vortex", "n": 8, "scheme": 3, "lmin": 8, "lmax": 8,
         "inst": 2, "bc": 0},
        # large patches, five-stage low-storage scheme, slip walls
        {"name": "steps large patches", "kind": "steps", "mesh": "fronts", "n": 16, "scheme": 5, "lmin": 4, "lmax": 7,
         "inst": 6, "bc": 1},
        # small patches (many quadrants), two-stage scheme, no-slip walls
        {"name": "steps small patches", "kind": "steps", "mesh": "fronts", "n": 4, "scheme": 2, "lmin": 4, "lmax": 8,
         "inst": 8, "bc": 2},
        # a host-resident solver's interval
        {"name": "seam interval", "kind": "seam", "mesh": "fronts", "n": 8, "scheme": 3, "lmin": 3, "lmax": 7,
         "inst": 1, "bc": 0},
        # residual and time step alone, small arrays
        {"name": "host residual", "kind": "rhs", "mesh": "fronts", "n": 4, "scheme": 3, "lmin": 3, "lmax": 6,
         "inst": 1, "bc": 1},
        # an adaptive run, and a batch of them
        {"name": "adaptive run", "kind": "evolve", "mesh": "riemann4", "n": 8, "scheme": 3, "lmin": 3, "lmax": 7,
         "inst": 1, "bc": 0, "t_end": 0.05},
        {"name": "adaptive batch", "kind": "evolve", "mesh": "riemann4", "n": 8, "scheme": 3, "lmin": 3, "lmax": 7,
         "inst": 16, "bc": 0, "t_end": 0.03},
        # the tagger learns, and answers at a regrid
        {"name": "tagger epoch", "kind": "train", "rows": 65536, "batch": 4096},
        {"name": "regrid tags", "kind": "tag", "mesh": "fronts", "n": 8, "scheme": 3, "lmin": 3, "lmax": 8,
         "inst": 32, "bc": 0},
    ]


def draw(rng):
    kind = rng.choice(["steps"] * 6 + ["seam", "rhs", "evolve", "train", "tag", "tag"])
    if kind == "train":
        batch = 64 * int(round(2 ** rng.uniform(2, 6.6)))
        return {"kind": kind, "rows": int(batch * rng.uniform(2, 16)), "batch": batch}
    if kind == "evolve":
        return {"kind": kind, "mesh": "riemann4", "n": rng.choice([8, 8, 8, 16]), "scheme": 3,
                "lmin": rng.choice([2, 3]), "lmax": rng.choice([5, 6]), "inst": rng.choice([1, 1, 3, 7]), "bc": 0,
                "t_end": round(rng.uniform(0.01, 0.03), 4)}
    n = rng.choice([8, 16]) if kind == "tag" else rng.choice([2, 4, 8, 8, 8, 16, 16])
    mesh = "fronts" if kind in ("tag", "seam", "rhs") else rng.choice(["fronts", "fronts", "vortex"])
    top = {2: 9, 4: 8, 8: 8, 16: 7}[n] - (1 if kind in ("seam", "rhs") else 0)
    if mesh == "vortex":
        lmin = lmax = rng.randint(3, top - 1)
    else:
        lmax = rng.randint(4, top)
        lmin = rng.randint(2, min(4, lmax - 1))
    # as many instances as keep the mesh below the largest listed one
    most = {2: 8, 4: 16, 8: 40, 16: 12}[n] if mesh == "fronts" else 2
    inst = 1 if kind in ("seam", "rhs") else max(1, int(round(math.exp(rng.uniform(0.0, math.log(most))))))
    return {"kind": kind, "mesh": mesh, "n": n, "scheme": rng.choice([1, 2, 3, 3, 3, 4, 5]), "lmin": lmin,
            "lmax": lmax, "inst": inst, "bc": rng.choice([0, 0, 1, 2]), "steps": rng.randint(5, 16),
            "fronts": rng.randint(2, 4)}


# ---------------------------------------------------------------------------
# meshes and states
# ---------------------------------------------------------------------------
def _fronts(n, lmin, lmax, fronts, place, rng):
    """a unit-box forest refined along circular fronts, which `place` sets,
    and a state from `rng`: inside and outside of each front other densities,
    velocities and pressures, with waves on top"""
    f = amrhip.Forest(1, 1, (0, 0), 0.0, 0.0, 1.0, n, lmin, lmax)
    front = np.array([[place.uniform(0.15, 0.85), place.uniform(0.15, 0.85), place.uniform(0.1, 0.35)]
                      for _ in range(fronts)])
    while True:
        nbr, level, org = f.mesh_table()
        size = np.ldexp(1.0, -level)
        mid = org.reshape(-1, 2) + 0.5 * size[:, None]
        gap = np.abs(np.hypot(mid[:, None, 0] - front[:, 0], mid[:, None, 1] - front[:, 1]) - front[:, 2]).min(axis=1)
        flags = (gap < 0.8 * size) & (level < lmax)
        if not flags.any():
            break
        f.refine(flags.astype(np.int32))
        f.balance()
    s = (np.arange(n) + 0.5) / n
    org = org.reshape(-1, 2)
    x = (org[:, 0, None] + size[:, None] * s)[:, None, :]            # (nq, 1, n)
    y = (org[:, 1, None] + size[:, None] * s)[:, :, None]            # (nq, n, 1)
    one = np.ones((level.size, n, n))
    rho, u, v, p = (a * one for a in (rng.uniform(0.6, 1.2), rng.uniform(-0.4, 0.4), rng.uniform(-0.4, 0.4),
                                       rng.uniform(0.6, 1.2)))
    for cx, cy, r in front:
        inside = (x - cx) ** 2 + (y - cy) ** 2 < r * r
        rho = rho + inside * rng.uniform(0.1, 0.5)
        p = p + inside * rng.uniform(0.1, 0.6)
        u = u + inside * rng.uniform(-0.3, 0.3)
        v = v + inside * rng.uniform(-0.3, 0.3)
    kx, ky = rng.randint(2, 6), rng.randint(2, 6)
    wave = np.sin(2 * math.pi * kx * x) * np.cos(2 * math.pi * ky * y)
    rho = rho * (1.0 + 0.05 * wave)
    u = u + 0.05 * wave
    q = f.soln()
    q[..., 0], q[..., 1], q[..., 2] = rho, rho * u, rho * v
    q[..., 3] = p / 0.4 + 0.5 * rho * (u * u + v * v)
    return f


def _vortex(n, level, rng):
    f = amrhip.Forest(1, 1, (1, 1), 0.0, 0.0, 10.0, n, level, level)
    f.apply_ic(amrhip.vortex_ic(strength=rng.uniform(4.0, 5.5), xo=rng.uniform(3.0, 7.0), yo=rng.uniform(3.0, 7.0)))
    return f


def _forests(case, seed):
    # the seed gives the states; the fronts lie where the case alone says, so
    # that its mesh is one size
    rng, place = random.Random(int(seed) * 7919 + 17), random.Random(case["n"] * 64 + case["lmax"])
    out = []
    for k in range(case["inst"]):
        if case["mesh"] == "vortex":
            out.append(_vortex(case["n"], case["lmax"], rng))
        else:
            # a batch's problems differ in their finest level, as the benchmark's do
            top = case["lmax"] - (k % 4 if case["inst"] > 1 else 0)
            out.append(_fronts(case["n"], case["lmin"], max(top, case["lmin"] + 1), case.get("fronts", 3), place, rng))
    return out


def _scale(case):
    return 10.0 if case["mesh"] == "vortex" else 1.0


def _cfl(case):
    return 0.25 * 0.4 * case["scheme"]


def _dt_cap(case):
    return DT_OVER_H * _scale(case) / (case["n"] << case["lmax"]) if case["scheme"] == 2 else 1.0


def _insts(case):
    bc = (case["bc"],) * 4
    return [amrhip.make_inst(_scale(case), bc, _cfl(case), _dt_cap(case)) for _ in range(case["inst"])]


def _steps(case):
    return case.get("steps", STEPS)


def _params(case, **kw):
    far = 2 ** 31 - 1
    given = dict(nelem_subgrid=case["n"], time_scheme=case["scheme"], time_steps=10 ** 9, dt=_dt_cap(case),
                 cfl=_cfl(case), coarse_grid_h=_scale(case), regrid_interval=_steps(case), checkpoint_interval=far,
                 visualization_interval=far, bc=(case["bc"],) * 4 + (1, 1), t_end=0.0, verbose=0)
    given.update(kw)
    amrhip.set_params(**given)


class _Device:
    """device memory of a context, for torch to look at; keeps the context"""

    def __init__(self, gpu, address, count):
        self.gpu = gpu
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f8", "data": (address, False), "version": 2}


def _state_view(gpu, views):
    """the context's state in its own layout, where it lies"""
    U, nq, n = ctypes.c_void_p(), ctypes.c_int(), ctypes.c_int()
    amrhip.check(amrhip.lib().amrgpu_device_state(gpu.h, ctypes.byref(U), None, ctypes.byref(nq), ctypes.byref(n), None),
                 "amrgpu_device_state")
    if U.value not in views:
        views[U.value] = torch.as_tensor(_Device(gpu, U.value, nq.value * 4 * n.value ** 2), device="cuda")
    return views[U.value]


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _prepare_resident(case, seed):
    fs = _forests(case, seed)
    ci, fi, geom, soln, cinst = amrhip.batch_external(fs)
    g = amrhip.Gpu()
    g.setup(case["n"], case["scheme"], _insts(case), ci, fi, geom, soln, cinst)
    return {"case": case, "gpu": g, "views": {}}


def _ints(**kw):
    return {k: ctypes.c_int(int(v)) for k, v in kw.items()}


def _prepare_host(case, seed):
    f = _forests(case, seed)[0]
    ci, fi, geom, soln = f.external()
    n = case["n"]
    i = _ints(dim=2, uns=0, nf=4, n=n, ncell=ci.size // 3, ngh=0, nface=fi.size // 11, dof=soln.size, zero=0)
    return {"case": case, "ci": ci, "fi": fi, "geom": geom, "soln": soln, "q": soln.copy(), "rhs": np.empty_like(soln),
            "i": i}


def _labelled_rows(rows, seed):
    """feature rows as the tagger sees them (channels of size at most one,
    smooth over the patch, a front through some) with their classes"""
    r = np.random.default_rng(int(seed))
    jump = r.random(rows, dtype=np.float32) ** 3
    angle = r.random(rows, dtype=np.float32) * np.float32(2 * math.pi)
    s = (np.arange(8, dtype=np.float32) - 3.5) / 4
    side = np.cos(angle)[:, None, None] * s[None, None, :] + np.sin(angle)[:, None, None] * s[None, :, None] > 0.1
    X = np.empty((rows, 6, 8, 8), np.float32)
    for c in range(4):
        a = (r.random(rows, dtype=np.float32) * 2 - 1)[:, None, None] if c in (1, 2) else np.float32(1.0)
        X[:, c] = a * (1 - jump[:, None, None] * side)
    X[:, 4] = np.gradient(X[:, 0], axis=2)
    X[:, 5] = np.gradient(X[:, 0], axis=1)
    X += r.standard_normal((rows, 1, 8, 8), dtype=np.float32) * np.float32(0.01)
    bits = X.reshape(rows, NIN).view(np.uint32)
    bf = ((bits + 0x7FFF + ((bits >> 16) & 1)) >> 16).astype(np.uint16)
    y = np.where(jump > 0.3, 2, np.where(jump > 0.05, 1, 0)).astype(np.int32)
    return bf, y


def prepare(case, seed):
    kind = case["kind"]
    if kind == "steps":
        return _prepare_resident(case, seed)
    if kind in ("seam", "rhs"):
        return _prepare_host(case, seed)
    if kind == "evolve":
        return {"case": case, "seeds": [1000 + (int(seed) * 131 + k) % 100000 for k in range(case["inst"])]}
    if kind == "train":
        X, y = _labelled_rows(case["rows"], seed)
        ts = amrhip.Tagset()
        ts.append(X, y)
        m = amrhip.Mlp(int(seed) % 1000)
        return {"case": case, "set": ts, "mlp": m, "start": m.params(), "seed": int(seed) % 1000}
    s = _prepare_resident(case, seed)
    s["mlp"] = amrhip.Mlp(int(seed) % 1000)
    s["X"] = torch.empty((s["gpu"].nquad(), NIN), dtype=torch.int16, device="cuda")
    return s


def run(s):
    case = s["case"]
    return {"steps": _run_steps, "seam": _run_seam, "rhs": _run_rhs, "evolve": _run_evolve, "train": _run_train,
            "tag": _run_tag}[case["kind"]](s, case)


def _run_steps(s, case):
    norm = s["gpu"].run(_steps(case))
    t, dt = s["gpu"].time()
    return {"state": _state_view(s["gpu"], s["views"]), "t": t, "dt": dt, "norm": norm}


def _run_seam(s, case):
    _params(case)
    np.copyto(s["q"], s["soln"])
    i = s["i"]
    flags = [ctypes.c_int(0) for _ in range(5)]                 # istep, regrid, visualize, checkpoint, evolve
    flags[4].value = 1
    sec = [ctypes.c_double(0.0) for _ in range(3)]
    zero = np.zeros(1, np.int32)
    by = ctypes.byref
    rc = amrhip.lib().physics_go_gpu(
        by(i["dim"]), by(i["uns"]), by(i["nf"]), by(i["n"]), by(i["ncell"]), by(i["ngh"]), by(i["nface"]),
        by(i["dof"]), amrhip.ipt(s["ci"]), amrhip.ipt(s["fi"]), by(i["zero"]), by(i["zero"]), amrhip.ipt(zero),
        amrhip.ipt(zero), amrhip.ipt(zero), amrhip.dpt(s["geom"]), amrhip.dpt(s["q"]), *[by(f) for f in flags], None,
        *[by(x) for x in sec])
    amrhip.check(rc, "physics_go_gpu")
    return {"state": s["q"], "t": amrhip.lib().physics_gpu_time(), "flags": [f.value for f in flags]}


def _run_rhs(s, case):
    _params(case)
    i, by, L = s["i"], ctypes.byref, amrhip.lib()
    dt = ctypes.c_double(1.0)
    amrhip.check(L.physics_time_step_gpu(by(i["dim"]), by(i["nf"]), by(i["n"]), by(i["ncell"]), amrhip.ipt(s["ci"]),
                                         amrhip.dpt(s["geom"]), amrhip.dpt(s["soln"]), by(dt)), "physics_time_step_gpu")
    amrhip.check(L.physics_rhs_structured_gpu(by(i["dim"]), by(i["nf"]), by(i["n"]), by(i["ncell"]),
                                              amrhip.ipt(s["ci"]), amrhip.dpt(s["geom"]), by(i["nface"]),
                                              amrhip.ipt(s["fi"]), by(i["dof"]), amrhip.dpt(s["soln"]),
                                              amrhip.dpt(s["rhs"])), "physics_rhs_structured_gpu")
    return {"rhs": s["rhs"], "dt": dt.value}


def _run_evolve(s, case):
    _params(case, t_end=case["t_end"])
    tol = 0.1
    fs = []
    for k, seed in enumerate(s["seeds"]):
        top = case["lmax"] - (k % 4 if case["inst"] > 1 else 0)
        ic = amrhip.riemann4_ic(seed)
        f = amrhip.Forest(1, 1, (0, 0), 0.0, 0.0, 1.0, case["n"], case["lmin"], max(top, case["lmin"] + 1))
        f.apply_ic(ic)
        f.regrid_initial(ic, tol)
        fs.append(f)
    if case["inst"] == 1:
        st = fs[0].evolve_device(tol, _steps(case))
    else:
        insts = [amrhip.make_inst(1.0, (case["bc"],) * 4, _cfl(case), _dt_cap(case), case["t_end"]) for _ in fs]
        _, st = amrhip.evolve_batch(fs, insts, tol, _steps(case))
    # the final states and levels, in arrays that any run's mesh fits
    size = case["n"] ** 2 * 4
    state, level = np.zeros(case["inst"] * 4 ** case["lmax"] * size), np.zeros(case["inst"] * 4 ** case["lmax"], np.int32)
    at = 0
    for f in fs:
        nq = f.nquad
        state[at * size:(at + nq) * size] = f.soln().reshape(-1)
        level[at:at + nq] = f.levels()
        at += nq
    return {"state": state, "level": level, "quads": at, "steps": st.steps, "regrids": st.regrids, "t": st.t}


def _run_train(s, case):
    s["mlp"].set_params(s["start"])
    loss = s["mlp"].train(s["set"], epochs=1, batch=case["batch"], lr=2e-3, cw=(1.0, 1.0, 2.0), seed=s["seed"])
    return {"loss": loss, "params": s["mlp"].params()}


def _run_tag(s, case):
    g = s["gpu"]
    ind = g.indicator()
    amrhip.check(amrhip.lib().amrgpu_tagger_features(g.h, ctypes.c_void_p(s["X"].data_ptr())), "amrgpu_tagger_features")
    cls = s["mlp"].predict_ctx(g)
    tags = g.feature_tags([1, 2], [0.8, 1.3])
    return {"indicator": ind, "features": s["X"], "classes": cls, "tags": tags}


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def _quads(case):
    """quadrants of a case's mesh (the fronts': of a mesh of those sizes)"""
    if case["mesh"] == "vortex":
        return case["inst"] * 4 ** case["lmax"]
    fs = _forests(dict(case, inst=min(case["inst"], 4)), 1)
    return sum(f.nquad for f in fs) * case["inst"] // len(fs)


def work(case):
    kind = case["kind"]
    if kind == "train":
        rows = case["rows"] // case["batch"] * case["batch"]
        weights = NIN * NH + NH * NH + NH * NOUT
        return {"bytes": rows * (2.0 * NIN + 8) + rows // case["batch"] * 24.0 * weights,
                "flops": rows * 2.0 * (3 * weights - NIN * NH)}
    if kind == "evolve":
        # the steps a mesh of the finest cells takes to t_end at wave speeds
        # of about 2.5, on about as many quadrants as the fronts need
        cells = _quads(dict(case, mesh="fronts")) * case["n"] ** 2 * 0.6
        steps = case["t_end"] * 2.5 * case["n"] * 2 ** case["lmax"] / _cfl(case)
        return {"bytes": cells * steps * 32.0 * VECTORS[3], "flops": cells * steps * 3 * 2 * FACE_FLOPS}
    cells = _quads(case) * case["n"] ** 2
    if kind == "tag":
        rows = cells // case["n"] ** 2
        return {"bytes": cells * (8.0 + 32 + 8) + rows * (2.0 * NIN + 16),
                "flops": rows * 2.0 * (NIN * NH + NH * NH + NH * NOUT) + cells * 20.0}
    if kind == "rhs":
        return {"bytes": cells * 32.0 * 3, "flops": cells * 2.0 * FACE_FLOPS}
    stages = STAGES[case["scheme"]] * _steps(case)
    return {"bytes": cells * 32.0 * (VECTORS[case["scheme"]] * _steps(case) + (2 if kind == "seam" else 0)),
            "flops": cells * stages * 2.0 * FACE_FLOPS}


# ---------------------------------------------------------------------------
# the same in plain numpy / torch, 64 bits
# ---------------------------------------------------------------------------
def _face_table(ncell, fi):
    """neighbour a (and b, on the coarse side of a hanging face) of every
    quadrant side from the reference-format face list; -1: none"""
    a = np.full((ncell, 4), -1, np.int64)
    b = np.full((ncell, 4), -1, np.int64)
    fi = fi.reshape(-1, 11)
    two = fi[fi[:, 0] == 2]
    a[two[:, 2], two[:, 1]] = two[:, 3]
    a[two[:, 3], two[:, 1] ^ 1] = two[:, 2]
    hang = fi[fi[:, 0] == 3]
    a[hang[:, 2], hang[:, 1]] = hang[:, 3]
    b[hang[:, 2], hang[:, 1]] = hang[:, 4]
    a[hang[:, 3], hang[:, 1] ^ 1] = hang[:, 2]
    a[hang[:, 4], hang[:, 1] ^ 1] = hang[:, 2]
    return a, b


def _prims(q):
    r, u, v, e = q[0], q[1] / q[0], q[2] / q[0], q[3]
    p = 0.4 * (e - 0.5 * r * (u * u + v * v))
    return r, u, v, p, (e + p) / r


def _upwind(L, R, x):
    """flux in the face's frame turned back: states (4, ...) left and right"""
    k, m = (1, 2) if x else (2, 1)
    L, R = np.stack([L[0], L[k], L[m], L[3]]), np.stack([R[0], R[k], R[m], R[3]])
    rl, ul, vl, pl, hl = _prims(L)
    rr, ur, vr, pr, hr = _prims(R)
    wl, wr = np.sqrt(rl), np.sqrt(rr)
    u, v, h = ((x1 * wl + x2 * wr) / (wl + wr) for x1, x2 in ((ul, ur), (vl, vr), (hl, hr)))
    rho = wl * wr
    c = np.sqrt(0.4 * (h - 0.5 * (u * u + v * v)))
    b1 = np.maximum(np.maximum(u + c, ur + c), 0.0)
    b2 = np.minimum(np.minimum(u - c, ul - c), 0.0)
    mc = 1.0 / (1.0 + np.abs(u / c))
    d1 = (rr - rl) - (pr - pl) / (c * c)
    fl = np.stack([L[1], L[1] * ul + pl, L[1] * vl, (L[3] + pl) * ul])
    fr = np.stack([R[1], R[1] * ur + pr, R[1] * vr, (R[3] + pr) * ur])
    jump = np.stack([rr - rl, R[1] - L[1], R[2] - L[2], rr * hr - rl * hl])
    weak = np.stack([d1, d1 * u, d1 * v + rho * (vr - vl), d1 * h + rho * (hr - hl)])
    F = (b1 * fl - b2 * fr + b1 * b2 * (jump - mc * weak)) / (b1 - b2)
    return np.stack([F[0], F[k], F[m], F[3]])


def _wall(Q, bc, x):
    r, u, v, p, _ = _prims(Q)
    if bc == 1:
        un = 0.0 * u
        ut = v if x else u
        p = 0.4 * (Q[3] - 0.5 * r * ut * ut)
    elif bc == 2:
        un = 0.0 * u
        ut = un
        p = 0.4 * (Q[3] - 0.5 * r * (u * u + v * v))
    else:
        un, ut = (u, v) if x else (v, u)
    e = Q[3] - (0.5 * r * (u * u + v * v) if bc == 2 else 0.0)
    F = [r * un, r * un * un + p, r * un * ut, un * (e + p)]
    return np.stack([F[0], F[1], F[2], F[3]] if x else [F[0], F[2], F[1], F[3]])


def _residual(Q, a, b, h, bc):
    """-R/V of Q (4, quads, n, n) over the face table"""
    n = Q.shape[2]
    h = h[:, None]

    def near(which, s):       # the edge cells next to side s
        return [which[:, :, :, 0], which[:, :, :, n - 1], which[:, :, 0, :], which[:, :, n - 1, :]][s]

    def face(s, mine, other):
        return _upwind(other, mine, s < 2) if s in (0, 2) else _upwind(mine, other, s < 2)

    edge = []
    for s in range(4):
        mine = near(Q, s)
        far = near(Q, s ^ 1)
        F = face(s, mine, far[:, np.maximum(a[:, s], 0)]) * np.where(b[:, s] >= 0, 0.5, 1.0)[:, None]
        k = np.nonzero(b[:, s] >= 0)[0]
        F[:, k] += 0.5 * face(s, mine[:, k], far[:, b[k, s]])
        k = np.nonzero(a[:, s] < 0)[0]
        F[:, k] = _wall(mine[:, k], bc, s < 2)
        edge.append(F * h)
    fx = _upwind(Q[:, :, :, :-1], Q[:, :, :, 1:], True) * h[:, :, None]
    fy = _upwind(Q[:, :, :-1, :], Q[:, :, 1:, :], False) * h[:, :, None]
    fx = np.concatenate([edge[0][:, :, :, None], fx, edge[1][:, :, :, None]], axis=3)
    fy = np.concatenate([edge[2][:, :, None, :], fy, edge[3][:, :, None, :]], axis=2)
    return -(fx[:, :, :, 1:] - fx[:, :, :, :-1] + fy[:, :, 1:, :] - fy[:, :, :-1, :]) / (h * h)[:, :, None]


def _time_step(Q, h, cfl, inst, ninst):
    r, u, v, p, _ = _prims(Q)
    d = cfl * h / (np.sqrt(u * u + v * v) + np.sqrt(1.4 * p / r)).max(axis=(1, 2))
    out = np.full(ninst, np.inf)
    np.minimum.at(out, inst, d)
    return out


_LA = (0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
       -1275806237668 / 842570457699)
_LB = (1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
       3134564353537 / 4481467310338, 2277821191437 / 14882151754819)


def _advance(Q, scheme, dt, res):
    """one step; returns the new state and the last stage's residual"""
    if scheme == 1:
        k = res(Q)
        return Q + dt * k, k
    if scheme == 2:
        q1 = Q + dt * res(Q)
        k = res(q1)
        return 0.5 * (Q + q1 + dt * k), k
    if scheme == 3:
        q1 = Q + dt * res(Q)
        q2 = 0.75 * Q + 0.25 * (q1 + dt * res(q1))
        k = res(q2)
        return Q / 3 + 2.0 / 3 * (q2 + dt * k), k
    if scheme == 4:
        k1 = res(Q)
        k2 = res(Q + 0.5 * dt * k1)
        k3 = res(Q + 0.5 * dt * k2)
        k4 = res(Q + dt * k3)
        return Q + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4), k4
    d = 0.0
    for la, lb in zip(_LA, _LB):
        k = res(Q)
        d = la * d + dt * k
        Q = Q + lb * d
    return Q, k


def _exact_solver(case, seed):
    fs = _forests(case, seed)
    ci, fi, _, soln, inst = amrhip.batch_external(fs)
    n, nq = case["n"], inst.size
    h = _scale(case) * np.ldexp(1.0, -ci.reshape(-1, 3)[:, 1]) / n
    a, b = _face_table(nq, fi)
    Q = np.ascontiguousarray(np.moveaxis(soln.reshape(nq, n, n, 4), 3, 0))

    def res(q):
        return _residual(q, a, b, h, case["bc"])

    if case["kind"] == "rhs":
        return {"rhs": np.moveaxis(res(Q), 0, 3).reshape(-1), "dt": float(_time_step(Q, h, _cfl(case), inst, 1)[0])}
    t = np.zeros(case["inst"])
    for _ in range(_steps(case)):
        cap = np.full(case["inst"], _dt_cap(case))
        dt = cap if case["scheme"] == 2 else np.minimum(cap, _time_step(Q, h, _cfl(case), inst, case["inst"]))
        Q, k = _advance(Q, case["scheme"], dt[inst][:, None, None], res)
        t = t + dt
    if case["kind"] == "seam":
        return {"state": np.moveaxis(Q, 0, 3).reshape(-1), "t": float(t[0]), "flags": [None] * 5}
    return {"state": np.moveaxis(Q, 0, 1).reshape(-1), "t": t, "dt": dt, "norm": float(np.sqrt((k * k).sum()))}


def _exact_features(case, seed):
    fs = _forests(case, seed)
    _, fi, _, soln, inst = amrhip.batch_external(fs)
    n, nq = case["n"], inst.size
    a, b = _face_table(nq, fi)
    rho = soln.reshape(nq, n, n, 4)[..., 0]

    def jump(p, q):
        return np.abs(p - q) / (0.5 * (p + q))

    ind = np.maximum(jump(rho[:, :, 1:], rho[:, :, :-1]).max(axis=(1, 2)),
                     jump(rho[:, 1:], rho[:, :-1]).max(axis=(1, 2)))
    edge = [rho[:, :, 0], rho[:, :, -1], rho[:, 0], rho[:, -1]]
    for s in range(4):
        for other in (a, b):
            k = np.nonzero(other[:, s] >= 0)[0]
            ind[k] = np.maximum(ind[k], jump(edge[s][k], edge[s ^ 1][other[k, s]]).max(axis=1))
    return {"indicator": ind, "features": None, "classes": None, "tags": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "tag":
        return _exact_features(case, seed)
    if kind not in ("steps", "seam", "rhs"):
        return None       # a whole adaptive run, an epoch of Adam: every step follows from the one before
    evals = 1 if kind == "rhs" else STAGES[case["scheme"]] * _steps(case)
    if _quads(case) * case["n"] ** 2 * evals > 1.5e7:
        return None
    return _exact_solver(case, seed)
