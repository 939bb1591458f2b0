"""Workloads of the particle pipeline as a user's program runs them.

Five kinds of work, all through the Python mirror of the C ABI
(flecsph_amd.BodySystem / BatchSystem):

run    a short job: upload initial data, run the initial iteration and
       `steps` driver iterations (fsph_step), fetch the snapshot by particle
       id and the conserved sums.  Periodic blasts, open tubes and boxes,
       self-gravitating stars, collapses with Newton-h or the learned h.
eval   one force evaluation on resident particles, for a program that keeps
       its own time loop over the finer entry points (tree and neighbours,
       density, acceleration, self-gravity, energy rate).
lists  the neighbour lists handed to a functor that runs on the host.
batch  a `run` of many uneven simulations in one batched context with graph
       replay.

A context in FP32 precision computes its pair sums, and with them
everything that evolves, to FP32; its outputs are returned as float32 (the
C ABI widens them to double), those of FP64 contexts as float64.
"""
import ctypes
import math

import numpy as np
import torch

from flecsph_amd import BatchSystem, BodySystem, _abi, generators

# ---- the cases -------------------------------------------------------------


def listed():
    return [
        # the smallest job in use: a test box of the smoke check's size
        # (latency of a step's launches and read-backs), FP64
        {"name": "box_2k_fp64", "kind": "run", "problem": "box", "n": 2000,
         "fp64": True, "steps": 20},
        # one force evaluation of a mid-sized FP64 box, variable smoothing
        # lengths, odd size: parity studies, callers with their own loop
        {"name": "eval_box_50k_fp64", "kind": "eval", "problem": "box",
         "n": 50021, "fp64": True},
        # the 3D Sod tube (38,880 particles, FP64, open boundaries)
        {"name": "sod_39k_fp64", "kind": "run", "problem": "sod", "n": 1,
         "fp64": True, "steps": 10},
        # neighbour lists of the Sod tube for a host functor
        {"name": "lists_sod_39k", "kind": "lists", "problem": "sod", "n": 1,
         "fp64": True},
        # the 64^3 Sedov blast in the periodic box (FP32, Wendland C6)
        {"name": "sedov_64", "kind": "run", "problem": "sedov", "n": 64,
         "fp64": False, "steps": 10},
        # the reference's default energy formulation (thermokinetic) with the
        # Cullen-Dehnen viscosity on a small odd-sided periodic blast
        {"name": "sedov_31_cullen", "kind": "run", "problem": "sedov",
         "n": 31, "fp64": False, "steps": 10, "thermokinetic": True,
         "cullen": True},
        # the reference's own FMM scheme (monopoles, single-particle leaves)
        # on a small star in FP64
        {"name": "star_10k_mono_fp64", "kind": "run", "problem": "star",
         "n": 10007, "fp64": True, "steps": 10, "fmm_order": 1, "leaf": 1},
        # one force evaluation with quadrupole FMM gravity, FP32, odd size
        {"name": "eval_star_200k", "kind": "eval", "problem": "star",
         "n": 200003, "fp64": False},
        # the self-gravitating polytrope of the headline benchmark, 1M
        {"name": "star_1m", "kind": "run", "problem": "star", "n": 1000000,
         "fp64": False, "steps": 8},
        # cold collapse, Newton smoothing lengths
        {"name": "collapse_1500k_newton", "kind": "run",
         "problem": "collapse", "n": 1500000, "fp64": False, "steps": 4,
         "h_mode": "newton"},
        # cold collapse, learned smoothing lengths (predictor trained before)
        {"name": "collapse_500k_learned", "kind": "run",
         "problem": "collapse", "n": 500000, "fp64": False, "steps": 6,
         "h_mode": "learned"},
        # 32 uneven Sedov blasts and Sod tubes in one context, graph replay
        {"name": "batch_32", "kind": "batch", "n_inst": 32, "lo": 8000,
         "hi": 100000, "sizes": 7, "steps": 6},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.15:
        return {"kind": "run", "problem": "box",
                "n": _log_int(rng, 2000, 150000) | 1,
                "fp64": rng.random() < 0.7, "steps": rng.randint(6, 12)}
    if pick < 0.25:
        return {"kind": "eval", "problem": "box",
                "n": _log_int(rng, 2000, 150000) | 1,
                "fp64": rng.random() < 0.7}
    if pick < 0.32:
        return {"kind": "run", "problem": "sod", "n": rng.randint(1, 2),
                "fp64": rng.random() < 0.5, "steps": rng.randint(4, 10)}
    if pick < 0.40:
        return {"kind": "lists", "problem": "box",
                "n": _log_int(rng, 2000, 60000) | 1,
                "fp64": rng.random() < 0.5}
    if pick < 0.55:
        return {"kind": "run", "problem": "sedov", "n": rng.randint(16, 80),
                "fp64": rng.random() < 0.2, "steps": rng.randint(4, 10),
                "thermokinetic": rng.random() < 0.5,
                "cullen": rng.random() < 0.3}
    if pick < 0.62:
        return {"kind": "run", "problem": "star",
                "n": _log_int(rng, 3000, 20000) | 1, "fp64": True,
                "steps": rng.randint(4, 10), "fmm_order": 1, "leaf": 1}
    if pick < 0.72:
        return {"kind": "eval", "problem": "star",
                "n": _log_int(rng, 5000, 250000) | 1,
                "fp64": rng.random() < 0.2}
    if pick < 0.82:
        return {"kind": "run", "problem": "star",
                "n": _log_int(rng, 5000, 1000000) | 1,
                "fp64": rng.random() < 0.1, "steps": rng.randint(3, 8)}
    if pick < 0.92:
        return {"kind": "run", "problem": "collapse",
                "n": _log_int(rng, 20000, 1000000), "fp64": False,
                "steps": rng.randint(3, 5),
                "h_mode": rng.choice(["newton", "learned"])}
    return {"kind": "batch", "n_inst": rng.randint(3, 40), "lo": 8000,
            "hi": 100000, "sizes": rng.randint(1, 1000),
            "steps": rng.randint(3, 6)}


# ---- inputs ----------------------------------------------------------------


def _jitter(parts, rng, amp):
    """Seeded noise on a lattice: positions by `amp` (an absolute length),
    internal energies by one part in a hundred, small random velocities."""
    n = len(parts["x"])
    for k in ("x", "y", "z"):
        parts[k] = parts[k] + amp * (2.0 * rng.random(n) - 1.0)
    parts["u"] = parts["u"] * (1.0 + 0.01 * (2.0 * rng.random(n) - 1.0))
    for k in ("vx", "vy", "vz"):
        parts[k] = 1e-2 * np.sqrt(np.minimum(parts["u"], 1.0)) * \
            rng.standard_normal(n)
    return parts


def _eta(n_ngb):
    return (3.0 * n_ngb / (4.0 * math.pi)) ** (1.0 / 3.0) / 2.0


def _box(n, rng):
    """n random points in the unit cube, smoothing lengths spread by 1.5
    around 40 neighbours, random velocities and energies (cubic spline)."""
    h0 = _eta(40) * 2.0 * (1.0 / n) ** (1.0 / 3.0)
    u = 1.0 + 0.5 * rng.random(n)
    parts = dict(x=rng.random(n), y=rng.random(n), z=rng.random(n),
                 vx=0.1 * rng.standard_normal(n),
                 vy=0.1 * rng.standard_normal(n),
                 vz=0.1 * rng.standard_normal(n), u=u,
                 h=h0 * (1.0 + 0.5 * rng.random(n)), m=np.full(n, 1.0 / n),
                 c=np.sqrt(1.4 * 0.4 * u))
    prm = dict(thermokinetic=0, kernel=_abi.KERNEL_CUBIC_SPLINE,
               eos=_abi.EOS_IDEAL, gamma=1.4, eta=_eta(40), adaptive_dt=1,
               initial_dt=1e-4, n_target=40)
    return parts, prm


def _fcc(n, rng):
    """The n innermost points of a jittered face-centred cubic lattice in the
    unit ball (no two closer than about half a spacing, as in
    generators.collapse: unsoftened gravity merges random close pairs)."""
    a = (4.0 * (4.0 * math.pi / 3.0) / n) ** (1.0 / 3.0)
    g = np.arange(-int(1.1 / a) - 1, int(1.1 / a) + 2) * a
    X, Y, Z = np.meshgrid(g, g, g, indexing="ij")
    corner = np.stack([X.ravel(), Y.ravel(), Z.ravel()], 1)
    corner = corner[(corner * corner).sum(1) < 1.3]
    basis = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]]) * a
    pts = (corner[:, None, :] + basis[None, :, :]).reshape(-1, 3)
    pts = pts + (rng.random(3) - 0.5) * a
    pts = pts + 0.15 * a / math.sqrt(2.0) * (2.0 * rng.random(pts.shape) - 1.0)
    r2 = (pts * pts).sum(1)
    return pts[np.argpartition(r2, n)[:n]]


def _star(n, rng, lattice):
    """The n=1 polytrope of generators.polytrope (R = M = G = K = 1): random
    points, or for runs over several steps a jittered lattice, stretched to
    the star's mass profile."""
    if lattice:
        pts = _fcc(n, rng)
        ru = np.linalg.norm(pts, axis=1)
        v = pts / np.maximum(ru, 1e-12)[:, None]
        q = (ru / (ru.max() * 1.001)) ** 3
    else:
        v = rng.standard_normal((n, 3))
        v /= np.linalg.norm(v, axis=1)[:, None]
        q = rng.random(n)
    grid = np.linspace(0.0, 1.0, 100001)
    mass = (np.sin(np.pi * grid) - np.pi * grid * np.cos(np.pi * grid)) / np.pi
    r = np.interp(q, mass, grid)
    pos = v * r[:, None]
    m = np.full(n, 1.0 / n)
    rho = np.sin(np.pi * r) / (4.0 * np.maximum(r, 1e-12))
    rho = np.maximum(rho, 0.05 * np.pi / 4.0)
    zero = np.zeros(n)
    parts = dict(x=pos[:, 0].copy(), y=pos[:, 1].copy(), z=pos[:, 2].copy(),
                 vx=zero, vy=zero, vz=zero, u=rho.copy(),
                 h=_eta(100) * 2.0 * (m / rho) ** (1.0 / 3.0), m=m, rho=rho,
                 P=rho ** 2, c=np.sqrt(2.0 * rho))
    prm = dict(thermokinetic=0, evolve_internal_energy=0,
               kernel=_abi.KERNEL_WENDLAND_C6, eos=_abi.EOS_POLYTROPIC,
               adaptive_dt=1, gamma=2.0, poly_K=1.0, eta=_eta(100),
               initial_dt=1e-4, gravity=_abi.GRAV_FMM, G=1.0, theta=0.5,
               leaf_size=32, n_target=100)
    return parts, prm


def _collapse(n, rng):
    """The cold collapse of generators.collapse with exactly n particles."""
    pos = _fcc(n, rng)
    m = np.full(n, (4.0 * math.pi / 3.0) / n)
    zero = np.zeros(n)
    gamma = 5.0 / 3.0
    parts = dict(x=pos[:, 0].copy(), y=pos[:, 1].copy(), z=pos[:, 2].copy(),
                 vx=zero, vy=zero, vz=zero, u=np.full(n, 0.05),
                 h=_eta(100) * 2.0 * m ** (1.0 / 3.0), m=m, rho=np.ones(n),
                 P=np.full(n, (gamma - 1.0) * 0.05),
                 c=np.full(n, math.sqrt(gamma * (gamma - 1.0) * 0.05)))
    prm = dict(thermokinetic=0, kernel=_abi.KERNEL_WENDLAND_C6,
               eos=_abi.EOS_IDEAL, adaptive_dt=1, gamma=gamma, eta=_eta(100),
               initial_dt=1e-4, gravity=_abi.GRAV_FMM, G=1.0, theta=0.5,
               leaf_size=32, n_target=100)
    return parts, prm


def _inputs(case, seed):
    rng = np.random.default_rng([seed, case["n"]])
    prob = case["problem"]
    if prob == "box":
        parts, prm = _box(case["n"], rng)
    elif prob == "star":
        parts, prm = _star(case["n"], rng, case["kind"] == "run")
    elif prob == "sod":
        parts, prm = generators.sod(scale=case["n"])
        parts = _jitter(parts, rng, 0.02 / (120 * case["n"]))
    elif prob == "sedov":
        parts, prm = generators.sedov(n_side=case["n"])
        if case.get("thermokinetic"):
            # u is recovered as e - v^2/2, which loses a cold background
            parts["u"] = parts["u"] + 0.05
        parts = _jitter(parts, rng, 0.05 / case["n"])
    else:
        parts, prm = _collapse(case["n"], rng)
    prm = dict(prm)
    prm["precision"] = _abi.PREC_FP64 if case["fp64"] else _abi.PREC_FP32
    if case.get("thermokinetic"):
        prm["thermokinetic"] = 1
    if case.get("cullen"):
        prm["viscosity"] = _abi.VISC_CULLEN
    if "fmm_order" in case:
        prm["fmm_order"] = case["fmm_order"]
        prm["leaf_size"] = case["leaf"]
    if case.get("h_mode") == "newton":
        prm["h_mode"] = _abi.H_NEWTON
    elif case.get("h_mode") == "learned":
        prm["h_mode"] = _abi.H_LEARNED
        prm["learn_steps"] = 4
    return parts, prm


def _batch_inputs(case, seed):
    """The mixed batch of blasts and tubes; which instances and how large is
    the case's (`sizes`), the noise on them the seed's."""
    sets, prm, periodic = generators.mixed_batch(
        case["n_inst"], case["lo"], case["hi"], seed=case["sizes"])
    rng = np.random.default_rng(seed)
    for i, parts in enumerate(sets):
        d = (1.0 if periodic[i] else 0.2) / np.cbrt(len(parts["x"]))
        sets[i] = _jitter(dict(parts), rng, 0.03 * d)
    return sets, prm, periodic


def _pinned(a):
    """The array in pinned host memory, as a loader would leave it."""
    t = torch.empty(len(a), dtype=torch.from_numpy(a[:1]).dtype,
                    pin_memory=True)
    t.numpy()[:] = a
    return t.numpy()


def _pin_all(parts):
    out = {k: _pinned(np.ascontiguousarray(v)) for k, v in parts.items()}
    out["id"] = np.arange(len(parts["x"]), dtype=np.int64)
    return out


# ---- one pass --------------------------------------------------------------


class _Snapshot:
    """Fetches fields of every particle into pinned host memory and hands
    them out on the GPU, ordered by particle id, without WALL copies."""

    def __init__(self, dtype):
        self.dtype = dtype
        self.buf = torch.empty(0)
        self.ids = torch.empty(0, dtype=torch.int64)

    def fetch(self, s, fields, offset=None):
        n, n_real = s.count()
        if self.buf.ndim < 2 or self.buf.shape[0] < len(fields) or \
                self.buf.shape[1] < n:
            self.buf = torch.empty(len(fields), n + n // 4,
                                   dtype=torch.float64, pin_memory=True)
        if len(self.ids) < n:
            self.ids = torch.empty(n + n // 4, dtype=torch.int64,
                                   pin_memory=True)
        for i, f in enumerate(fields):
            s._call("download", _abi.FIELD_INDEX[f],
                    ctypes.c_void_p(self.buf[i].data_ptr()))
        s._call("download", _abi.FIELD_INDEX["id"],
                ctypes.c_void_p(self.ids.data_ptr()))
        ids = self.ids[:n].cuda()
        real = None
        if offset is not None:  # batched: ids count within an instance
            first, count = offset
            real = ids < count
            ids = ids + first
        elif n > n_real:
            real = ids < n_real
        out = {}
        for i, f in enumerate(fields):
            v = self.buf[i, :n].cuda()
            v = v.to(torch.int32 if f == "nngb" else self.dtype)
            o = torch.empty(n_real, dtype=v.dtype, device=v.device)
            if real is None:
                o[ids] = v
            else:
                o[ids[real]] = v[real]
            out[f] = o
        return out


def prepare(case, seed):
    dtype = torch.float64 if case.get("fp64") else torch.float32
    st = {"case": case, "snap": _Snapshot(dtype), "dtype": dtype}
    if case["kind"] == "batch":
        sets, prm, periodic = _batch_inputs(case, seed)
        s = BatchSystem(_abi.default_params(**prm), case["n_inst"])
        st["parts"] = [_pin_all(p) for p in sets]
        for i, p in enumerate(periodic):
            s.instance_set_periodic(i, p)
        s.enable_graph(True)
        s.upload(st["parts"])
    else:
        parts, prm = _inputs(case, seed)
        s = BodySystem(_abi.default_params(**prm))
        st["parts"] = _pin_all(parts)
        s.upload(st["parts"])
        if case.get("h_mode") == "learned":
            # train the predictor on the first steps of this collapse
            for _ in range(7):
                s.step()
    if case["kind"] == "lists":
        # the functor program's list buffers, unused entries -1
        n = len(parts["x"])
        st["off"] = np.zeros(n + 1, np.int64)
        st["idx"] = np.full(3 * prm["n_target"] * n, -1, np.int64)
    st["sys"] = s
    return st


def _run_job(st):
    case, s = st["case"], st["sys"]
    s.upload(st["parts"])
    for _ in range(case["steps"] + 1):
        s.step()
    fields = ["x", "y", "z", "vx", "vy", "vz", "h", "rho"]
    if case["problem"] in ("sod", "sedov", "box"):
        fields.append("u")
    if case["problem"] in ("star", "collapse"):
        fields.append("phi")
    out = st["snap"].fetch(s, fields)
    out["sums"] = torch.from_numpy(s.reductions()).to(st["dtype"])
    out["time"] = torch.tensor(s.time()[1:]).to(st["dtype"])
    return out


def _run_eval(st):
    s = st["sys"]
    s.update_iteration()
    s.density_eos()
    out = st["snap"].fetch(s, ["rho", "P", "c", "vsig", "nngb"])
    s.acceleration()
    rates = ["ax", "ay", "az"]
    if st["case"]["problem"] == "star":
        s.gravity()
        rates += ["gx", "gy", "gz", "phi"]
    else:
        s.dudt()
        rates.append("dudt")
    out.update(st["snap"].fetch(s, rates))
    return out


def _run_lists(st):
    s = st["sys"]
    s.update_iteration()
    pi64 = ctypes.POINTER(ctypes.c_int64)
    s._call("neighbor_lists", st["off"].ctypes.data_as(pi64),
            st["idx"].ctypes.data_as(pi64), len(st["idx"]))
    return {"id": s.get("id"), "off": st["off"], "idx": st["idx"]}


def _run_batch(st):
    case, s = st["case"], st["sys"]
    s.upload(st["parts"])
    for _ in range(case["steps"] + 1):
        s.step()
    tot, real = zip(*(s.instance_count(i) for i in range(s.n_inst)))
    tot, real = torch.tensor(tot), torch.tensor(real)
    first = torch.cumsum(real, 0) - real
    offset = (torch.repeat_interleave(first, tot).cuda(),
              torch.repeat_interleave(real, tot).cuda())
    out = st["snap"].fetch(
        s, ["x", "y", "z", "vx", "vy", "vz", "h", "rho", "u"], offset)
    out["time"] = torch.tensor(
        [s.instance_time(i)[1:] for i in range(s.n_inst)]).to(st["dtype"])
    return out


def run(state):
    return {"run": _run_job, "eval": _run_eval, "lists": _run_lists,
            "batch": _run_batch}[state["case"]["kind"]](state)


# ---- work ------------------------------------------------------------------


def _count(case):
    if case["kind"] == "batch":
        return sum(len(p["x"]) for p in generators.mixed_batch(
            case["n_inst"], case["lo"], case["hi"], seed=case["sizes"])[0])
    return {"sod": 38880 * case["n"] ** 3, "sedov": case["n"] ** 3}.get(
        case["problem"], case["n"])


def work(case):
    """Per particle and step: the state read and written once by each pass
    (864 bytes, 968 with gravity), about 130 flops per neighbour pair (density
    25, acceleration 60, energy rate 45) and, with gravity, about 2,050 direct
    interactions of 20 flops and 44 M2L of 150 (opening angle 0.5, leaves of
    32; some 250 interactions per particle in the monopole scheme)."""
    n = _count(case)
    prob = case.get("problem", "sedov")
    ngb = {"box": 40, "sod": 60}.get(prob, 100)
    grav = prob in ("star", "collapse")
    g_flops = 0
    if grav:
        g_flops = 250 * 20 if case.get("leaf") == 1 else 2050 * 20 + 44 * 150
    if case["kind"] == "lists":
        return {"bytes": n * (4 * 8.0 + 16 + 8.0 * ngb), "flops": n * ngb * 9.0}
    if case["kind"] == "eval":
        return {"bytes": n * (9 * 8.0 + 12 * 8.0),
                "flops": n * (ngb * (130.0 if not grav else 85.0) + g_flops)}
    steps = case["steps"] + 1
    return {"bytes": n * (steps * (968.0 if grav else 864.0) + 13 * 8 + 9 * 8),
            "flops": n * steps * (ngb * 130.0 + g_flops)}


# ---- exact values ----------------------------------------------------------


def exact(case, seed):
    """Force evaluations as direct sums in FP64 (the other cases: None).
    The signal speed and the neighbour counts follow the tree's lists, which
    hold pairs outside the kernel's support, and have no value here."""
    if case["kind"] != "eval" or case["n"] > 260000:
        return None
    parts, prm = _inputs(case, seed)
    d = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda()
         for k, v in parts.items()}
    n = len(d["x"])
    pos = torch.stack([d["x"], d["y"], d["z"]])
    vel = torch.stack([d["vx"], d["vy"], d["vz"]])
    h, m = d["h"], d["m"]
    hmax = float(h.max())
    star = case["problem"] == "star"
    rows = max(1, int(1.5e8 // n))
    ia, ib = [], []
    gx = torch.zeros(3, n, dtype=torch.float64, device="cuda")
    phi = torch.zeros(n, dtype=torch.float64, device="cuda")
    for a in range(0, n, rows):
        e = min(n, a + rows)
        r2 = torch.zeros(e - a, n, dtype=torch.float64, device="cuda")
        for k in range(3):
            r2 += (pos[k, a:e, None] - pos[k][None, :]) ** 2
        near = torch.nonzero(r2 < hmax * hmax)
        ia.append(near[:, 0] + a)
        ib.append(near[:, 1])
        if star:
            ir = torch.rsqrt(r2)
            ir[torch.arange(e - a), torch.arange(a, e)] = 0.0
            phi[a:e] = -(ir * m[None, :]).sum(1)
            w = ir ** 3 * m[None, :]
            for k in range(3):
                gx[k, a:e] = w @ pos[k] - w.sum(1) * pos[k, a:e]
    ia, ib = torch.cat(ia), torch.cat(ib)

    def summed(v):
        return torch.zeros(n, dtype=torch.float64,
                           device="cuda").index_add_(0, ia, v)

    dx = pos[:, ia] - pos[:, ib]
    r = (dx * dx).sum(0).sqrt()
    hab = 0.5 * (h[ia] + h[ib])
    q = r / hab
    rp = torch.where(r > 0, r, torch.ones_like(r))
    if prm["kernel"] == _abi.KERNEL_CUBIC_SPLINE:
        s = 2.0 * q
        t = torch.clamp(2.0 - s, min=0.0)
        sig = 8.0 / math.pi / hab ** 3
        W = sig * torch.where(s < 1, 1 - 1.5 * s ** 2 + 0.75 * s ** 3,
                              0.25 * t ** 3)
        dW = 2.0 * sig / hab * torch.where(s < 1, -3 * s + 2.25 * s ** 2,
                                           -0.75 * t ** 2)
    else:
        t = torch.clamp(1.0 - q, min=0.0)
        sig = 1365.0 / (64.0 * math.pi) / hab ** 3
        W = sig * t ** 8 * (1 + 8 * q + 25 * q ** 2 + 32 * q ** 3)
        dW = sig / hab * -22.0 * q * t ** 7 * (1 + 7 * q + 16 * q ** 2)
    rho = summed(m[ib] * W)
    gamma = prm["gamma"]
    if prm["eos"] == _abi.EOS_POLYTROPIC:
        P = prm["poly_K"] * rho ** gamma
        c = torch.sqrt(prm["poly_K"] * gamma * rho ** (gamma - 1.0))
    else:
        P = (gamma - 1.0) * rho * d["u"]
        c = torch.sqrt(gamma * (gamma - 1.0) * d["u"])
    vr = ((vel[:, ia] - vel[:, ib]) * dx).sum(0)
    mu = torch.where(vr < 0, hab * vr / (r * r + 0.01 * hab * hab),
                     torch.zeros_like(vr))
    cab, rab = 0.5 * (c[ia] + c[ib]), 0.5 * (rho[ia] + rho[ib])
    Pi = (-1.0 * cab + 2.0 * mu) * mu / rab
    F = torch.where(r > 0, dW / rp, torch.zeros_like(r))
    pr = P / rho ** 2
    f = -m[ib] * (pr[ia] + pr[ib] + Pi) * F
    out = {"rho": rho, "P": P, "c": c, "vsig": None, "nngb": None}
    for k, name in enumerate(("ax", "ay", "az")):
        out[name] = summed(f * dx[k])
    if star:
        for k, name in enumerate(("gx", "gy", "gz")):
            out[name] = gx[k]
        out["phi"] = phi
    else:
        out["dudt"] = summed(m[ib] * (pr[ia] + 0.5 * Pi) * vr * F)
    return out
