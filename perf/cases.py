"""Workloads on which this library's speed is measured, and what they compute.

Every case is work a program has the library do through the `elasticapp_amd`
package: it builds a block of rods once, steps it, and reads the state back.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the block (or server) such a program holds
    run(state)           one pass: the steps, and the state read back
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    what the first pass returns, from a plain torch
                         restatement of the rod step in 64 bits

A case says how the rods are stepped (`path`): "fused" (the persistent
kernels, in chunks of 100 steps), "plain" (the op-by-op FP64 step), "calls"
(the stepper's per-block calls issued one by one, as a program that drives
its own stepper does) or "serve" (requests served from a pool of slots).
"""
import numpy as np
import torch

import elasticapp_amd as ea
from elasticapp_amd.workloads import UniformRods, stable_dt

CHUNK = 100  # steps per launch, and per captured graph, of the fused path

STATE = ("Position", "Velocity", "Director", "AngularVelocity")
# what a program reads beside the state after op-by-op steps
DERIVED = ("InternalLoads", "InternalTorques", "Curvature", "ShearStretchStrain")


# ---- cases -------------------------------------------------------------------


def _case(name, path, rods, n_min, n_max, steps, precision="fp64", hooks="none", tuned=False):
    c = dict(path=path, rods=rods, n_min=n_min, n_max=n_max, steps=steps, precision=precision, hooks=hooks, tuned=tuned)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one clamped cantilever with a tip force, a few steps between two looks
        # at it: an interactive or control loop, where latency is everything
        _case("cantilever_fp64", "fused", 1, 100, 100, 20, hooks="clamp"),
        # the same rod on the op-by-op path: the first thing a user who switches runs
        _case("cantilever_plain", "plain", 1, 100, 100, 20, hooks="clamp"),
        # a program that keeps its own stepper and issues the per-block calls
        _case("stepper_calls", "calls", 1024, 64, 64, 10, hooks="tip"),
        # op-by-op stepping of a ragged batch with odd lengths
        _case("ragged_plain", "plain", 1024, 16, 1024, 100, hooks="tip"),
        # the 1024 x 64 batch in double precision and in FP32-bulk
        _case("uniform_fp64", "fused", 1024, 64, 64, 500),
        _case("uniform_fp32", "fused", 1024, 64, 64, 2000, precision="fp32"),
        # a few short odd rods: a batch that fills a corner of the chip
        _case("few_odd_fp32", "fused", 61, 3, 301, 400, precision="fp32", hooks="tip"),
        # the ragged batch in double precision (the tuned plan cuts long rods)
        _case("ragged_fp64", "fused", 2048, 16, 1024, 300, hooks="tip", tuned=True),
        # the ragged batch in FP32-bulk, the largest one
        _case("ragged_fp32", "fused", 4096, 16, 1024, 3000, precision="fp32", hooks="tip", tuned=True),
        # rods lying on a plane under gravity, with contact and friction
        _case("plane_fp32", "fused", 8192, 128, 128, 2000, precision="fp32", hooks="plane", tuned=True),
        # rods longer than a tile
        _case("long_fp32", "fused", 24, 2500, 6000, 1000, precision="fp32", hooks="tip"),
        # a stream of requests of a few rods each, every result read and released
        _case("serve_fp32", "serve", 512, 32, 512, 1500, precision="fp32", hooks="tip"),
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["one", "plain", "calls", "fp64", "fp32", "fp32", "plane", "long", "serve"])
    if kind == "one":
        return _case("", rng.choice(["fused", "plain"]), 1, *([_log(rng, 20, 400)] * 2), _log(rng, 10, 100), hooks="clamp")
    if kind in ("plain", "calls"):
        lo = _log(rng, 2, 64)
        hi = _log(rng, lo, 1024)
        rods = max(1, min(_log(rng, 8, 2048), 260000 // hi))
        return _case("", kind, rods, lo, hi, _log(rng, 4, 60), hooks=rng.choice(["none", "tip", "plane", "tilt"]))
    if kind in ("fp64", "fp32"):
        lo = _log(rng, 3, 128)
        hi = _log(rng, lo, 1024)
        rods = max(1, min(_log(rng, 8, 4096), 500000 // hi))
        return _case("", "fused", rods, lo, hi, _log(rng, 40, 400 if kind == "fp64" else 1500), precision=kind,
                     hooks=rng.choice(["none", "tip", "tip", "tilt"]), tuned=rng.random() < 0.5)
    if kind == "plane":
        n = _log(rng, 24, 300)
        rods = max(1, min(_log(rng, 64, 8192), 500000 // n))
        precision = rng.choice(["fp32", "fp32", "fp64"])
        return _case("", "fused", rods, n, n, _log(rng, 60, 200 if precision == "fp64" else 1500), precision=precision,
                     hooks=rng.choice(["plane", "plane", "tilt"]))
    if kind == "long":
        lo = _log(rng, 1100, 3000)
        return _case("", "fused", _log(rng, 2, 32), lo, _log(rng, lo, 6000), _log(rng, 40, 600),
                     precision=rng.choice(["fp32", "fp64"]), hooks="tip")
    return _case("", "serve", _log(rng, 32, 512), 32, _log(rng, 64, 512), _log(rng, 200, 1500),
                 precision=rng.choice(["fp32", "fp32", "fp64"]), hooks="tip")


# ---- the rods of a case --------------------------------------------------------


def _lengths(case):
    """Element counts: log-uniform between the case's bounds, in a mixed order."""
    rods, lo, hi = case["rods"], case["n_min"], case["n_max"]
    n = np.exp(np.log(lo) + (np.log(hi) - np.log(lo)) * (np.arange(rods) + 0.5) / rods)
    n = np.clip(np.rint(n).astype(int), lo, hi)
    return [int(x) for x in np.random.default_rng(7).permutation(n)]


def _rods(case, seed):
    """Lengths, per-rod states, a stable dt per rod and tip forces."""
    rng = np.random.default_rng(int(seed))
    ns = _lengths(case)
    rods = len(ns)
    g = 1.0 / 1.99  # G / E
    if case["hooks"] in ("plane", "tilt"):
        # rods of 1 m lying just on the plane z = 0 along x, 5 cm apart
        L, r, rho, E, gam = np.full(rods, 1.0), np.full(rods, 0.01), np.full(rods, 1000.0), np.full(rods, 1e6), np.full(rods, 0.1)
        z = 0.01
    elif case["n_min"] == case["n_max"]:
        L, r, rho, E, gam = np.full(rods, 3.0), np.full(rods, 0.25), np.full(rods, 5000.0), np.full(rods, 1e6), np.full(rods, 0.1)
        z = 0.0
    else:
        L, r = rng.uniform(0.5, 3.0, rods), rng.uniform(0.005, 0.05, rods)
        E, rho = np.exp(rng.uniform(np.log(1e5), np.log(1e7), rods)), rng.uniform(500.0, 5000.0, rods)
        gam = rng.uniform(0.01, 0.5, rods)
        z = 0.0
    origin = lambda i: [0.0, 0.05 * i, z]  # noqa: E731
    make = lambda i: ea.straight_rod_state(ns[i], r[i], L[i], origin(i), [1.0, 0.0, 0.0], [0.0, 0.0, 1.0],  # noqa: E731
                                           rho[i], E[i], g * E[i], gam[i], gam[i])
    one = rods == 1
    if case["n_min"] == case["n_max"] and not one:
        n = ns[0]
        offsets = np.zeros((rods, 3))
        offsets[:, 1] = 0.05 * np.arange(rods)
        states = UniformRods(make(0), offsets, rng.normal(0.0, 0.5, (rods, 3, n - 1)))
        vel = rng.normal(0.0, 1e-2, (rods, 3, n + 1))
    else:
        states = [make(i) for i in range(rods)]
        vel = []
        for st in states:
            n = st["Director"].shape[1]
            if not one:
                st["ReferenceCurvature"] = rng.normal(0.0, 0.5, (3, n - 1))
            vel.append(rng.normal(0.0, 1e-2, (3, n + 1)))
    forces = rng.normal(0.0, 1.0, (rods, 3)) if not one else np.array([[0.0, -15.0, 0.0]]) * rng.uniform(0.5, 1.5)
    return ns, states, vel, stable_dt(L, np.array(ns), E, rho, r, g * E, gam), forces


GRAVITY = (0.0, 0.0, -9.81)
CONTACT = (1e3, 10.0, 0.3, 10.0, 0.0, 0.01)
TILT = (0.0, 0.6, 0.8)


def _build(case, seed):
    ns, states, vel, dt, forces = _rods(case, seed)
    blk = ea.DeviceBlock(ns)
    ea.assemble(blk, states)
    v = blk.get_field("Velocity")
    for s, a in zip(blk.starts, vel):
        v[:, s:s + a.shape[1]] = a
    blk.set_field("Velocity", v)
    if case["hooks"] == "clamp":
        st = states[0]
        blk.add_clamp(0, st["Position"][:, 0], st["Director"][:, 0])
    if case["hooks"] in ("clamp", "tip"):
        for i, f in enumerate(forces):
            blk.add_end_force(i, f)
    if case["hooks"] in ("plane", "tilt"):
        blk.set_gravity(GRAVITY)
        blk.set_plane_contact(*CONTACT, normal=TILT if case["hooks"] == "tilt" else None)
    blk.set_rod_dt(dt)
    return blk, dt


def _precision(case):
    return ea.FP64 if case["precision"] == "fp64" else ea.FP32_BULK


def _requests(case):
    """Requests of 1 to 16 library rods, with horizons up to the case's steps."""
    rng = np.random.default_rng(11)
    out = []
    left = max(16, case["rods"] // 2)
    while left > 0:
        k = int(rng.integers(1, 17))
        out.append((rng.integers(0, case["rods"], k), int(rng.integers(max(1, case["steps"] // 4), case["steps"] + 1))))
        left -= k
    return out


def prepare(case, seed):
    blk, dt = _build(case, seed)
    precision = _precision(case)
    state = {"case": case, "block": blk, "dt": float(np.min(dt)), "precision": precision}
    if case["path"] == "fused":
        blk.set_fused_config(0, 0, CHUNK)
        if case["tuned"]:
            blk.autotune(precision, CHUNK)
        if case["steps"] >= CHUNK:
            blk.capture_fused_graph(CHUNK, precision)
    elif case["path"] == "serve":
        caps = [c for c in (64, 128, 256, 512) if c < 2 * case["n_max"]]
        state["server"] = ea.Server(blk, [(c, case["rods"]) for c in caps], precision, CHUNK)
        state["requests"] = _requests(case)
        state["next"] = 0
    blk.synchronize()
    return state


# ---- one pass ---------------------------------------------------------------------


def _serve(state):
    srv, first = state["server"], state["next"]
    state["next"] += len(state["requests"])
    for i, (rods, steps) in enumerate(state["requests"]):
        srv.submit(first + i, rods, steps)
    got, left = {}, len(state["requests"])
    while left:
        for rid in srv.tick():
            rods = state["requests"][rid - first][0]
            got[rid - first] = [[srv.read(rid, j, tag) for j in range(len(rods))] for tag in ("Position", "Director")]
            srv.release(rid)
            left -= 1
    # results in the requests' order, a rod's lines one after another
    return {tag: np.concatenate([a.ravel() for i in range(len(got)) for a in got[i][t]])
            for t, tag in enumerate(("Position", "Director"))}


def run(state):
    case, blk = state["case"], state["block"]
    if case["path"] == "serve":
        return _serve(state)
    if case["path"] == "fused":
        if case["steps"] < CHUNK:
            blk.step_fused(case["steps"], state["precision"])
        else:
            blk.step_fused_graph(case["steps"], CHUNK, state["precision"])
        return {tag: blk.get_field(tag) for tag in STATE}
    dt = state["dt"]
    if case["path"] == "plain":
        blk.step(dt, case["steps"])
    else:
        t = 0.0
        for _ in range(case["steps"]):
            blk.kinematic_update(dt)
            t += 0.5 * dt
            blk.apply_post_kinematic(t)
            blk.compute_internal_dynamics(t)
            blk.apply_pre_dynamic(t)
            blk.dynamic_update(dt)
            blk.apply_post_dynamic(t)
            t += 0.5 * dt
            blk.kinematic_update(dt)
    return {tag: blk.get_field(tag) for tag in STATE + DERIVED}


# ---- what a pass cannot do without ---------------------------------------------------

# additions, multiplications, divisions and roots of one step of one element
# (with its node and Voronoi region), a sine, cosine or arc cosine counted as 20:
# two director updates 2 x 140, geometry and strain 45, forces and couples 60,
# curvature 85, torques 70, damping, accelerations and updates 60
FLOPS = 600.0


def work(case):
    ns = _lengths(case)
    if case["path"] == "serve":
        ns = [ns[int(r)] for rods, _ in _requests(case) for r in rods]
    elements = float(sum(ns))
    # x, v, Q, w read and written; m, 1/m, l0, sigma0, S, J, 1/J, D0, kappa0, B
    # read (in FP64, or in FP32)
    per = 2 * 18 * 8 + 22 * (8 if case["precision"] == "fp64" else 4)
    if case["path"] in ("plain", "calls"):
        per += 58 * 8  # the fields that derive from the state, written once
    steps = case["steps"] * (5.0 / 8.0 if case["path"] == "serve" else 1.0)
    return {"bytes": elements * per, "flops": elements * steps * FLOPS}


# ---- the same in plain torch, in 64 bits -----------------------------------------------


class _Exact:
    """The rod step over a ghost-padded block in torch.float64: rod i starts at
    slot s_i of the node, element and Voronoi lines, s_{i+1} = s_i + n_i + 2."""

    def __init__(self, case, rods, dev):
        ns, states, vel, dt, forces = rods
        self.case, self.ns = case, ns
        self.starts = np.concatenate([[0], np.cumsum(np.array(ns) + 2)[:-1]]).astype(np.int64)
        E = int(sum(ns) + 2 * len(ns) - 2)
        self.count = {"n": E + 1, "e": E, "v": E - 1}
        gn = self.starts[:-1] + np.array(ns[:-1], dtype=np.int64) + 1
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.ghost = {"n": t(gn), "e": t(np.concatenate([gn, gn - 1])), "v": t(np.concatenate([gn, gn - 1, gn - 2]))}

        def full(tag, kind, fill):
            nc = states[0][tag].shape[0]
            a = np.zeros((nc, self.count[kind]))
            for s, st in zip(self.starts, states):
                a[:, s:s + st[tag].shape[1]] = st[tag]
            a = t(a)
            a[:, self.ghost[kind]] = torch.as_tensor(fill, dtype=torch.float64, device=dev).reshape(-1, 1)
            return a

        self.x, self.v = full("Position", "n", 0.0), torch.zeros(3, E + 1, dtype=torch.float64, device=dev)
        v = np.zeros((3, E + 1))
        for s, a in zip(self.starts, vel):
            v[:, s:s + a.shape[1]] = a
        self.v = t(v)
        self.Q = full("Director", "e", [0.8, 0.6, 0.0, 0.0, 0.0, 1.0, 0.6, -0.8, 0.0]).reshape(3, 3, E)
        self.w = torch.zeros(3, E, dtype=torch.float64, device=dev)
        self.m, self.im = full("Mass", "n", 1.0)[0], full("InvMass", "n", 0.0)[0]
        self.l0 = full("ReferenceElementLength", "e", 1.0)[0]
        self.D0 = full("ReferenceVoronoiLength", "v", 1.0)[0]
        self.S, self.B = full("ShearStretchRigidityMatrix", "e", 0.0), full("BendingTwistRigidityMatrix", "v", 0.0)
        self.J, self.iJ = full("MassSecondMomentOfInertia", "e", 0.0), full("InvMassSecondMomentOfInertia", "e", 0.0)
        self.k0 = full("ReferenceCurvature", "v", 0.0)
        self.gf, self.gt = full("ForceDampingRate", "n", 0.0)[0], full("TorqueDampingRate", "e", 0.0)[0]
        self.is_rod = torch.ones(E + 1, dtype=torch.bool, device=dev)
        self.is_rod[self.ghost["n"]] = False
        self.forces = t(forces).T.contiguous() if case["hooks"] in ("clamp", "tip") else None
        self.tips = t(self.starts + np.array(ns))
        self.normal = t(np.array(TILT if case["hooks"] == "tilt" else (0.0, 0.0, 1.0))).reshape(3, 1)
        self.g = t(np.array(GRAVITY)).reshape(3, 1)
        if case["hooks"] == "clamp":
            self.x0, self.Q0 = self.x[:, 0].clone(), self.Q[:, :, 0].clone()
        # the rod of every slot (a ghost slot goes with the rod before it)
        owner = np.searchsorted(self.starts, np.arange(E + 1), side="right") - 1
        self.owner = t(owner.astype(np.int64))

    def lines(self, per_rod):
        a = per_rod[self.owner]
        return a, a[:-1]

    def kinematic(self, cn, ce):
        self.x = self.x + cn * self.v
        u = ce * self.w
        th = torch.sqrt((u * u).sum(0))
        u = u / (th + 1e-14)
        c, s = torch.cos(th), torch.sin(th)
        com = (self.Q * u[:, None]).sum(0)
        cr = torch.stack([self.Q[1] * u[2] - self.Q[2] * u[1], self.Q[2] * u[0] - self.Q[0] * u[2], self.Q[0] * u[1] - self.Q[1] * u[0]])
        self.Q = c * self.Q + (1.0 - c) * u[:, None] * com + s * cr

    @staticmethod
    def cross(a, b):
        return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])

    @staticmethod
    def diff(a):
        z = a.new_zeros(a.shape[0], 1)
        return torch.cat([a, z], 1) - torch.cat([z, a], 1)

    @staticmethod
    def quad(a):
        z = a.new_zeros(a.shape[0], 1)
        return 0.5 * (torch.cat([a, z], 1) + torch.cat([z, a], 1))

    def forces_and_torques(self):
        x, Q, l0 = self.x, self.Q, self.l0
        d = x[:, 1:] - x[:, :-1]
        l = torch.sqrt((d * d).sum(0))
        l[self.ghost["e"]] = 1.0
        t = d / l
        e = l / l0
        eps = 0.5 * (l[:-1] + l[1:]) / self.D0
        qt = (Q * t).sum(1)
        sigma = qt * e
        sigma[2] -= 1.0
        n = self.S * sigma
        c = (Q * n[:, None]).sum(0) / e
        c[:, self.ghost["e"]] = 0.0
        self.loads = self.diff(c) - self.m * self.gf * self.v
        a, b = Q[:, :, :-1], Q[:, :, 1:]
        th = torch.acos(0.5 * (a * b).sum((0, 1)) - (0.5 + 1e-10))
        f = 0.5 * th / torch.sin(th + 1e-14) / self.D0
        k = f * torch.stack([(a[2] * b[1] - a[1] * b[2]).sum(0), (a[0] * b[2] - a[2] * b[0]).sum(0), (a[1] * b[0] - a[0] * b[1]).sum(0)])
        k[:, self.ghost["v"]] = 0.0
        M = self.B * (k - self.k0)
        ic = 1.0 / (eps * eps * eps)
        jw = self.J * self.w / e
        rate = (t * (self.v[:, 1:] - self.v[:, :-1])).sum(0) / (e * l0)
        tau = self.diff(M * ic) + self.quad(self.cross(k, M) * (ic * self.D0)) + self.cross(qt, n) * l0
        tau = tau + self.cross(jw, self.w) + jw * rate - 0.5 * (self.m[:-1] + self.m[1:]) * self.gt * self.w
        self.torques, self.kappa, self.sigma, self.e = tau, k, sigma, e

    def external(self):
        fe = torch.zeros_like(self.v)
        if self.forces is not None:
            fe[:, self.tips] = self.forces
        if self.case["hooks"] in ("plane", "tilt"):
            k, c, mu, ct, z0, offset = CONTACT
            fe = fe + self.g * self.m
            gap = (self.normal * self.x).sum(0) - z0 - offset
            vn = (self.normal * self.v).sum(0)
            touch = (gap < 0.0) & self.is_rod
            fn = torch.where(touch, torch.clamp(-k * gap - c * vn, min=0.0), torch.zeros_like(gap))
            vt = self.v - vn * self.normal
            s = torch.sqrt((vt * vt).sum(0))
            ft = torch.minimum(ct * s, mu * fn)
            fe = fe + fn * self.normal - torch.where(touch & (s > 0.0), ft / torch.where(s > 0.0, s, torch.ones_like(s)), torch.zeros_like(s)) * vt
        return fe

    def step(self, dn, de):
        self.kinematic(0.5 * dn, 0.5 * de)
        if self.case["hooks"] == "clamp":
            self.x[:, 0], self.Q[:, :, 0] = self.x0, self.Q0
        self.forces_and_torques()
        self.v = self.v + dn * ((self.loads + self.external()) * self.im)
        self.w = self.w + de * (self.iJ * self.torques * self.e)
        if self.case["hooks"] == "clamp":
            self.v[:, 0] = 0.0
            self.w[:, 0] = 0.0
        self.kinematic(0.5 * dn, 0.5 * de)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["path"] == "serve":
        return _exact_serve(case, seed, dev)
    if sum(_lengths(case)) * case["steps"] > 4e9 or case["steps"] > 4000:
        return None  # over about 20 seconds
    rods = _rods(case, seed)
    with torch.no_grad():
        b = _Exact(case, rods, dev)
        dt = np.asarray(rods[3])
        if case["path"] != "fused":
            dt = np.full_like(dt, float(np.min(dt)))
        dn, de = b.lines(torch.as_tensor(dt, device=dev))
        for _ in range(case["steps"]):
            b.step(dn, de)
        E = b.count["e"]
        out = {"Position": b.x, "Velocity": b.v, "Director": b.Q.reshape(9, E), "AngularVelocity": b.w}
        if case["path"] != "fused":
            # (beyond a rod's ends the derived fields hold what the block-wide
            # operators leave there: nothing with an exact value)
            out |= {"InternalLoads": b.loads, "InternalTorques": None, "Curvature": b.kappa, "ShearStretchStrain": None}
        return {k: None if a is None else a.cpu().numpy() for k, a in out.items()}


def _exact_serve(case, seed, dev):
    requests = _requests(case)
    ns, states, vel, dt, forces = _rods(case, seed)
    which = np.concatenate([r for r, _ in requests]).astype(int)
    horizon = np.concatenate([np.full(len(r), s) for r, s in requests])
    rods = ([ns[i] for i in which], [states[i] for i in which], [vel[i] for i in which], dt[which], forces[which])
    if sum(rods[0]) * case["steps"] > 4e9 or case["steps"] > 4000:
        return None
    with torch.no_grad():
        b = _Exact(case, rods, dev)
        d, h = torch.as_tensor(rods[3], device=dev), torch.as_tensor(horizon, device=dev)
        for i in range(int(horizon.max())):
            # a rod past its horizon keeps its state (a step of dt = 0)
            b.step(*b.lines(torch.where(h > i, d, torch.zeros_like(d))))
        x, q = b.x.cpu().numpy(), b.Q.reshape(9, -1).cpu().numpy()
        return {"Position": np.concatenate([x[:, s:s + n + 1].ravel() for s, n in zip(b.starts, rods[0])]),
                "Director": np.concatenate([q[:, s:s + n].ravel() for s, n in zip(b.starts, rods[0])])}
