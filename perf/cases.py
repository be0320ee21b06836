"""The work a user of this framework has it do, as cases that can be timed.

Seven ways into the cycle, each over the range of sizes it is used at:

  step    one lagrangeLeapFrog on fields the caller holds in device memory
          (lulesh_lagrange_leapfrog_noalloc), as a function of a state: the
          state is copied into the working fields, then stepped.  Serving
          loops and programs that own their arrays; launches and latency count.
  loop    the reference's while-loop stepped from the host, timeIncrement and
          lagrangeLeapFrog per cycle, with every field kept (keep_aux).
  run     the driver loop on the device from the initial state for a number of
          cycles, then the fields the simulation was run for.
  batch   many independent uneven domains in one driver loop (c5_instances).
  enzyme  the reference's loop under reverse mode: timeIncrement, then the
          cycle with the shadow mapped through it (vjp_cycle).
  grad    a gradient over many cycles, checkpointed every `every` cycles.
  revolve the same in bounded memory, with `snapshots` saved states.

Every domain is a Sedov problem whose deposited energy and hourglass
coefficient come from the seed.  exact() restates the cycle in plain torch,
64 bits, with torch's own autograd for the gradients.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "lulesh.jl_amd"))
import lulesh_amd as L  # noqa: E402
from lulesh_amd import _lib  # noqa: E402

NODE_STATE = ("x", "y", "z", "xd", "yd", "zd")
ELEM_STATE = ("e", "p", "q", "v", "ss")
STATE = NODE_STATE + ELEM_STATE
AUX = ("fx", "fy", "fz", "xdd", "ydd", "zdd", "dxx", "dyy", "dzz", "ql", "qq")
STEP_ELEM = ("e", "p", "q", "v", "ss", "delv", "vdov", "arealg")
WARM = 24  # cycles a step's starting state is into its simulation


def listed():
    return [
        # a small caller-held domain stepped inside another program's loop
        {"name": "step_12", "kind": "step", "s": 12, "quirks": 7},
        # the largest domain that entry point takes, the corrected arithmetic
        {"name": "step_68", "kind": "step", "s": 68, "quirks": 0},
        # the reference's smoke configuration (s=8, 10 iterations), host-stepped
        {"name": "loop_8", "kind": "loop", "s": 8, "cycles": 10, "quirks": 7},
        # small domains on the device loop: a cycle is four short launches
        {"name": "run_16", "kind": "run", "s": 16, "cycles": 100, "quirks": 7},
        # the size LULESH is quoted at by default
        {"name": "run_30", "kind": "run", "s": 30, "cycles": 200, "quirks": 7},
        # an odd size, mid range, the corrected arithmetic
        {"name": "run_63", "kind": "run", "s": 63, "cycles": 200, "quirks": 0},
        # a domain that about fills the chip
        {"name": "run_96", "kind": "run", "s": 96, "cycles": 200, "quirks": 7},
        # the headline benchmark: s=192, the first 500 cycles
        {"name": "run_192", "kind": "run", "s": 192, "cycles": 500, "quirks": 7},
        # the ragged batch: 64 domains of 16..64 elements per edge
        {"name": "batch_64", "kind": "batch", "n": 64, "cycles": 300, "quirks": 7},
        # the reference's differentiated loop on a small domain
        {"name": "enzyme_24", "kind": "enzyme", "s": 24, "cycles": 8, "quirks": 7},
        # the gradient benchmark: s=48, 200 cycles, a checkpoint every 20
        {"name": "grad_48", "kind": "grad", "s": 48, "cycles": 200, "every": 20, "quirks": 7},
        # a gradient in bounded memory
        {"name": "revolve_30", "kind": "revolve", "s": 30, "cycles": 60, "snapshots": 8,
         "quirks": 7},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "loop", "run", "run", "run", "batch", "enzyme", "grad", "revolve"))
    c = {"kind": kind, "quirks": rng.choice((7, 7, 0))}
    if kind == "step":
        c["s"] = _log_int(rng, 8, 68)
    elif kind == "loop":
        c.update(s=_log_int(rng, 8, 96), cycles=rng.randint(6, 20))
    elif kind == "run":
        s = _log_int(rng, 10, 192)
        c.update(s=s, cycles=rng.randint(40, 80 if s < 20 else 220))
    elif kind == "batch":
        c.update(n=_log_int(rng, 3, 64), cycles=rng.randint(80, 300))
    elif kind == "enzyme":
        c.update(s=_log_int(rng, 8, 64), cycles=rng.randint(4, 10))
    elif kind == "grad":
        c.update(s=_log_int(rng, 12, 64), cycles=rng.randint(30, 120), every=rng.randint(5, 40))
    else:
        c.update(s=_log_int(rng, 12, 48), cycles=rng.randint(20, 80), snapshots=rng.randint(3, 12))
    return c


def _problem(seed):
    """Deposited energy (times the reference's) and hourglass coefficient."""
    r = random.Random(1000003 * int(seed) + 17)
    return math.exp(r.uniform(math.log(0.5), math.log(2.0))), r.uniform(2.0, 4.0)


def _batch_problem(case, seed):
    """Sizes as c5_instances draws them for the case, energies and hourglass
    coefficients from the seed."""
    nx = L.c5_instances(case["n"])[0]
    r = random.Random(1000003 * int(seed) + 29)
    scale = [math.exp(r.uniform(math.log(0.5), math.log(2.0))) for _ in nx]
    return nx, scale, [r.uniform(2.0, 4.0) for _ in nx]


def _shadow(case, seed):
    """The adjoint the loop starts from, at random."""
    s = case["s"]
    g = np.random.default_rng([int(seed), s, 5])
    n = {f: (s + 1) ** 3 if f in NODE_STATE else s ** 3 for f in STATE}
    return {f: g.standard_normal(n[f]) for f in STATE}


# -- the framework's side -----------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        nx, scale, hg = _batch_problem(case, seed)
        b = L.Batch(nx, scale, hg, quirks=case["quirks"])
        return case, b, None
    scale, hg = _problem(seed)
    b = L.Batch([case["s"]], [scale], [hg], quirks=case["quirks"])
    d = b.instance(0)
    if kind == "step":
        L.run(d, WARM)
        L.timeIncrement(d)
        return case, None, _StepState(case, d, b)
    if kind == "loop":
        d.keep_aux(True)
    return case, b, _shadow(case, seed) if kind == "enzyme" else None


class _StepState:
    """A caller's own device arrays: the state to step from, the working
    fields the step is made in, and the scalars."""

    def __init__(self, case, d, b):
        cuda = {"device": "cuda"}
        fields = {f: torch.from_numpy(d.get(f)).to(**cuda)
                  for f in STATE + ("delv", "vdov", "arealg", "volo", "elemMass", "nodalMass")}
        bc = torch.from_numpy(d.get("elemBC").view(np.int32)).to(**cuda)
        self.start = [fields[f] for f in STATE]
        self.out = {f: fields[f].clone() for f in NODE_STATE + STEP_ELEM}
        self.work = [self.out[f] for f in STATE]
        self.keep = (fields, bc)
        self.scalars = np.array([float(d.get(n)) for n in L.SCALARS])
        dom = _lib.DeviceDomain()
        dom.nx, dom.quirks = case["s"], case["quirks"]
        for f in ("e", "p", "q", "v", "ss", "delv", "vdov", "arealg") + NODE_STATE:
            setattr(dom, f, ctypes.cast(self.out[f].data_ptr(), _lib.P_double))
        for f in ("volo", "elemMass", "nodalMass"):
            setattr(dom, f, ctypes.cast(fields[f].data_ptr(), _lib.P_double))
        dom.elemBC = ctypes.cast(bc.data_ptr(), _lib.P_uint32)
        self.dom = dom
        self.lib = _lib.load()
        b.close()


def run(state):
    case, b, extra = state
    return _RUN[case["kind"]](case, b, extra)


def _run_step(case, b, st):
    torch._foreach_copy_(st.work, st.start)
    sc = st.scalars.copy()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = st.lib.lulesh_lagrange_leapfrog_noalloc(ctypes.byref(st.dom),
                                                 sc.ctypes.data_as(_lib.P_double), stream, 0)
    if rc:
        raise L.LuleshError(rc, st.lib.lulesh_error_string(rc).decode())
    return {**st.out, "dtcourant": float(sc[3]), "dthydro": float(sc[4])}


def _run_loop(case, b, _):
    d = b.instance(0)
    d.reset()
    while d.time < d.stoptime:
        L.timeIncrement(d)
        L.lagrangeLeapFrog(d)
        if d.cycle >= case["cycles"]:
            break
    return {f: d.get(f) for f in STATE + AUX + ("time",)}


def _run_run(case, b, _):
    d = b.instance(0)
    d.reset()
    L.run(d, case["cycles"])
    return {f: d.get(f) for f in STATE + ("time",)}


def _run_batch(case, b, _):
    b.instance(0).reset()
    b.run(case["cycles"])
    return {f: np.concatenate([v.get(f) for v in b.views]) for f in STATE}


def _run_enzyme(case, b, shadow):
    d = b.instance(0)
    d.reset()
    params = np.zeros(3)
    sh = shadow
    for _ in range(case["cycles"]):
        L.timeIncrement(d)
        out, _ = L.vjp_cycle(d, sh, params)
        sh = None  # the shadow stays on the device between cycles
    return {**out, "params": params, "end_e": d.e, "end_x": d.x}


def _run_grad(case, b, _):
    d = b.instance(0)
    d.reset()
    return L.grad_run(d, case["cycles"], case["every"])


def _run_revolve(case, b, _):
    d = b.instance(0)
    d.reset()
    return L.grad_run_revolve(d, case["cycles"], case["snapshots"])


_RUN = {"step": _run_step, "loop": _run_loop, "run": _run_run, "batch": _run_batch,
        "enzyme": _run_enzyme, "grad": _run_grad, "revolve": _run_revolve}


# -- what a pass cannot do without --------------------------------------------
def work(case):
    """Bytes: per cycle the node state and mass (13 doubles) and the element
    state, volume and mass (12 doubles) once, and the three kinematic fields
    the cycle leaves; once per pass what the caller gets back.  A reversed
    cycle reads the state again and moves the adjoint state.  Operations:
    the cycle's additions, products, divisions and roots, about 2000 per
    element and 20 per node; twice that for the adjoint of a cycle."""
    kind = case["kind"]
    sizes = L.c5_instances(case["n"])[0] if kind == "batch" else [case["s"]]
    E = float(sum(s ** 3 for s in sizes))
    N = float(sum((s + 1) ** 3 for s in sizes))
    cyc = case.get("cycles", 1)
    cycle_bytes, cycle_flops = 104 * N + 120 * E, 2000 * E + 20 * N
    state = 8 * (6 * N + 5 * E)
    if kind == "step":
        return {"bytes": cycle_bytes, "flops": cycle_flops}
    if kind in ("loop", "run", "batch"):
        out = state + (8 * (6 * N + 5 * E) if kind == "loop" else 0)
        return {"bytes": cyc * cycle_bytes + out, "flops": cyc * cycle_flops}
    back_bytes = 2 * state + state
    if kind == "enzyme":
        return {"bytes": cyc * (cycle_bytes + back_bytes + state), "flops": cyc * 3 * cycle_flops}
    # the recomputation a schedule costs is its own affair: forward once, back once
    return {"bytes": cyc * (cycle_bytes + back_bytes) + 8 * E, "flops": cyc * 3 * cycle_flops}


# -- the cycle in plain torch, 64 bits ----------------------------------------
def exact(case, seed):
    if case["kind"] == "batch":
        nx, scale, hg = _batch_problem(case, seed)
        if sum(case["cycles"] for _ in nx) * 0.014 > 20.0:
            return None
        ends = []
        for s, sc, h in zip(nx, scale, hg):
            sim = _Sim(s, case["quirks"], sc, h)
            while sim.time < sim.stoptime and sim.cycle < case["cycles"]:
                sim.advance()
            ends.append(sim)
        return {f: np.concatenate([_flat(x.st[f]) for x in ends]) for f in STATE}
    s, cyc = case["s"], case.get("cycles", WARM + 1)
    if cyc * (0.014 + s ** 3 * 1.0e-8) * (4 if case["kind"] in ("enzyme", "grad", "revolve") else 1) > 20.0:
        return None
    sim = _Sim(s, case["quirks"], *_problem(seed))
    kind = case["kind"]
    if kind == "step":
        for _ in range(WARM + 1):
            sim.advance()
        got = {f: _flat(sim.st[f]) for f in STATE}
        got.update({f: _flat(sim.aux[f]) for f in ("delv", "vdov", "arealg")})
        return {**got, "dtcourant": sim.dtcourant, "dthydro": sim.dthydro}
    if kind in ("loop", "run"):
        while sim.time < sim.stoptime and sim.cycle < cyc:
            sim.advance()
        got = {f: _flat(sim.st[f]) for f in STATE}
        if kind == "loop":
            got.update({f: _flat(sim.aux[f]) for f in AUX})
        return {**got, "time": sim.time}
    if kind == "enzyme":
        sh = {f: sim.tensor(f, a) for f, a in _shadow(case, seed).items()}
        params = np.zeros(3)
        for _ in range(cyc):
            before = sim.st
            sim.advance()
            sh, gp = sim.pull_back(before, sim.dt, sh)
            params += gp
        return {**{f: _flat(sh[f]) for f in STATE}, "params": params, "end_e": _flat(sim.st["e"]),
                "end_x": _flat(sim.st["x"])}
    states, dts = [], []
    for _ in range(cyc):
        states.append(sim.st)
        sim.advance()
        dts.append(sim.dt)
    loss = float((sim.st["e"] * sim.elemMass).sum())
    sh = {f: torch.zeros_like(sim.st[f]) for f in STATE}
    sh["e"] = sim.elemMass.clone()
    params = np.zeros(3)
    for st, dt in zip(reversed(states), reversed(dts)):
        sh, gp = sim.pull_back(st, dt, sh)
        params += gp
    got = {"loss": loss, "grad_e": _flat(sh["e"]), "grad_hgcoef": params[0],
           "grad_qlc_monoq": params[1], "grad_qqc_monoq": params[2], "dt": np.array(dts)}
    if kind == "revolve":
        got["forward_cycles"] = None
    return got


def _flat(t):
    return t.detach().reshape(-1).cpu().numpy()


def _cbrt(x):
    y = x ** (1.0 / 3.0)
    return y - (y * y * y - x) / (3.0 * (y * y))


_GAMMA = ((1, 1, 1, -1), (1, -1, -1, 1), (-1, -1, 1, -1), (-1, 1, -1, 1),
          (-1, -1, 1, 1), (-1, 1, -1, -1), (1, 1, 1, 1), (1, -1, -1, -1))
# where an element's corner n sits among the nodes: (plane, row, column) offsets
_CORNER = ((0, 0, 0), (0, 0, 1), (0, 1, 1), (0, 1, 0), (1, 0, 0), (1, 0, 1), (1, 1, 1), (1, 1, 0))
_FACES = ((0, 1, 2, 3), (0, 4, 5, 1), (1, 5, 6, 2), (2, 6, 7, 3), (3, 7, 4, 0), (4, 7, 6, 5))


def _at(n, s):
    return tuple(slice(o, o + s) for o in _CORNER[n])


def _add(a):
    out = a[0]
    for t in a[1:]:
        out = out + t
    return out


def _dot(a, b):
    return _add([x * y for x, y in zip(a, b)])


def _volume(x, y, z):
    def d(a, b):
        return [c[a] - c[b] for c in (x, y, z)]

    def triple(a, b, c):
        (x1, y1, z1), (x2, y2, z2), (x3, y3, z3) = a, b, c
        return (x1 * (y2 * z3 - z2 * y3) + x2 * (z1 * y3 - y1 * z3)) + x3 * (y1 * z2 - z1 * y2)

    def plus(a, b):
        return [u + v for u, v in zip(a, b)]

    return ((triple(plus(d(3, 1), d(7, 2)), d(6, 3), d(2, 0))
             + triple(plus(d(4, 3), d(5, 7)), d(6, 4), d(7, 0)))
            + triple(plus(d(1, 4), d(2, 5)), d(6, 1), d(5, 0))) * (1.0 / 12.0)


def _jacobian(c):
    out = []
    for a in c:
        d60, d53, d71, d42 = a[6] - a[0], a[5] - a[3], a[7] - a[1], a[4] - a[2]
        out.append((0.125 * (d60 + d53 - d71 - d42), 0.125 * (d60 - d53 + d71 - d42),
                    0.125 * (d60 + d53 + d71 + d42)))
    return out


def _vol_derivative(x, y, z, quirks):
    slots = [(1, 2, 3, 4, 5, 7), (0, 1, 2, 7, 4, 6), (3, 0, 1, 6, 7, 5), (2, 3, 0, 5, 6, 4),
             (7, 6, 5, 0, 3, 1), (4, 7, 6, 1, 0, 2), (5, 4, 7, 2, 1, 3), (6, 5, 4, 3, 2, 0)]
    if not quirks & 2:
        slots[1], slots[3] = slots[3], slots[1]

    def one(u, w, i):
        u, w = [u[k] for k in i], [w[k] for k in i]
        return ((u[1] + u[2]) * (w[0] + w[1]) - (u[0] + u[1]) * (w[1] + w[2])
                + (u[0] + u[4]) * (w[3] + w[4]) - (u[3] + u[4]) * (w[0] + w[4])
                - (u[2] + u[5]) * (w[3] + w[5]) + (u[3] + u[5]) * (w[2] + w[5])) * (1.0 / 12.0)

    # d/dx from (y, z), d/dy from (z, x), d/dz from (x, y), cyclically
    return [[one(u, w, i) for i in slots] for u, w in ((y, z), (z, x), (x, y))]


class _Sim:
    """A Sedov domain: its state as grids (plane, row, column), its scalars."""

    def __init__(self, s, quirks, scale, hgcoef):
        self.s, self.quirks = s, quirks
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        kw = {"dtype": torch.float64, "device": self.dev}
        ax = 1.125 * torch.arange(s + 1, **kw) / s
        one = torch.ones((s + 1,) * 3, **kw)
        st = {"x": one * ax[None, None, :], "y": one * ax[None, :, None], "z": one * ax[:, None, None]}
        for f in ("xd", "yd", "zd"):
            st[f] = torch.zeros_like(one)
        for f in ELEM_STATE:
            st[f] = torch.zeros((s,) * 3, **kw)
        st["v"] = torch.ones_like(st["v"])
        self.volo = _volume(*self.corners(st, "xyz"))
        self.elemMass = self.volo.clone()
        self.nodalMass = self.gather([self.volo / 8.0] * 8)
        e0 = 3.948746e+7 * (s / 45.0) * (s / 45.0) * (s / 45.0) * scale
        st["e"][0, 0, 0] = e0
        self.st = st
        self.hgcoef, self.qlc, self.qqc = hgcoef, 0.5, 2.0 / 3.0
        self.dt = 0.5 * float(_cbrt(self.volo[0, 0, 0])) / math.sqrt(2.0 * e0)
        self.time, self.stoptime, self.dtmax, self.cycle = 0.0, 1.0e-2, 1.0e-2, 0
        self.dtcourant = self.dthydro = 1e20

    def tensor(self, f, a):
        n = self.s + (1 if f in NODE_STATE else 0)
        return torch.from_numpy(a).to(self.dev).reshape(n, n, n)

    def corners(self, st, names):
        return [[st[f][_at(n, self.s)] for n in range(8)] for f in names]

    def gather(self, c):
        s = self.s
        f = torch.zeros((s + 1,) * 3, dtype=torch.float64, device=self.dev)
        for n in (6, 7, 5, 4, 2, 3, 1, 0):  # a node's elements in ascending order
            f[_at(n, s)] += c[n]
        return f

    def advance(self):
        self.time_increment()
        with torch.no_grad():
            self.st, self.aux = self.cycle_map(self.st, self.dt, self.hgcoef, self.qlc, self.qqc, True)

    def time_increment(self):
        target = self.stoptime - self.time
        if self.cycle:
            old, new = self.dt, 1e20
            if self.dtcourant < new:
                new = self.dtcourant / 2.0
            if self.dthydro < new:
                new = self.dthydro * 2.0 / 3.0
            ratio = new / old
            if ratio >= 1.0:
                new = old if ratio < 1.1 else (old * 1.2 if ratio > 1.2 else new)
            self.dt = min(new, self.dtmax)
        if self.dt < target < 4.0 * self.dt / 3.0:
            target = 2.0 * self.dt / 3.0
        self.dt = min(self.dt, target)
        self.time += self.dt
        self.cycle += 1

    def pull_back(self, st, dt, shadow):
        """The adjoint of `st` from the adjoint of the state a cycle later,
        and of (hgcoef, qlc_monoq, qqc_monoq)."""
        leaf = {f: st[f].detach().clone().requires_grad_(True) for f in STATE}
        par = [torch.tensor(p, dtype=torch.float64, device=self.dev, requires_grad=True)
               for p in (self.hgcoef, self.qlc, self.qqc)]
        new, _ = self.cycle_map(leaf, dt, *par, False)
        ins = [leaf[f] for f in STATE] + par
        g = torch.autograd.grad([new[f] for f in STATE], ins, [shadow[f] for f in STATE],
                                allow_unused=True)
        g = [torch.zeros_like(i) if x is None else x for x, i in zip(g, ins)]
        return dict(zip(STATE, g)), np.array([float(x) for x in g[len(STATE):]])

    def cycle_map(self, st, dt, hgcoef, qlc, qqc, constraints):
        new, aux = self.nodal(st, dt, hgcoef)
        kin = self.kinematics(st, new, dt)
        self.material(st, new, kin, qlc, qqc, aux)
        aux.update(kin)
        if constraints:
            self.constraints(new, kin)
        return new, aux

    def nodal(self, st, dt, hgcoef):
        X = self.corners(st, "xyz")
        x, y, z = X
        # stress: face normals to their four corners, sigma = -p - q
        B = [[0.0] * 8 for _ in range(3)]
        for k, (a, b, c, d) in enumerate(_FACES):
            e0 = [0.5 * (t[d] + t[c] - t[b] - t[a]) for t in X]
            e1 = [0.5 * (t[c] + t[b] - t[d] - t[a]) for t in X]
            area = [0.25 * (e0[(i + 1) % 3] * e1[(i + 2) % 3] - e0[(i + 2) % 3] * e1[(i + 1) % 3])
                    for i in range(3)]
            for n in (a, b, c, d):
                for i in range(3):
                    B[i][n] = B[i][n] + area[i]
            if k == 4 and self.quirks & 1:  # the reference's face 5: y twice at node 1, no z
                B[1][0] = B[1][0] + area[1]
                B[2][0] = B[2][0] - area[2]
        ms = st["p"] + st["q"]
        stress = [[ms * B[i][n] for n in range(8)] for i in range(3)]
        # Flanagan-Belytschko hourglass
        determ = self.volo * st["v"]
        dv = _vol_derivative(x, y, z, self.quirks)
        V = self.corners(st, ("xd", "yd", "zd"))
        force = [[0.0] * 8 for _ in range(3)]
        for m in range(4):
            hm = [_add([_GAMMA[n][m] * t[n] for n in range(8)]) for t in X]
            g = [_GAMMA[n][m] - (1.0 / determ) * (dv[0][n] * hm[0] + dv[1][n] * hm[1] + dv[2][n] * hm[2])
                 for n in range(8)]
            for i in range(3):
                h = _dot(g, V[i])
                for n in range(8):
                    force[i][n] = force[i][n] + g[n] * h
        coef = -hgcoef * 0.01 * st["ss"] * self.elemMass / _cbrt(determ)
        f = [self.gather(stress[i]) + self.gather([coef * force[i][n] for n in range(8)])
             for i in range(3)]
        new, aux = {}, {}
        for i, (pos, vel) in enumerate((("x", "xd"), ("y", "yd"), ("z", "zd"))):
            acc = f[i] / self.nodalMass
            still = torch.zeros_like(acc)
            still[tuple(0 if a == 2 - i else slice(None) for a in range(3))] = 1.0
            acc = torch.where(still > 0, torch.zeros_like(acc), acc)
            v = st[vel] + acc * dt
            v = torch.where(v.abs() < 1e-7, torch.zeros_like(v), v)
            new[vel], new[pos] = v, st[pos] + v * dt
            aux["f" + pos], aux[vel + "d"] = f[i], acc
        return new, aux

    def kinematics(self, st, new, dt):
        X, V = self.corners(new, "xyz"), self.corners(new, ("xd", "yd", "zd"))
        volume = _volume(*X)
        vnew = volume / self.volo
        kin = {"vnew": vnew, "delv": vnew - st["v"]}
        with torch.no_grad():  # no field of the state depends on these
            big = torch.zeros_like(volume)
            for a, b, c, d in ((0, 1, 2, 3), (4, 5, 6, 7), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6),
                               (3, 0, 4, 7)):
                f = [(t[c] - t[a]) - (t[d] - t[b]) for t in X]
                g = [(t[c] - t[a]) + (t[d] - t[b]) for t in X]
                fg = _dot(f, g)
                big = torch.maximum(big, _dot(f, f) * _dot(g, g) - fg * fg)
            kin["arealg"] = 4.0 * volume / torch.sqrt(big)
            H = [[t[n] - 0.5 * dt * w[n] for n in range(8)] for t, w in zip(X, V)]
            (xx, xe, xz), (yx, ye, yz), (zx, ze, zz) = _jacobian(H)
            cof = ((ye * zz - ze * yz, zx * yz - yx * zz, yx * ze - zx * ye),
                   (ze * xz - xe * zz, xx * zz - zx * xz, zx * xe - xx * ze),
                   (xe * yz - ye * xz, yx * xz - xx * yz, xx * ye - yx * xe))
            det = 8.0 * (xe * cof[0][1] + ye * cof[1][1] + ze * cof[2][1])
            D = []
            for (cx, ce, cz), v in zip(cof, V):
                b = (-cx - ce - cz, cx - ce - cz, cx + ce - cz, -cx + ce - cz)
                D.append((b[0] * (v[0] - v[6]) + b[1] * (v[1] - v[7]) + b[2] * (v[2] - v[4])
                          + b[3] * (v[3] - v[5])) / det)
            kin["vdov"] = D[0] + D[1] + D[2]
            for i, f in enumerate(("dxx", "dyy", "dzz")):
                kin[f] = D[i] - kin["vdov"] / 3.0
        # monotonic-q gradients
        vol = self.volo * vnew
        norm = 1.0 / (vol + 1e-36)

        def side(t, a, b):
            return 0.25 * (_add([t[n] for n in a]) - _add([t[n] for n in b]))

        lo_hi = {"xi": ((1, 2, 6, 5), (0, 3, 7, 4)), "eta": ((3, 2, 6, 7), (0, 1, 5, 4)),
                 "zeta": ((4, 5, 6, 7), (0, 1, 2, 3))}
        d = {k: [side(t, *v) for t in X] for k, v in lo_hi.items()}
        for k, (a, b) in {"zeta": ("xi", "eta"), "xi": ("eta", "zeta"), "eta": ("zeta", "xi")}.items():
            u, w = d[a], d[b]
            n = [u[(i + 1) % 3] * w[(i + 2) % 3] - u[(i + 2) % 3] * w[(i + 1) % 3] for i in range(3)]
            kin["delx_" + k] = vol / torch.sqrt(_dot(n, n) + 1e-36)
            kin["delv_" + k] = _dot([t * norm for t in n], [side(t, *lo_hi[k]) for t in V])
        return kin

    def limiter(self, dv, axis):
        s = self.s
        own, zero = dv, torch.zeros_like(dv)
        first = own.narrow(axis, 0, 1)
        minus = torch.cat([first, own.narrow(axis, 0, s - 1)], axis)  # symmetry face: its own
        if axis == 2 and self.quirks & 4:  # the reference's xi-plus read is the element's own
            plus = torch.cat([own.narrow(2, 0, s - 1), zero.narrow(2, 0, 1)], 2)
        else:  # free face: zero
            plus = torch.cat([own.narrow(axis, 1, s - 1), zero.narrow(axis, 0, 1)], axis)
        norm = 1.0 / (dv + 1e-36)
        m, p = minus * norm, plus * norm
        phi = 0.5 * (m + p)
        m, p = m * 2.0, p * 2.0
        phi = torch.where(m < phi, m, phi)
        phi = torch.where(p < phi, p, phi)
        phi = torch.where(phi < 0.0, zero, phi)
        return torch.where(phi > 1.0, torch.ones_like(phi), phi)

    def material(self, st, new, kin, qlc, qqc, aux):
        vnew, delv = kin["vnew"], kin["delv"]
        zero = torch.zeros_like(vnew)
        lin, quad = zero, zero
        for k, axis in (("xi", 2), ("eta", 1), ("zeta", 0)):
            dv = kin["delv_" + k]
            phi = self.limiter(dv, axis)
            w = dv * kin["delx_" + k]
            w = torch.where(w > 0.0, zero, w)
            lin, quad = lin + w * (1.0 - phi), quad + w * w * (1.0 - phi * phi)
        rho = self.elemMass / (self.volo * vnew)
        grows = kin["vdov"] > 0.0
        ql = torch.where(grows, zero, -qlc * rho * lin)
        qq = torch.where(grows, zero, qqc * rho * quad)
        aux["ql"], aux["qq"] = ql, qq

        def pressure(e, comp):
            bvc = (2.0 / 3.0) * (comp + 1.0)
            p = bvc * e
            p = torch.where(p.abs() < 1e-7, zero, p)
            return bvc, torch.where(p < 0.0, zero, p)

        def sound(e, v2, bvc, p):
            c = (2.0 / 3.0) * e + v2 * bvc * p
            small = c <= 0.111111e-36
            return torch.where(small, zero + 0.333333e-18, torch.sqrt(torch.where(small, zero + 1.0, c)))

        def snap(e):
            return torch.where(e.abs() < 1e-7, zero, e)

        comp = 1.0 / vnew - 1.0
        half = 1.0 / (vnew - 0.5 * delv) - 1.0
        opens = delv > 0.0
        p0, q0 = st["p"], st["q"]
        e = st["e"] - 0.5 * delv * (p0 + q0)
        bvc, ph = pressure(e, half)
        vh = 1.0 / (1.0 + half)
        qn = torch.where(opens, zero, sound(e, vh * vh, bvc, ph) * ql + qq)
        e = snap(e + 0.5 * delv * (3.0 * (p0 + q0) - 4.0 * (ph + qn)))
        bvc, p = pressure(e, comp)
        qt = torch.where(opens, zero, sound(e, vnew * vnew, bvc, p) * ql + qq)
        e = snap(e - (7.0 * (p0 + q0) - 8.0 * (ph + qn) + (p + qt)) * delv * (1.0 / 6.0))
        bvc, p = pressure(e, comp)
        c = sound(e, vnew * vnew, bvc, p)
        qn = torch.where(opens, qn, snap(c * ql + qq))
        new["e"], new["p"], new["q"], new["ss"] = e, p, qn, c
        new["v"] = torch.where((vnew - 1.0).abs() < 1e-10, zero + 1.0, vnew)

    def constraints(self, new, kin):
        vdov, l = kin["vdov"], kin["arealg"]
        moves = vdov != 0.0
        far = torch.full_like(vdov, 1e20)
        c2 = new["ss"] * new["ss"]
        c2 = torch.where(vdov < 0.0, c2 + 256.0 * l * l * vdov * vdov, c2)
        courant = float(torch.where(moves, l / torch.sqrt(c2), far).min())
        hydro = float(torch.where(moves, 0.1 / (vdov.abs() + 1e-20), far).min())
        if courant < 1e20:
            self.dtcourant = courant
        if hydro < 1e20:
            self.dthydro = hydro
