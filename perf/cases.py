"""Workloads of the MCV step for timing two builds against each other.

Each case is work that a program hands to the public entry points
(mcv_sw_amd.capi): a solve advanced to its next output time and read back, an
ensemble or a mixed batch advanced together, one request served through a
resident batch, the spatial operator alone, one history record.  Sizes, time
steps and schemes are those of this repository's configurations and bench, or
generic sizes of the same range (odd ones among them).

  listed()      the named cases
  draw(rng)     one more case of the same ranges
  prepare       mesh, seeded initial state and the tuned handle or batch
  run           one pass; call it again to continue from where it ended
  exact         the same outputs in FP64 from plain torch, written from the
                scheme's formulas (no code of this repository)
  work          bytes and operations of one pass
  tolerance     distance that another correct implementation may show
"""
import functools
import math

import numpy as np
import torch

from mcv_sw_amd import capi, hostlib, serve

PRECISION = {"fp64": capi.FP64, "fp32c": capi.FP32C}
FIELDS = ("phi", "u", "v")
FILL = -9999999999999999.0
GRAVITY, RADIUS, OMEGA = 9.80616, 6371220.0, 7.292e-5


def listed():
    return [
        # the CPU-runnable configuration, hourly output: a step is a few
        # dependent launches on a nearly empty chip
        dict(name="solve_mcv3_n32_fp64_rk4", kind="solve", dof=3, n=32, prec="fp64",
             scheme="RK4", steps=15, dt=240.0, hill=False),
        # an odd small size in the FP32C form, three-stage scheme
        dict(name="solve_mcv4_n45_fp32c_rk3", kind="solve", dof=4, n=45, prec="fp32c",
             scheme="RK3_TVD", steps=60, dt=60.0, hill=False),
        # a middle resolution, hourly output
        dict(name="solve_mcv4_n96_fp64_rk4", kind="solve", dof=4, n=96, prec="fp64",
             scheme="RK4", steps=90, dt=40.0, hill=False),
        # about half a degree, odd, with orography (phi_s is read), RK3
        dict(name="solve_mcv3_n181_fp64_rk3_hill", kind="solve", dof=3, n=181, prec="fp64",
             scheme="RK3_TVD", steps=150, dt=24.0, hill=True),
        # the headline solve of the bench, hourly output, in both forms
        dict(name="solve_mcv4_n384_fp64_rk4", kind="solve", dof=4, n=384, prec="fp64",
             scheme="RK4", steps=360, dt=10.0, hill=False),
        dict(name="solve_mcv4_n384_fp32c_rk4", kind="solve", dof=4, n=384, prec="fp32c",
             scheme="RK4", steps=360, dt=10.0, hill=False),
        # the bench's uniform ensemble (its members' size, scheme and form), hourly output
        dict(name="ensemble_20x_mcv3_n90_fp32c_rk3", kind="ensemble", dof=3, n=90, prec="fp32c",
             scheme="RK3_TVD", members=20, steps=60, dt=60.0),
        # solves of several orders, sizes, schemes and forms in one batch, as serving holds them
        dict(name="batch_mixed_12", kind="mixed", count=12, mix=3, nmax=180, stages=120),
        # one served request on an otherwise idle batch: admit, run 6 h, read back, retire
        dict(name="request_mcv3_n64_fp32c", kind="request", dof=3, n=64, prec="fp32c",
             scheme="RK4", steps=290, dt=75.0),
        # the operator alone for a caller with its own time integration
        dict(name="tendency_mcv3_n90_fp64", kind="tendency", dof=3, n=90, noalloc=True),
        # ten minutes and one record of the output block
        dict(name="history_mcv4_n180_fp64_rk4", kind="history", dof=4, n=180, prec="fp64",
             scheme="RK4", steps=30, dt=20.0),
    ]


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "ensemble", "mixed", "request",
                       "tendency", "history"])
    dof = rng.choice([3, 4])
    prec = rng.choice(["fp64", "fp32c"])
    scheme = rng.choice(["RK4", "RK3_TVD"])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "tendency":
        return dict(kind=kind, dof=dof, n=size(8, 110), noalloc=rng.random() < 0.5)
    if kind == "mixed":
        return dict(kind=kind, count=rng.randint(4, 12), mix=rng.randint(0, 10 ** 6),
                    nmax=rng.choice([90, 128, 180]), stages=12 * rng.randint(4, 10))
    n = {"solve": lambda: size(16, 384 if dof == 4 else 512), "ensemble": lambda: size(24, 100),
         "request": lambda: size(32, 128), "history": lambda: size(24, 200)}[kind]()
    case = dict(kind=kind, dof=dof, n=n, prec=prec, scheme=scheme, dt=_dt(dof, n))
    if kind == "request":
        case["steps"] = rng.randint(40, 300)
    elif kind == "history":
        case["steps"] = rng.randint(2, 40)
    else:
        # the steps of an hour, fewer where that would pass the largest listed case
        per = 6 * n * n * (1 if kind == "solve" else 8)
        case["steps"] = max(2, min(int(3600 / case["dt"]), int(2.0e8 / per)))
    if kind == "solve":
        case["hill"] = rng.random() < 0.4
    if kind == "ensemble":
        case["members"] = rng.randint(4, 12)
    return case


def _dt(dof, n):
    """A whole-second time step at Courant 0.5 of the fastest gravity wave."""
    return max(1.0, math.floor(serve.cfl_dt(dof, n, 25.0, 6000.0)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=24)
def _mesh(dof, n):
    """Geometry and ghost tables, kept as a program that runs many solves does."""
    return hostlib.mesh(dof, n)


def _state(dof, n, seed, hill=False, h0=5960.0):
    """A zonal flow in balance about a tilted axis (Williamson case 2), its
    speed, tilt and a low height anomaly drawn from the seed; with `hill`, a
    mountain of Williamson case 5's shape drawn from the seed as well."""
    m = dict(_mesh(dof, n))
    r = np.random.default_rng(seed)
    u0, tilt, amp = r.uniform(15.0, 25.0), r.uniform(-0.3, 0.3), r.uniform(2.0, 5.0)
    lon0, lat0 = r.uniform(-math.pi, math.pi), r.uniform(-1.0, 1.0)
    lon, lat = m["lonP"], m["latP"]
    cl, sl, ct, st = np.cos(lon), np.sin(lon), np.cos(lat), np.sin(lat)
    ca, sa = math.cos(tilt), math.sin(tilt)
    axis = st * ca - cl * ct * sa
    # cosine of the angle to the anomaly's centre
    near = st * math.sin(lat0) + ct * math.cos(lat0) * np.cos(lon - lon0)
    phi = GRAVITY * h0 - (RADIUS * OMEGA * u0 + 0.5 * u0 * u0) * axis * axis
    phi += GRAVITY * amp * np.exp(10.0 * (near - 1.0))
    m["phi_s"] = np.zeros_like(phi)
    if hill:
        m["phi_s"] = GRAVITY * 500.0 * np.maximum(0.0, 1.0 - np.arccos(
            np.clip(near, -1.0, 1.0)) / (math.pi / 6))
        phi = phi - m["phi_s"]
    return m, hostlib.handoff(m, phi, u0 * (ct * ca + cl * st * sa), -u0 * sl * sa)


def _members(case, seed):
    """(dof, n, dt, scheme, precision name, seed) of every solve of a batch."""
    if case["kind"] == "ensemble":
        return [(case["dof"], case["n"], case["dt"], case["scheme"], case["prec"],
                 1000 * seed + k) for k in range(case["members"])]
    r = np.random.default_rng(case["mix"])
    out = []
    for k in range(case["count"]):
        dof = int(r.choice((3, 4)))
        n = int(round(math.exp(r.uniform(math.log(24), math.log(case["nmax"])))))
        out.append((dof, n, _dt(dof, n), ("RK4", "RK3_TVD")[int(r.integers(2))],
                    ("fp64", "fp32c")[int(r.integers(2))], 1000 * seed + k))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "mixed"):
        specs = _members(case, seed)
        b = capi.Batch(len(specs))
        slots = []
        for dof, n, dt, scheme, prec, sd in specs:
            m, st = _state(dof, n, sd)
            slots.append(b.add(dof, n, dt, m, st, 1 << 40, scheme=scheme,
                               precision=PRECISION[prec]))
        b.autotune(reps=3)
        stages = case["stages"] if kind == "mixed" else case["steps"] * _stages(case["scheme"])
        return dict(kind=kind, batch=b, slots=slots, stages=stages)
    if kind == "request":
        m, st = _state(case["dof"], case["n"], seed)
        return dict(kind=kind, case=case, batch=capi.Batch(8), mesh=m, state=st)
    if kind == "tendency":
        m, st = _state(case["dof"], case["n"], seed)
        s = capi.Solver(case["dof"], case["n"], _dt(case["dof"], case["n"]), m, st)
        s.autotune(reps=3)
        return dict(kind=kind, solver=s, state=st, noalloc=case["noalloc"])
    m, st = _state(case["dof"], case["n"], seed, hill=case.get("hill", False))
    s = capi.Solver(case["dof"], case["n"], case["dt"], m, st, scheme=case["scheme"],
                    precision=PRECISION[case["prec"]])
    s.autotune(reps=3)
    return dict(kind=kind, solver=s, steps=case["steps"])


def _stages(scheme):
    return 4 if scheme == "RK4" else 3


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "solve":
        s = state["solver"]
        s.step(state["steps"])
        return s.sync(fields=FIELDS)
    if kind == "history":
        s = state["solver"]
        s.step(state["steps"])
        return s.history_fields()
    if kind == "tendency":
        return state["solver"].tendency(state["state"], noalloc=state["noalloc"])
    b = state["batch"]
    if kind == "request":
        c = state["case"]
        slot = b.add(c["dof"], c["n"], c["dt"], state["mesh"], state["state"], c["steps"],
                     scheme=c["scheme"], precision=PRECISION[c["prec"]])
        b.run(c["steps"] * _stages(c["scheme"]))
        out = b.sync(slot, fields=FIELDS)
        b.remove(slot)
        return out
    b.run(state["stages"])
    outs = [b.sync(slot, fields=FIELDS) for slot in state["slots"]]
    return {"states": [{k: o[k] for k in FIELDS} for o in outs],
            "mass": np.array([o["mass"] for o in outs]),
            "energy": np.array([o["energy"] for o in outs])}


# ---------------------------------------------------------------------------
# What one pass cannot do without, and how far another implementation may be
# ---------------------------------------------------------------------------
def _step_bytes(dof, n, prec, scheme):
    """State words one step has to move through memory when its stages are
    separate sweeps: RK4 51 words per point (stage input and output, base
    state, tendency sum), RK3 24; the FP32C form 4-byte words, plus the
    residue of the base state read and written once, and per stage the FP64
    reference mass term and three FP32 constants."""
    pts = 6 * (n * (dof - 1) + 1) ** 2
    words = 51 if scheme == "RK4" else 24
    if prec == "fp64":
        return pts * words * 8
    return pts * (words * 4 + 24 + 20 * _stages(scheme))


def _step_flops(dof, n, scheme):
    """About 230 (MCV4) or 180 (MCV3) operations a point and stage: fits,
    fluxes and interior derivatives of three pairs in two directions, the
    tendencies and the update."""
    return 6 * (n * (dof - 1) + 1) ** 2 * (230 if dof == 4 else 180) * _stages(scheme)


def work(case):
    kind = case["kind"]
    if kind in ("ensemble", "mixed"):
        b = f = 0.0
        for dof, n, _, scheme, prec, _ in _members(case, 0):
            steps = case["stages"] / _stages(scheme) if kind == "mixed" else case["steps"]
            b += steps * _step_bytes(dof, n, prec, scheme) + _points(dof, n) * 3 * 8
            f += steps * _step_flops(dof, n, scheme)
        return {"bytes": b, "flops": f}
    pts = _points(case["dof"], case["n"])
    if kind == "tendency":
        # five input fields, three metric terms and f, three tendencies
        return {"bytes": pts * 12 * 8.0, "flops": _step_flops(case["dof"], case["n"], "RK4") / 4.0}
    b = case["steps"] * float(_step_bytes(case["dof"], case["n"], case["prec"], case["scheme"]))
    f = case["steps"] * float(_step_flops(case["dof"], case["n"], case["scheme"]))
    # read-back: phi, u, v, or the eight point fields of a record; a request's
    # mesh (four 2x2 matrices, sqrtG, f, phi_s) and state come in as well
    b += pts * 8.0 * {"solve": 3, "history": 8, "request": 3 + 19 + 6}[kind]
    return {"bytes": b, "flops": f}


def _points(dof, n):
    return 6 * (n * (dof - 1) + 1 + 2 * (dof - 1)) ** 2


def tolerance(case):
    # FP64: rounding in another order, grown over the pass (measured against
    # the restatement below: at most 2e-14; 1e-12 for the tendency of phiG,
    # whose terms cancel).  FP32C: the form's own distance from FP64, whose
    # stencil is FP32 (measured: at most 8e-7, in the small wind component).
    if case["kind"] == "tendency":
        return {"rel": 4e-12}
    if case["kind"] == "mixed" or case["prec"] == "fp32c":
        return {"rel": 4e-6}
    if case["kind"] == "history":
        # the fill values at the halo corners would hide every other point in
        # a norm; the FP64 form is bit-identical to the reference by contract
        return "exact"
    return {"rel": 1e-13}


# ---------------------------------------------------------------------------
# The scheme in plain torch, FP64
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "mixed"):
        specs = _members(case, seed)
        stages = [case["stages"] if kind == "mixed" else case["steps"] * _stages(s[3])
                  for s in specs]
        if not _affordable(sum(_points(s[0], s[1]) * k for s, k in zip(specs, stages)),
                           sum(stages)):
            return None
        outs = []
        for (dof, n, dt, scheme, _, sd), k in zip(specs, stages):
            e = _Exact(dof, n, *_state(dof, n, sd))
            e.step(dt, scheme, k // _stages(scheme))
            outs.append(e.output())
        return {"states": [{k: o[k] for k in FIELDS} for o in outs],
                "mass": np.array([o["mass"] for o in outs]),
                "energy": np.array([o["energy"] for o in outs])}
    if kind == "tendency":
        e = _Exact(case["dof"], case["n"], *_state(case["dof"], case["n"], seed))
        return dict(zip(("phiG", "u", "v"), (t.cpu().numpy() for t in e.tendency())))
    stages = case["steps"] * _stages(case["scheme"])
    if not _affordable(_points(case["dof"], case["n"]) * stages, stages):
        return None
    e = _Exact(case["dof"], case["n"],
               *_state(case["dof"], case["n"], seed, hill=case.get("hill", False)))
    e.step(case["dt"], case["scheme"], case["steps"])
    return e.history() if kind == "history" else e.output()


def _affordable(point_stages, stages):
    """Whether the torch restatement ends within about 20 seconds."""
    return point_stages < (2.5e9 if torch.cuda.is_available() else 1e8) and stages < 3000


class _Exact:
    """One solve: fields (6, nh, nh) as [panel, j, i], H halo points each side."""

    def __init__(self, dof, n, mesh, state):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.D, self.H, self.n, self.dx = dof, dof - 1, n, mesh["dx"]
        self.npv = n * self.H + 1
        t = self._t
        self.sg, self.f, self.phis = t(mesh["sqrtG"]), t(mesh["f"]), t(mesh["phi_s"])
        IG, G, A, IA = t(mesh["IG"]), t(mesh["G"]), t(mesh["A"]), t(mesh["IA"])
        self.g11, self.g12, self.g22 = IG[..., 0, 0], IG[..., 1, 0], IG[..., 1, 1]
        self.p2s, self.s2p = self._mul(A, IG), self._mul(G, IA)  # [..., col, row]
        self.phi, self.u, self.v = (t(state[k]).clone() for k in FIELDS)
        self.cu, self.cv = t(state["contraU"]), t(state["contraV"])
        self._connect(mesh["lonP"], mesh["latP"])
        self.cell = torch.as_tensor(np.asarray(mesh["iref"]) - 1, device=self.dev).long()
        self.off = t(mesh["coef"]) / self.dx
        self.inner = (slice(None), slice(self.H, self.H + self.npv),
                      slice(self.H, self.H + self.npv))

    def _t(self, a):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=self.dev)

    @staticmethod
    def _mul(a, b):
        return torch.stack([torch.stack([a[..., 0, r] * b[..., c, 0] + a[..., 1, r] * b[..., c, 1]
                                         for r in range(2)], -1) for c in range(2)], -2)

    # --- cube topology, from the coordinates of the panels' edge points ---
    def _line(self, side, depth, along=None):
        """(rows, columns) of line `depth` (0 = the edge, negative = halo) at
        side W, E, S, N, for along-line positions (default all owned)."""
        H, npv = self.H, self.npv
        s = (torch.arange(npv, device=self.dev) if along is None else along) + H
        at = torch.full_like(s, H + depth if side in (0, 2) else H + npv - 1 - depth)
        return (s, at) if side < 2 else (at, s)

    def _connect(self, lon, lat):
        xyz = torch.stack([self._t(np.cos(lat) * np.cos(lon)), self._t(np.cos(lat) * np.sin(lon)),
                           self._t(np.sin(lat))], -1)
        edges = {(p, s): xyz[p][self._line(s, 0)] for p in range(6) for s in range(4)}
        self.link = {}
        for a, ea in edges.items():
            for b, eb in edges.items():
                if a[0] != b[0]:
                    for rev in (False, True):
                        if (ea - (eb.flip(0) if rev else eb)).abs().max() < 1e-9:
                            self.link[a] = (b[0], b[1], rev)
        assert len(self.link) == 24
        H, e = self.H, self.H + self.npv - 1
        corners = [(p, j, i) for p in range(6) for j in (H, e) for i in (H, e)]
        self.vertices = []
        while corners:
            p, j, i = corners[0]
            same = [c for c in corners
                    if (xyz[c[0], c[1], c[2]] - xyz[p, j, i]).abs().max() < 1e-9]
            assert len(same) == 3
            self.vertices.append(same)
            corners = [c for c in corners if c not in same]

    # --- boundary pass: halo from the neighbours' lines, shared points averaged ---
    def _wind(self, M, p, at, a, b):
        m = M[p][at]
        return m[..., 0, 0] * a + m[..., 1, 0] * b, m[..., 0, 1] * a + m[..., 1, 1] * b

    def _interp(self, q, c):
        """Lagrange interpolation over a cell's DOF points at offset c in [0, 1]."""
        k = torch.arange(self.D, device=self.dev, dtype=torch.float64) / self.H
        out = 0.0
        for a in range(self.D):
            w = q[a]
            for b in range(self.D):
                if b != a:
                    w = w * (c - k[b]) / (k[a] - k[b])
            out = out + w
        return out

    def _boundary(self, phi, u, v):
        H, npv = self.H, self.npv
        raw = phi.clone(), u.clone(), v.clone()

        def sphere(p, at):
            return (raw[0][p][at],) + self._wind(self.p2s, p, at, raw[1][p][at], raw[2][p][at])

        for (p, side), (q, sd, rev) in self.link.items():
            for k in range(1, H + 1):
                pts = []
                for a in range(self.D):
                    t = self.cell[k - 1] * H + a
                    pts.append(sphere(q, self._line(sd, k, npv - 1 - t if rev else t)))
                at = self._line(side, -k)
                g = [self._interp([x[f] for x in pts], self.off[k - 1]) for f in range(3)]
                phi[p][at] = g[0]
                u[p][at], v[p][at] = self._wind(self.s2p, p, at, g[1], g[2])
        mid = torch.arange(1, npv - 1, device=self.dev)
        for (p, side), (q, sd, rev) in self.link.items():
            at = self._line(side, 0, mid)
            a, b = sphere(p, at), sphere(q, self._line(sd, 0, npv - 1 - mid if rev else mid))
            g = [0.5 * (x + y) for x, y in zip(a, b)]
            phi[p][at] = g[0]
            u[p][at], v[p][at] = self._wind(self.s2p, p, at, g[1], g[2])
        for same in self.vertices:
            pts = [sphere(p, (j, i)) for p, j, i in same]
            g = [(pts[0][f] + pts[1][f] + pts[2][f]) / 3.0 for f in range(3)]
            for p, j, i in same:
                phi[p, j, i] = g[0]
                u[p, j, i], v[p, j, i] = self._wind(self.s2p, p, (j, i), g[1], g[2])

    # --- spatial operator ---
    def _fits(self, a):
        """Derivatives at the right end of the cell left of every cell end, and
        at the left end of the cell right of it; and the owned cells' points."""
        c = a.unfold(-1, self.D, self.H)
        p, dx = [c[..., k] for k in range(self.D)], self.dx
        if self.D == 3:
            left = -(p[2] - 4 * p[1] + 3 * p[0]) / dx
            right = (p[0] - 4 * p[1] + 3 * p[2]) / dx
        else:
            left = (-11 * p[0] + 18 * p[1] - 9 * p[2] + 2 * p[3]) / (2 * dx)
            right = (11 * p[3] - 18 * p[2] + 9 * p[1] - 2 * p[0]) / (2 * dx)
        return right[..., :-1], left[..., 1:], c[..., 1:-1, :]

    def _derivative(self, flux, q, speed):
        """d(flux) along the last axis at the owned points, dissipation on q."""
        fl, fr, c = self._fits(flux)
        ql, qr, _ = self._fits(q)
        end = 0.5 * (fl + fr - speed * (qr - ql))
        out = torch.empty(flux.shape[:-1] + (self.npv,), dtype=torch.float64, device=self.dev)
        out[..., ::self.H] = end
        l, r, dx = end[..., :-1], end[..., 1:], self.dx
        if self.D == 3:
            out[..., 1::2] = 1.5 * (c[..., 2] - c[..., 0]) / dx - 0.25 * (l + r)
        else:
            via = 4.0 / 3.0 * (c[..., 3] - c[..., 0]) / dx
            curv = 4.0 / 27.0 * dx * (4.5 * (c[..., 0] - c[..., 1] - c[..., 2] + c[..., 3])
                                      / (dx * dx))
            out[..., 1::3] = via - (4 * l + 5 * r) / 27.0 - curv
            out[..., 2::3] = via - (5 * l + 4 * r) / 27.0 + curv
        return out

    def _sweep(self, E, PG, along, across, c, g, phi):
        ends = slice(self.H, self.H + self.npv, self.H)
        ce, gw = c[..., ends], torch.sqrt(g[..., ends] * phi[..., ends])
        lam = torch.maximum((ce - gw).abs(), (ce + gw).abs())
        up = torch.where(ce < 0, -1.0, 1.0).to(torch.float64)
        return (self._derivative(E, along, lam), self._derivative(PG * c, PG, lam),
                self._derivative(across, across, up))

    def _operator(self, phi, u, v, cu, cv):
        PG = phi * self.sg
        E = phi + self.phis + 0.5 * (cu * u + cv * v)
        own = slice(self.H, self.H + self.npv)
        rows = [x[:, own, :] for x in (E, PG, u, v, cu, self.g11, phi)]
        cols = [x[:, :, own].transpose(1, 2) for x in (E, PG, v, u, cv, self.g22, phi)]
        fx, dx, vx = self._sweep(*rows)
        fy, dy, uy = (x.transpose(1, 2) for x in self._sweep(*cols))
        i = self.inner
        sg = self.sg[i]
        turn = sg * ((vx - uy) / sg + self.f[i])
        return -dx - dy, -fx + turn * cv[i], -fy - turn * cu[i]

    def _contra(self, u, v):
        return self.g11 * u + self.g12 * v, self.g12 * u + self.g22 * v

    def tendency(self):
        return self._operator(self.phi, self.u, self.v, self.cu, self.cv)

    def step(self, dt, scheme, count):
        i, first = self.inner, True
        sg = self.sg[i]
        for _ in range(count):
            base = [self.phi[i] * sg, self.u[i].clone(), self.v[i].clone()]
            cur, ks = [self.phi, self.u, self.v], []

            def advance(new):
                out = [x.clone() for x in (self.phi, self.u, self.v)]
                out[0][i], out[1][i], out[2][i] = new[0] / sg, new[1], new[2]
                self._boundary(*out)
                return out

            for s in range(_stages(scheme)):
                c = (self.cu, self.cv) if first else self._contra(cur[1], cur[2])
                first = False
                k = self._operator(*cur, *c)
                now = [cur[0][i] * sg, cur[1][i], cur[2][i]]
                if scheme == "RK4":
                    ks.append(k)
                    if s < 3:
                        h = dt if s == 2 else 0.5 * dt
                        new = [b + h * x for b, x in zip(base, k)]
                    else:
                        new = [b + dt * (w + 2 * x + 2 * y + z) / 6.0
                               for b, w, x, y, z in zip(base, *ks)]
                else:
                    a, w = ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0))[s]
                    new = [a * b + w * (x + dt * y) for b, x, y in zip(base, now, k)]
                cur = advance(new)
            self.phi, self.u, self.v = cur
        self.cu, self.cv = self._contra(self.u, self.v)

    # --- read-back ---
    def _weights(self):
        w = [1.0, 4.0, 1.0] if self.D == 3 else [1.0, 3.0, 3.0, 1.0]
        return [[x * y / sum(w) ** 2 for x in w] for y in w]

    def _cell_sum(self, a):
        w, n, H = self._weights(), self.n, self.H
        e = (n - 1) * H + 1
        return sum(w[b][c] * a[:, b:b + e:H, c:c + e:H]
                   for b in range(self.D) for c in range(self.D))

    def output(self):
        i, norm = self.inner, {3: 1.0, 4: 64.0 / 80.0}[self.D]
        phi, sg = self.phi[i], self.sg[i]
        kin = 0.5 * phi * (self.u[i] * self.cu[i] + self.v[i] * self.cv[i])
        pot = 0.5 * (phi + self.phis[i]) ** 2
        out = {k: getattr(self, k).cpu().numpy() for k in FIELDS}
        out["mass"] = float(norm * self._cell_sum(phi * sg).sum())
        out["energy"] = float(norm * self._cell_sum(sg * (kin + pot)).sum())
        return out

    def history(self):
        phi, u, v = (x.clone() for x in (self.phi, self.u, self.v))
        edge = torch.ones(phi.shape[-1], dtype=torch.bool, device=self.dev)
        edge[self.H:self.H + self.npv] = False
        for x in (phi, u, v):
            x[:, edge[:, None] & edge[None, :]] = FILL
        cu, cv = self._contra(u, v)
        m = self.p2s
        rec = dict(u=u, v=v, contraU=cu, contraV=cv, phi=phi, phi_t=phi + self.phis,
                   zonal=m[..., 0, 0] * u + m[..., 1, 0] * v,
                   meridional=m[..., 0, 1] * u + m[..., 1, 1] * v)
        norm = {3: 1.0, 4: 64.0 / 80.0}[self.D]
        for k, x in (("uC", u), ("vC", v), ("phiC", phi)):
            rec[k] = torch.zeros((6, self.n + 2, self.n + 2), dtype=torch.float64,
                                 device=self.dev)
            rec[k][:, 1:-1, 1:-1] = norm * self._cell_sum(x[self.inner])
        return {k: x.cpu().numpy() for k, x in rec.items()}
