"""What a user of this framework has it do, as cases that can be timed.

Every case goes through the public entry points of `lbmflow_amd`: a solver is
built once with its geometry, rotating body, closures and initial flow
(`prepare`), and one pass steps it on and reads back what the caller of such a
run looks at (`run`): the torque of every step, the tracer's CV samples, the
velocity field, the gradients.

Kinds
  cavity   lid-driven cavity: six walls, the top one moving (plain method)
  box      periodic box with a uniform body force (no wall at all, odd sizes)
  channel  Zou-He inlet and outlet in x, walls in y, periodic z
  tank     stirred tank with a rotating immersed-boundary impeller, and as
           options the WALE closure before every step, a passive scalar
           (D3Q7 or on the hydro lattice) with its CV sampled, the blade
           lattice or the surface-sampled markers
  batch    several tanks stepped together by one persistent launch
  adjoint  gradient of the mean shaft torque (binomial checkpoints)

`exact` recomputes the closed ones and the channel in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import lbmflow_amd as L

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def _case(kind, dims, steps, lattice, collision, storage, nu, **more):
    d = {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "steps": steps, "lattice": lattice,
         "collision": collision, "storage": storage, "nu": nu}
    if kind in ("tank", "batch", "adjoint"):
        d.update({"wale": False, "scalar": "none", "cv_every": 0, "markers": "lattice"})
    d.update(more)
    return d


def _cube(n):
    return (n, n, n)


def listed():
    out = [
        # a small cavity stepped a few times between looks at its field: the
        # interactive and test-suite scale, all latency and launches
        _case("cavity", _cube(32), 10, 19, "trt", "f32", 0.015, name="cavity32_trt_f32"),
        # the plain-method configuration: the 64^3 cavity at Re 100
        _case("cavity", _cube(64), 250, 19, "trt", "f32", 0.031, name="cavity64_trt_f32"),
        # decaying turbulence in a periodic box of ragged size, bf16 storage
        _case("box", (201, 147, 173), 50, 27, "trt", "bf16", 0.01, name="box201_q27_trt_bf16"),
        # the open channel (velocity inlet, pressure outlet)
        _case("channel", (384, 128, 128), 60, 19, "trt", "f32", 0.02, name="channel384_trt_f32"),
        # a screening tank as the scenario runner sets one up: TRT, scalar on
        # the hydro lattice, CV at the probe steps
        _case("tank", _cube(96), 60, 19, "trt", "f32", 0.02, scalar="hydro", cv_every=20, name="tank96_trt_scalar"),
        # the tank of the adjoint configuration stepped forward (one body, LDS path)
        _case("tank", _cube(128), 200, 19, "trt", "f32", 0.01, name="tank128_trt_f32"),
        # the storage-precision run: central moments, fp16 storage, D3Q7 tracer
        # with a CV sample every ten steps
        _case("tank", _cube(128), 100, 27, "cm", "f16", 0.01, scalar="d3q7", cv_every=10, name="tank128_cm_f16_tracer"),
        # 12k surface-sampled blade markers and the WALE closure every step
        _case("tank", _cube(256), 60, 27, "cm", "f32", 0.00025, wale=True, markers="surface",
              name="tank256_surface_wale"),
        # the headline tank
        _case("tank", _cube(512), 24, 27, "cm", "f32", 0.005, name="tank512_cm_f32"),
        # the 512^3 precision run: fp16 storage, WALE, D3Q7 tracer
        _case("tank", _cube(512), 14, 27, "cm", "f16", 0.0005, wale=True, scalar="d3q7", cv_every=7,
              name="tank512_f16_wale_tracer"),
        # a sweep of tanks of uneven size in one persistent launch
        _case("batch", (48, 160, 0), 60, 19, "trt", "f32", 0.01, members=15, sizes_seed=20260512,
              name="batch15_trt_f32"),
        # torque gradient with binomial checkpointing
        _case("adjoint", _cube(128), 48, 19, "trt", "f32", 0.01, window=12, snapshots=8, name="adjoint128_trt_f32"),
    ]
    return out


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sizes spread over their logarithm,
    mostly ragged, every storage and option."""
    kind = rng.choice(["cavity", "box", "channel", "tank", "tank", "tank", "tank", "batch", "adjoint"])
    storage = rng.choice(["f32", "f32", "f16", "bf16"])
    lattice, collision = rng.choice([(19, "trt"), (27, "cm"), (27, "cm"), (27, "trt"), (19, "bgk")])
    nu = round(math.exp(rng.uniform(math.log(0.008), math.log(0.03))), 5)
    if kind == "cavity":
        n = _log_int(rng, 24, 200)
        return _case("cavity", _cube(n), rng.randint(10, 120), lattice, collision, storage, nu)
    if kind == "box":
        d = tuple(_log_int(rng, 40, 260) for _ in range(3))
        return _case("box", d, rng.randint(10, 60), lattice, collision, storage, nu)
    if kind == "channel":
        d = (_log_int(rng, 96, 512), _log_int(rng, 40, 160), _log_int(rng, 40, 160))
        return _case("channel", d, rng.randint(10, 60), 19, "trt", storage, max(nu, 0.012))
    if kind == "batch":
        lo = rng.randint(40, 72)
        return _case("batch", (lo, lo + rng.randint(16, 88), 0), rng.randint(10, 60), 19, "trt", "f32", nu,
                     members=rng.randint(2, 15), sizes_seed=rng.randint(1, 10 ** 6))
    if kind == "adjoint":
        n = rng.randint(40, 120)
        steps = rng.randint(16, 48)
        return _case("adjoint", _cube(n), steps, 19, rng.choice(["trt", "bgk"]), "f32", nu, window=steps // 4,
                     snapshots=rng.randint(3, 10))
    n = _log_int(rng, 48, 320)
    wale = rng.random() < 0.5
    scalar = rng.choice(["none", "d3q7", "d3q7", "hydro"])
    return _case("tank", _cube(n), rng.randint(10, 60 if n < 200 else 24), lattice, collision, storage,
                 round(nu / 10, 6) if wale else nu, wale=wale, scalar=scalar, cv_every=rng.choice([5, 10]),
                 markers="surface" if rng.random() < 0.3 else "lattice")


# ---------------------------------------------------------------------------
# geometry and inputs
# ---------------------------------------------------------------------------

LID = 0.05
INLET = 0.05


def _tank_numbers(n, tip=0.05):
    T = 15.0 * n / 16.0
    D = T / 3.0
    return {"T": T, "D": D, "C": T / 3.0, "bw": T / 10.0, "bt": T / 48.0, "omega": tip / (0.5 * D)}


def _markers(n, g, kind):
    args = ((n, n, n), 1.0, g["T"], g["T"], g["D"], g["C"], 6, 0.0, g["omega"])
    if kind == "surface":
        pos, w, _, c = L.impeller_surface_markers(*args, 0.04, 0.1, 20260512)
    else:
        pos, w, _, c = L.radial_impeller(*args)
    return pos, w, c


def _members(case):
    """Edges, tip speeds and viscosities of a batch's tanks."""
    r = np.random.RandomState(case["sizes_seed"])
    lo, hi = case["nx"], case["ny"]
    return [(int(r.randint(lo, hi + 1)), float(r.uniform(0.02, 0.06)), float(r.uniform(0.6, 1.6)) * case["nu"])
            for _ in range(case["members"])]


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _flow(dims, seed, base=(0.0, 0.0, 0.0), amp=0.012):
    """A smooth seeded flow: three modes per component over the box, density
    within 1e-3 of one.  rho (N,), u (N, 3), float32 on the device."""
    nx, ny, nz = dims
    r = np.random.RandomState(seed % (2 ** 31))
    dev = _device()
    ax = [torch.arange(n, device=dev, dtype=torch.float32) * (2.0 * math.pi / n) for n in (nx, ny, nz)]

    def mode():
        k = r.randint(1, 4, 3)
        p = r.uniform(0.0, 2.0 * math.pi, 3)
        s = [torch.sin(int(k[a]) * ax[a] + float(p[a])) for a in range(3)]
        return s[2][:, None, None] * s[1][None, :, None] * s[0][None, None, :]

    u = torch.empty((nz, ny, nx, 3), device=dev, dtype=torch.float32)
    for a in range(3):
        u[..., a] = base[a] + amp * (mode() + 0.6 * mode() + 0.4 * mode())
    rho = 1.0 + 1e-3 * mode()
    return rho.reshape(-1), u.reshape(-1, 3)


def _blob(n, seed):
    """Tracer pulse: a Gaussian near the liquid's surface, its place seeded."""
    r = np.random.RandomState((seed + 77) % (2 ** 31))
    dev = _device()
    sig = max(3.0, n / 16.0)
    c = [n / 2 + float(r.uniform(-0.1, 0.1)) * n, n / 2 + float(r.uniform(-0.1, 0.1)) * n, 0.75 * n]
    e = [torch.exp(-(torch.arange(n, device=dev, dtype=torch.float64) + 0.5 - c[a]) ** 2 / (2 * sig * sig))
         for a in range(3)]
    return (e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]).float().reshape(-1)


def _host(t):
    return t.cpu().numpy()


def _make_tank(n, lattice, collision, storage, nu, seed, tip=0.05, markers="lattice"):
    g = _tank_numbers(n, tip)
    s = L.Solver(lattice, _cube(n), nu=nu, collision=collision, storage=storage)
    s.build_stirred_tank(1.0, g["T"], g["T"], 4, g["bw"], g["bt"])
    pos, w, c = _markers(n, g, markers)
    s.set_rotating_body(pos, w, c, (0.0, 0.0, g["omega"]))
    rho, u = _flow(_cube(n), seed)
    s.init_with(_host(rho), _host(u))
    return s


def _force(case):
    return (1e-5, 0.0, -2e-6) if case["kind"] == "box" else (0.0, 0.0, 0.0)


def prepare(case, seed):
    kind, dims = case["kind"], (case["nx"], case["ny"], case["nz"])
    st = {"case": case}
    if kind == "batch":
        st["solvers"] = [_make_tank(n, case["lattice"], case["collision"], case["storage"], nu, seed + 31 * k, tip)
                         for k, (n, tip, nu) in enumerate(_members(case))]
        st["batch"] = L.Batch(st["solvers"])
        return st
    if kind in ("tank", "adjoint"):
        n = dims[0]
        s = _make_tank(n, case["lattice"], case["collision"], case["storage"], case["nu"], seed,
                       markers=case["markers"])
        if kind == "adjoint":
            s.set_omega_field(_host(_omega(case, seed)))
        if case["wale"]:
            s.set_wale(True)
        if case["scalar"] != "none":
            st["k"] = s.enable_scalar_distribution(_diffusivity(case), case["scalar"])
            b = _blob(n, seed)
            b[torch.from_numpy(s.solid() != 0).to(b.device)] = 0.0
            s.set_scalar_concentration(st["k"], _host(b))
        st["s"] = s
        return st
    if kind == "cavity":
        s = L.Solver(case["lattice"], dims, nu=case["nu"], collision=case["collision"], storage=case["storage"])
        lid = np.zeros((6, 3))
        lid[5, 0] = LID
        s.build_wall_rims([1] * 6, lid)
        rho, u = _flow(dims, seed)
    elif kind == "box":
        s = L.Solver(case["lattice"], dims, nu=case["nu"], collision=case["collision"], storage=case["storage"],
                     periodic=(True, True, True), force=_force(case))
        rho, u = _flow(dims, seed)
    else:
        solid = np.zeros((dims[2], dims[1], dims[0]), np.uint8)
        solid[:, 0, :] = solid[:, -1, :] = 1
        s = L.Solver(case["lattice"], dims, nu=case["nu"], collision=case["collision"], storage=case["storage"],
                     periodic=(False, False, True), solid=solid.reshape(-1))
        s.set_face_bc("x-", "velocity", (INLET, 0.0, 0.0))
        s.set_face_bc("x+", "pressure", (1.0,))
        rho, u = _flow(dims, seed, base=(INLET, 0.0, 0.0), amp=0.004)
    s.init_with(_host(rho), _host(u))
    st["s"] = s
    return st


def _diffusivity(case):
    return max(case["nu"], 0.005)


def _omega(case, seed):
    """Per-cell omega_plus of a viscosity field within 10 % of the base."""
    dims = (case["nx"], case["ny"], case["nz"])
    rho, _ = _flow(dims, seed + 5)
    nu = case["nu"] * (1.0 + 100.0 * (rho - 1.0))
    return 1.0 / (3.0 * nu + 0.5)


def _fields(s):
    rho, ux, uy, uz = s.moments()
    return {"rho": rho, "ux": ux, "uy": uy, "uz": uz}


def run(state):
    case = state["case"]
    kind, steps = case["kind"], case["steps"]
    if kind == "batch":
        out = {"torque": state["batch"].run(steps)}
        for k, s in enumerate(state["solvers"]):
            rho, ux, uy, uz = s.moments()
            out[f"u{k:02d}"] = [ux, uy, uz]
        return out
    s = state["s"]
    if kind == "adjoint":
        return s.adjoint_torque(steps, case["window"], case["snapshots"])
    if kind == "tank":
        every = case["cv_every"] if case["scalar"] != "none" else steps
        torque, cv, done = [], [], 0
        while done < steps:
            k = min(every, steps - done)
            tq, _ = s.run_with_ibm(k)
            torque.append(tq)
            done += k
            if case["scalar"] != "none":
                cv.append(s.scalar_cv(state["k"]))
        out = {"torque": np.concatenate(torque)}
        if case["scalar"] != "none":
            out["cv"] = np.array(cv)
            out["conc"] = s.gather_scalar_concentration(state["k"])
        out.update(_fields(s))
        return out
    s.run(steps)
    return _fields(s)


def _tank_fluid(n):
    """Fluid cells of the tank's mask, near enough for the byte count."""
    return 0.64 * n ** 3


def work(case):
    """Each population, scalar, velocity and omega value once in and once out
    per step, plus the read-back; the closure reads the populations once more
    (its velocities have to be known before any cell collides)."""
    kind, Q, steps = case["kind"], case["lattice"], case["steps"]
    S = 4 if case["storage"] == "f32" else 2
    flop_cell = 250 if Q == 19 else (500 if case["collision"] == "cm" else 350)
    n_all = case["nx"] * case["ny"] * max(case["nz"], 1)
    if kind == "batch":
        fluid = sum(_tank_fluid(n) for n, _, _ in _members(case))
        n_all = sum(n ** 3 for n, _, _ in _members(case))
        return {"bytes": fluid * steps * 2 * Q * S + 12 * n_all, "flops": fluid * steps * flop_cell}
    fluid = _tank_fluid(case["nx"]) if kind in ("tank", "adjoint") else float(n_all)
    cell = 2 * Q * S
    if kind == "adjoint":
        # forward, forward again once, and the adjoint populations in f64 both ways
        return {"bytes": fluid * steps * (2 * cell + Q * S + 2 * Q * 8), "flops": fluid * steps * 4 * flop_cell}
    if kind == "tank":
        if case["wale"]:
            cell += Q * S + 2 * 12 + 2 * 4
        if case["scalar"] != "none":
            cell += 2 * 4 * (7 if case["scalar"] == "d3q7" else Q)
    return {"bytes": fluid * steps * cell + 16 * n_all, "flops": fluid * steps * flop_cell}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------

_C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
      (1, 0, 1), (-1, 0, -1), (0, 1, 1), (0, -1, -1), (1, -1, 0), (-1, 1, 0), (1, 0, -1), (-1, 0, 1), (0, 1, -1),
      (0, -1, 1), (1, 1, 1), (-1, -1, -1), (1, 1, -1), (-1, -1, 1), (1, -1, 1), (-1, 1, -1), (1, -1, -1), (-1, 1, 1)]


def _opp(q):
    return 0 if q == 0 else (q + 1 if q % 2 else q - 1)


def _weights(Q):
    by = {7: (1 / 4, 1 / 8), 19: (1 / 3, 1 / 18, 1 / 36), 27: (8 / 27, 2 / 27, 1 / 54, 1 / 216)}[Q]
    return [by[sum(abs(v) for v in _C[q])] for q in range(Q)]


def _dot(c, v):
    """c . v with the zero terms left out; None when all are."""
    acc = None
    for a in range(3):
        if c[a]:
            t = v[a] if c[a] > 0 else -v[a]
            acc = t if acc is None else acc + t
    return acc


def _roll(t, c):
    s = [(-a - 1, c[a]) for a in range(3) if c[a]]
    return torch.roll(t, [v for _, v in s], [d for d, _ in s]) if s else t


class _Exact:
    """One domain in 64 bits: planes f[q] of shape (nz, ny, nx), deviation form."""

    def __init__(self, Q, dims, nu, collision, solid, rho, u, periodic=False, wall=None, force=(0.0, 0.0, 0.0),
                 omega=None):
        self.Q, self.dims, self.nu, self.kind = Q, dims, nu, collision
        nx, ny, nz = dims
        self.shape = (nz, ny, nx)
        self.dev = _device()
        self.W = _weights(Q)
        self.solid = None if solid is None else torch.from_numpy(solid.reshape(self.shape) != 0).to(self.dev)
        self.wall = wall
        self.F = [float(np.float32(v)) for v in force]
        tau = 3.0 * nu + 0.5
        self.op = float(np.float32(1.0 / tau))
        self.om = float(np.float32(1.0 / ((3.0 / 16.0) / (tau - 0.5) + 0.5) if collision == "trt" else 1.0 / tau))
        self.tau = tau
        self.omega = None if omega is None else omega.double().reshape(self.shape)
        self.links = None
        if self.solid is not None:
            self.links = [None] + [_roll(self.solid, _C[q]) & ~self.solid for q in range(1, Q)]
        self.ibm = self.hs = None
        self.wale = False
        self.Fm = self.Fc = None  # per listed cell
        self.face = False
        self._init(rho.double().reshape(self.shape), [u[:, a].double().reshape(self.shape) for a in range(3)],
                   periodic, tau)

    def _init(self, r, u, periodic, tau):
        f = self.equilibrium(r, u)
        per = periodic if isinstance(periodic, tuple) else (periodic,) * 3
        grad = []
        for ax in range(3):
            e = [0, 0, 0]
            e[ax] = 1
            okp = torch.ones(self.shape, dtype=torch.bool, device=self.dev)
            okm = okp.clone()
            if self.solid is not None:
                okp &= ~_roll(self.solid, [-v for v in e])
                okm &= ~_roll(self.solid, e)
            if not per[ax]:
                d = 2 - ax
                okp.select(d, self.shape[d] - 1).fill_(False)
                okm.select(d, 0).fill_(False)
            g = []
            for b in range(3):
                p, m = _roll(u[b], [-v for v in e]), _roll(u[b], e)
                z = torch.zeros_like(p)
                g.append(torch.where(okp & okm, 0.5 * (p - m),
                                     torch.where(okp, p - u[b], torch.where(okm, u[b] - m, z))))
            grad.append(g)
        div = grad[0][0] + grad[1][1] + grad[2][2]
        for q in range(self.Q):
            c = _C[q]
            cc = 0.0
            for a in range(3):
                for b in range(3):
                    if c[a] * c[b]:
                        cc = cc + c[a] * c[b] * grad[a][b]
            neq = self.W[q] * r * tau * (div - 3.0 * cc)
            if self.solid is not None:
                neq = torch.where(self.solid, torch.zeros_like(neq), neq)
            f[q] = f[q] + neq
        self.f = f

    def equilibrium(self, r, u):
        usq = 1.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
        base = (r - 1.0) - r * usq
        out = []
        for q in range(self.Q):
            cu = _dot(_C[q], u)
            out.append(self.W[q] * (base if cu is None else base + r * (3.0 * cu + 4.5 * cu * cu)))
        return out

    def moments(self, force=True):
        r = 1.0 + sum(self.f)
        m = []
        for a in range(3):
            acc = torch.zeros_like(r)
            for q in range(self.Q):
                if _C[q][a]:
                    acc = acc + _C[q][a] * self.f[q]
            m.append(acc)
        if force:
            for a in range(3):
                if self.F[a]:
                    m[a] = m[a] + 0.5 * self.F[a]
                if self.Fm is not None:
                    m[a].view(-1).index_add_(0, self.ibm["cell"], 0.5 * self.Fm[:, a])
        return r, [v / r for v in m]

    # -- rotating body: multi-direct forcing over frozen markers
    def set_body(self, pos, center, omega):
        nx, ny, nz = self.dims
        pos = np.asarray(pos)
        lo = np.floor(pos).astype(np.int64)
        ent = []
        for d in np.ndindex(2, 2, 2):
            p = lo + np.array(d)
            w = np.prod(np.maximum(1.0 - np.abs(pos - p), 0.0), axis=1)
            ok = (w > 0) & (p >= 0).all(1) & (p < np.array([nx, ny, nz])).all(1)
            cell = (p[:, 2] * ny + p[:, 1]) * nx + p[:, 0]
            m = np.flatnonzero(ok)
            m = m[~self.solid.reshape(-1).cpu().numpy()[cell[m]]]
            ent.append((m, cell[m], w[m]))
        m, cell, w = (np.concatenate([e[k] for e in ent]) for k in range(3))
        uc, pu = np.unique(cell, return_inverse=True)
        t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(self.dev)  # noqa: E731
        r = pos - np.asarray(center)
        tgt = np.stack([-omega * r[:, 1], omega * r[:, 0], 0 * r[:, 0]], 1)
        self.ibm = {"m": t(m), "u": t(pu), "w": t(w), "cell": t(uc), "target": t(tgt), "r": t(r), "M": len(pos),
                    "ksum": t(np.bincount(pu, w, len(uc))), "scale": max(1.0, float(np.sqrt((tgt ** 2).sum(1)).max()))}
        self.Fm = torch.zeros((len(uc), 3), dtype=torch.float64, device=self.dev)

    def body(self):
        b = self.ibm
        cell = b["cell"]
        fl = [p.reshape(-1)[cell] for p in self.f]
        rho = 1.0 + sum(fl)
        un = torch.stack([sum(_C[q][a] * fl[q] for q in range(self.Q) if _C[q][a]) / rho for a in range(3)], 1)
        du, spread = torch.zeros_like(un), torch.zeros_like(un)
        w = b["w"][:, None]
        mob = torch.zeros(b["M"], dtype=torch.float64, device=self.dev)
        mob.index_add_(0, b["m"], b["w"] * (b["ksum"] / rho)[b["u"]])
        torque = torch.zeros(3, dtype=torch.float64, device=self.dev)

        def interp():
            v = torch.zeros((b["M"], 3), dtype=torch.float64, device=self.dev)
            return v.index_add_(0, b["m"], w * (un + du)[b["u"]])

        um = interp()
        for _ in range(3):
            imp = torch.where(mob[:, None] == 0, torch.zeros_like(um), (b["target"] - um) / mob[:, None])
            s = torch.zeros_like(un).index_add_(0, b["u"], w * imp[b["m"]])
            spread += s
            du += s / rho[:, None]
            rep = torch.zeros_like(um).index_add_(0, b["m"], w * imp[b["m"]])
            torque -= torch.linalg.cross(b["r"], rep).sum(0)
            um = interp()
            if float((b["target"] - um).norm(dim=1).max()) / b["scale"] <= 1e-2:
                break
        self.Fc = spread
        return torque.cpu().numpy()

    # -- WALE closure: omega_plus of every cell from the state before the step
    def closure(self):
        r, u = self.moments()
        eq = self.equilibrium(r, u)
        pi = {}
        for a, b in ((0, 1), (0, 2), (1, 2)):
            acc = torch.zeros_like(r)
            for q in range(self.Q):
                if _C[q][a] * _C[q][b]:
                    acc = acc + _C[q][a] * _C[q][b] * (self.f[q] - eq[q])
            if self.Fc is not None:
                cell = self.ibm["cell"]
                g = 0.5 * (u[a].reshape(-1)[cell] * self.Fc[:, b] + u[b].reshape(-1)[cell] * self.Fc[:, a])
                acc.view(-1).index_add_(0, cell, g)
            pi[a, b] = pi[b, a] = acc * (-1.0 / ((2.0 / 3.0) * r * self.tau))
        del eq
        fd = [[None] * 3 for _ in range(3)]
        zero = torch.zeros_like(r)
        for ax in range(3):
            e = [0, 0, 0]
            e[ax] = 1
            sp, sm = _roll(self.solid, [-v for v in e]), _roll(self.solid, e)
            for k in range(3):
                p, m = _roll(u[k], [-v for v in e]), _roll(u[k], e)
                both = 0.5 * (p - m)
                lowwall = u[k] + p / 3.0  # resting wall half a cell below
                upwall = -u[k] - m / 3.0
                fd[k][ax] = torch.where(~sp & ~sm, both, torch.where(~sp & sm, lowwall, torch.where(sp & ~sm, upwall,
                                                                                                   zero)))
        g = [[fd[i][j] if i == j else pi[i, j] + 0.5 * (fd[i][j] - fd[j][i]) for j in range(3)] for i in range(3)]
        g2 = [[sum(g[i][k] * g[k][j] for k in range(3)) for j in range(3)] for i in range(3)]
        tr = (g2[0][0] + g2[1][1] + g2[2][2]) / 3.0
        s2 = sum((0.5 * (g[i][j] + g[j][i])) ** 2 for i in range(3) for j in range(3))
        sd = sum((0.5 * (g2[i][j] + g2[j][i]) - (tr if i == j else 0.0)) ** 2 for i in range(3) for j in range(3))
        den = s2 ** 2.5 + sd ** 1.25
        nut = torch.where(den > 0, 0.325 ** 2 * sd ** 1.5 / den, zero)
        self.omega = 1.0 / (3.0 * (self.nu + nut) + 0.5)

    # -- collisions
    def _lines(self, G, u, inverse):
        for ax in ((0, 1, 2) if inverse else (2, 1, 0)):
            st = (9, 3, 1)[ax]
            for k in range(27):
                if (k // st) % 3:
                    continue
                a, b, c = G[k], G[k + st], G[k + 2 * st]
                v = u[ax]
                if not inverse:
                    s, t = c + a, c - a
                    G[k] = s + b
                    G[k + st] = t - v * G[k]
                    G[k + 2 * st] = s - 2.0 * v * t + v * v * G[k]
                else:
                    m1, m2 = b + v * a, c + 2.0 * v * b + v * v * a
                    G[k], G[k + st], G[k + 2 * st] = 0.5 * (m2 - m1), a - m2, 0.5 * (m1 + m2)
        return G

    def collide(self, f, r, u, op, F):
        """Post-collision planes of f (a list of arrays of any one shape)."""
        eq = self.equilibrium(r, u)
        src = None
        if F is not None:
            uf = u[0] * F[0] + u[1] * F[1] + u[2] * F[2]
            src = []
            for q in range(self.Q):
                cu, cf = _dot(_C[q], u), _dot(_C[q], F)
                src.append(self.W[q] * (-3.0 * uf if cu is None else 3.0 * (cf - uf) + 9.0 * cu * cf))
        if self.kind == "cm":
            idx = [(_C[q][0] + 1) * 9 + (_C[q][1] + 1) * 3 + _C[q][2] + 1 for q in range(27)]
            K, S = [None] * 27, [None] * 27
            for q in range(27):
                K[idx[q]] = f[q] - eq[q]
            self._lines(K, u, False)
            if src is not None:
                for q in range(27):
                    S[idx[q]] = src[q]
                self._lines(S, u, False)
            os = torch.clamp(op * (1.0 - 0.16 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)), max=2.0)
            kb = (K[18] + K[6] + K[2]) / 3.0
            sb = (S[18] + S[6] + S[2]) / 3.0 if src is not None else 0.0
            for k in range(27):
                e = (k // 9, (k // 3) % 3, k % 3)
                sk = S[k] if src is not None else 0.0
                if sum(e) <= 1:
                    K[k] = K[k] + sk
                elif sum(e) == 2 and max(e) == 2:
                    K[k] = (1.0 - os) * (K[k] - kb) + 0.5 * sb + (1.0 - 0.5 * os) * (sk - sb)
                elif sum(e) == 2:
                    K[k] = (1.0 - os) * K[k] + (1.0 - 0.5 * os) * sk
                else:
                    K[k] = 0.5 * sk if src is not None else torch.zeros_like(r)
            self._lines(K, u, True)
            return [eq[q] + K[idx[q]] for q in range(27)]
        om = self.om
        out = [None] * self.Q
        for q in range(self.Q):
            o = _opp(q)
            if q == 0:
                out[0] = f[0] - op * (f[0] - eq[0])
                if src is not None:
                    out[0] = out[0] + (1.0 - 0.5 * op) * src[0]
                continue
            p = 0.5 * ((f[q] + f[o]) - (eq[q] + eq[o]))
            m = 0.5 * ((f[q] - f[o]) - (eq[q] - eq[o]))
            out[q] = f[q] - op * p - om * m
            if src is not None:
                out[q] = out[q] + (1.0 - 0.5 * op) * 0.5 * (src[q] + src[o]) + (1.0 - 0.5 * om) * 0.5 * (src[q] - src[o])
        return out

    def step(self):
        tq = self.body() if self.ibm is not None else None
        if self.wale:
            self.closure()
        r, u = self.moments()
        op = self.omega if self.omega is not None else self.op
        uniform = [torch.full_like(r, v) for v in self.F] if any(self.F) else None
        post = self.collide(self.f, r, u, op, uniform)
        if self.ibm is not None:  # the listed cells, with their force
            cell = self.ibm["cell"]
            at = lambda t: t.reshape(-1)[cell]  # noqa: E731
            lp = self.collide([at(p) for p in self.f], at(r), [at(v) for v in u],
                              at(op) if self.omega is not None else op, [self.Fc[:, a] for a in range(3)])
            for q in range(self.Q):
                post[q] = post[q].contiguous()
                post[q].view(-1)[cell] = lp[q]
            self.Fm = self.Fc
        new = [post[0]]
        for q in range(1, self.Q):
            t = _roll(post[q], _C[q])
            if self.links is not None:
                back = post[_opp(q)]
                if self.wall is not None:
                    cw = sum(_C[q][a] * self.wall[a] for a in range(3))
                    if torch.is_tensor(cw):
                        back = back + 6.0 * self.W[q] * r * _roll(cw, _C[q])
                t = torch.where(self.links[q], back, t)
            new.append(t)
        del post
        self.f = new
        if self.solid is not None:
            for q in range(self.Q):
                self.f[q] = self.f[q].masked_fill(self.solid, 0.0)
        if self.face:
            self._channel_faces()
        if self.hs is not None:
            self._scalar_step()
        return tq

    def _channel_faces(self):
        """Zou-He at x = 0 (velocity) and x = nx - 1 (density 1), D3Q19."""
        wet = ~self.solid
        for x, s in ((0, 1), (self.dims[0] - 1, -1)):
            g = [p[:, :, x] for p in self.f]
            flat = [q for q in range(19) if _C[q][0] == 0]
            out = [q for q in range(19) if _C[q][0] == -s]
            closure = 1.0 + sum(g[q] for q in flat) + 2.0 * sum(g[q] for q in out)
            if s > 0:
                vn = float(np.float32(INLET))
                r = closure / (1.0 - vn)
            else:
                r = torch.ones_like(closure)
                vn = 1.0 - closure
            n = [None, *(-0.5 * sum(_C[q][a] * g[q] for q in flat if _C[q][a]) for a in (1, 2))]
            for q in range(19):
                if _C[q][0] != s:
                    continue
                diag = _C[q][1] or _C[q][2]
                v = g[_opp(q)] + (1.0 / 6.0 if diag else 1.0 / 3.0) * r * vn
                for a in (1, 2):
                    if _C[q][a]:
                        v = v + _C[q][a] * n[a]
                self.f[q][:, :, x] = torch.where(wet[:, :, x], v, g[q])

    # -- passive scalar
    def set_scalar(self, conc, D, lattice):
        Qs = 7 if lattice == "d3q7" else self.Q
        k = 4.0 if Qs == 7 else 3.0
        _, u = self.moments()
        c = conc.double().reshape(self.shape)
        self.hs = {"Q": Qs, "k": k, "w": _weights(Qs), "om": float(np.float32(1.0 / (k * D + 0.5))), "c": c}
        self.hs["h"] = self._heq(c, u)

    def _heq(self, c, u):
        hs, out = self.hs, []
        for q in range(hs["Q"]):
            cu = _dot(_C[q], u)
            out.append(hs["w"][q] * c * (1.0 if cu is None else 1.0 + hs["k"] * cu))
        return out

    def _scalar_step(self):
        hs = self.hs
        _, u = self.moments()
        eq = self._heq(hs["c"], u)
        post = [h - hs["om"] * (h - e) for h, e in zip(hs["h"], eq)]
        new = []
        for q in range(hs["Q"]):
            t = post[q] if q == 0 else torch.where(self.links[q], post[_opp(q)], _roll(post[q], _C[q]))
            new.append(t.masked_fill(self.solid, 0.0))
        hs["h"], hs["c"] = new, sum(new)

    def cv(self):
        c = self.hs["c"][~self.solid]
        return float(torch.sqrt(((c - c.mean()) ** 2).mean()) / c.mean().abs())

    def fields(self):
        r, u = self.moments()
        v = [r, *u]
        if self.solid is not None:
            v = [t.masked_fill(self.solid, 1.0 if k == 0 else 0.0) for k, t in enumerate(v)]
        return dict(zip(("rho", "ux", "uy", "uz"), [t.reshape(-1) for t in v]))


def _tank_solid(n):
    g = _tank_numbers(n)
    R = 0.5 * g["T"]
    a = np.arange(n) + 0.5
    dx, dy = a[None, :] - 0.5 * n, a[:, None] - 0.5 * n
    r = np.sqrt(dx * dx + dy * dy)
    disc = r >= R
    baffle = (r < R) & (r >= R - g["bw"]) & ((np.abs(dy) <= 0.5 * g["bt"]) | (np.abs(dx) <= 0.5 * g["bt"]))
    s = np.zeros((n, n, n), bool)
    s[:] = (disc | baffle)[None]
    s[a >= g["T"]] = True
    for ax in range(3):
        for k in (0, -1):
            s[tuple(k if d == ax else slice(None) for d in range(3))] = True
    return s


def _exact_tank(n, lattice, collision, nu, seed, tip=0.05, markers="lattice", omega=None):
    g = _tank_numbers(n, tip)
    rho, u = _flow(_cube(n), seed)
    x = _Exact(lattice, _cube(n), nu, collision, _tank_solid(n), rho, u, omega=omega)
    pos, _, c = _markers(n, g, markers)
    x.set_body(pos, c, g["omega"])
    return x


def exact(case, seed):
    kind, steps, Q = case["kind"], case["steps"], case["lattice"]
    if (kind in ("tank", "cavity") and Q == 19 and case["collision"] == "cm") or _device() == "cpu":
        return None
    dims = (case["nx"], case["ny"], case["nz"])
    if kind == "batch":
        tq, out = [], {}
        for k, (n, tip, nu) in enumerate(_members(case)):
            x = _exact_tank(n, Q, case["collision"], nu, seed + 31 * k, tip)
            tq.append(np.array([x.step() for _ in range(steps)]))
            f = x.fields()
            out[f"u{k:02d}"] = [f["ux"], f["uy"], f["uz"]]
        return {"torque": np.array(tq), **out}
    if kind == "adjoint":
        x = _exact_tank(dims[0], Q, case["collision"], case["nu"], seed, omega=_omega(case, seed))
        tq = [x.step()[2] for _ in range(steps)]
        return {"J": -float(np.mean(tq[-case["window"]:])), "forward_steps": None, "dJ_domega": None, "dJ_dnu": None}
    if kind == "tank":
        x = _exact_tank(dims[0], Q, case["collision"], case["nu"], seed, markers=case["markers"])
        x.wale = case["wale"]
        scalar = case["scalar"] != "none"
        if scalar:
            x.set_scalar(_blob(dims[0], seed).masked_fill(x.solid.reshape(-1), 0.0), _diffusivity(case), case["scalar"])
        tq, cv = [], []
        for k in range(1, steps + 1):
            tq.append(x.step())
            if scalar and (k % case["cv_every"] == 0 or k == steps):
                cv.append(x.cv())
        out = {"torque": np.array(tq)}
        if scalar:
            out["cv"] = np.array(cv)
            out["conc"] = x.hs["c"].reshape(-1)
        return {**out, **x.fields()}
    if kind == "cavity":
        s = np.ones((dims[2], dims[1], dims[0]), bool)
        s[1:-1, 1:-1, 1:-1] = False
        lid = torch.zeros((dims[2], dims[1], dims[0]), dtype=torch.float64, device=_device())
        lid[-1] = float(np.float32(LID))
        rho, u = _flow(dims, seed)
        x = _Exact(Q, dims, case["nu"], case["collision"], s, rho, u, wall=(lid, 0.0, 0.0))
    elif kind == "box":
        rho, u = _flow(dims, seed)
        x = _Exact(Q, dims, case["nu"], case["collision"], None, rho, u, periodic=True, force=_force(case))
    else:
        s = np.zeros((dims[2], dims[1], dims[0]), bool)
        s[:, 0] = s[:, -1] = True
        rho, u = _flow(dims, seed, base=(INLET, 0.0, 0.0), amp=0.004)
        x = _Exact(Q, dims, case["nu"], case["collision"], s, rho, u, periodic=(False, False, True))
        x.face = True
    for _ in range(steps):
        x.step()
    return x.fields()
