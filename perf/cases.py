"""The work a user of the framework has it do, as cases that can be timed and checked.

A case is one pass through the public entry points: a time step of a
``nonlinear_solver`` (``strang_timestep``), the replay of a captured step, a
gradient through a run of steps (``adjoint.evolve``) or some steps of an
``Ensemble``.  ``prepare`` builds the problem as a user's modules do (domain,
boundary conditions, parameters, initial conditions drawn from the seed),
``run`` makes one pass and returns the whole updated state, and ``exact`` gives
the same result in plain torch FP64, written from the reference's formulas
(QuazarTech/Bolt, bolt/lib/nonlinear/finite_volume/ and
bolt/src/nonrelativistic_boltzmann/).
"""
import math
import types

import torch

F64 = torch.float64
TAU = 0.05
ENSEMBLE_Q, ENSEMBLE_P = (32, 64, 128, 256), (24, 32, 48, 64)


def _step(name, q, p, recon, stepper, **more):
    c = {"name": name, "kind": "step", "q1": q[0], "q2": q[1], "p1": p[0], "p2": p[1], "p3": p[2],
         "recon_q": recon[0], "recon_p": recon[1], "stepper": stepper, "riemann": "lax-friedrichs",
         "precision": "fp64", "fields": "off", "walls": False, "species": 1}
    c.update(more)
    return c


def listed():
    return [
        # the smallest problem of the reference's tests and examples: latency and launches
        _step("1d1v_minmod", (32, 1), (32, 1, 1), ("minmod", "minmod"), "RK2",
              riemann="upwind-flux"),
        # electrons and ions in one dimension with the Poisson field: small, many launches
        _step("1d1v_two_species_es", (96, 1), (64, 1, 1), ("weno5", "minmod"), "RK2",
              fields="es", species=2),
        # Landau damping in two dimensions: p-advection with the limiter of the reference's examples
        _step("2d2v_es_minmod", (32, 32), (24, 24, 1), ("minmod", "minmod"), "RK2", fields="es"),
        # a channel between reflecting walls
        _step("2d2v_walls", (48, 40), (20, 24, 1), ("weno5", "weno5"), "SSP-RK3", walls=True,
              riemann="upwind-flux"),
        # a grid of no round numbers, fields off
        _step("2d2v_ragged_ppm", (100, 75), (30, 28, 1), ("ppm", "ppm"), "SSP-RK3"),
        # a small problem in a tight loop, captured once and replayed
        _step("2d2v_replay_fp32", (64, 64), (24, 24, 1), ("weno5", "weno5"), "SSP-RK3",
              precision="fp32-bulk", kind="replay"),
        # the benchmark's headline problem in both precisions
        _step("2d2v_weno5_fp64", (128, 128), (48, 48, 1), ("weno5", "weno5"), "SSP-RK3"),
        _step("2d2v_weno5_fp32", (128, 128), (48, 48, 1), ("weno5", "weno5"), "SSP-RK3",
              precision="fp32-bulk"),
        # the electromagnetic problem: self-consistent Yee fields, three velocity dimensions
        _step("2d3v_em_fp32", (64, 64), (24, 24, 24), ("ppm", "weno5"), "SSP-RK3",
              precision="fp32-bulk", fields="em"),
        _step("2d3v_em_fp64", (64, 64), (24, 24, 24), ("ppm", "weno5"), "SSP-RK3", fields="em"),
        # the gradient of a run with respect to its initial state and collision time
        {"name": "adjoint_2d2v", "kind": "adjoint", "q1": 64, "q2": 64, "p1": 32, "p2": 32,
         "steps": 10, "every": 5},
        # a parameter study: many uneven one-dimensional problems advanced together
        {"name": "ensemble_96", "kind": "ensemble", "members": 96, "sizes": 0, "steps": 10,
         "precision": "fp32-bulk"},
    ]


def draw(rng):
    def size(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def precision():
        return rng.choice(("fp64", "fp32-bulk"))

    kind = rng.choice(("1d", "2d2v", "lines", "es", "walls", "em", "em", "adjoint", "ensemble"))
    if kind == "1d":
        return _unnamed((size(24, 1024), 1), (size(16, 256), 1, 1),
                        (rng.choice(("minmod", "ppm", "weno5")), "minmod"),
                        "SSP-RK3", fields=rng.choice(("off", "es")),
                        species=rng.choice((1, 2)))
    if kind == "2d2v":
        r = rng.choice(("minmod", "ppm", "weno5"))
        return _unnamed((size(20, 160), size(20, 160)), (size(10, 40), size(10, 40), 1), (r, r),
                        "SSP-RK3", precision=precision())
    if kind == "lines":
        return _unnamed((rng.choice((64, 128, 256)), size(16, 128)),
                        (size(12, 40), size(12, 40), 1), ("weno5", "weno5"), "SSP-RK3",
                        precision=precision(), kind=rng.choice(("step", "replay")))
    if kind == "es":
        return _unnamed((size(16, 96), size(16, 96)), (size(12, 40), size(12, 40), 1),
                        (rng.choice(("minmod", "ppm")), rng.choice(("minmod", "weno5"))),
                        "RK2", precision=precision(), fields="es")
    if kind == "walls":
        return _unnamed((size(16, 96), size(16, 96)), (size(10, 36), size(10, 36), 1),
                        (rng.choice(("ppm", "weno5")), "weno5"), "SSP-RK3", walls=True,
                        precision=precision())
    if kind == "em":
        return _unnamed((size(16, 56), size(16, 56)), (size(10, 26), size(10, 26), size(10, 26)),
                        ("ppm", "weno5"), "SSP-RK3", fields="em", precision=precision())
    if kind == "adjoint":
        return {"kind": "adjoint", "q1": rng.choice((64, 128, size(24, 100))), "q2": size(16, 64),
                "p1": size(12, 32), "p2": size(12, 32), "steps": rng.randint(2, 8), "every": 4}
    return {"kind": "ensemble", "members": size(4, 64), "sizes": rng.randrange(1 << 20),
            "steps": rng.randint(1, 10), "precision": precision()}


def _unnamed(*a, **more):
    c = _step("", *a, **more)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# One problem, as the reference's user modules define it
# ---------------------------------------------------------------------------
MASSES, CHARGES, P_MAX = (1.0, 4.0), (-1.0, 1.0), {1: 8.0, 2: 10.0, 3: 8.0}


def _p_dim(c):
    return 3 if c["p3"] > 1 else 2 if c["p2"] > 1 else 1


def _p_max(c, s):
    return P_MAX[_p_dim(c)] * (0.5 if s else 1.0)


def _dt(c):
    """A time step inside the stability limit of every case drawn."""
    v = _p_max(c, 0)
    inv = v * c["q1"] + (v * c["q2"] if c["q2"] > 1 else 0.0)
    return min(0.3 / inv, 0.2 * TAU) if c["fields"] == "off" else min(0.3 / inv, 1e-3)


def _uniforms(seed, n):
    g = torch.Generator().manual_seed(int(seed) * 7919 + 13)
    return [float(x) for x in torch.rand(n, generator=g, dtype=F64)]


def _density(q1, q2, r, two_d):
    """1 + a few modes with amplitudes and phases from the seed (r: uniforms)."""
    n = 1.0 + 0.0 * q1
    for k, (kx, ky) in enumerate(((1, 1), (2, 1), (1, 2))):
        n = n + (1e-3 + 9e-3 * r[2 * k]) * torch.cos(
            2 * math.pi * (kx * q1 + (ky * q2 if two_d else 0.0)) + 2 * math.pi * r[2 * k + 1])
    return n


def _drifting(p1, p2, p3, n, r, m, dim):
    """Density n with a bulk velocity along p1 and a temperature along p1 that is not the
    others', so that collisions have something to relax."""
    a = 0.7 + 0.2 * r[7]
    e = a * (p1 - 0.2 * r[6]) ** 2
    if dim >= 2:
        e = e + p2 ** 2
    if dim >= 3:
        e = e + p3 ** 2
    return n * math.sqrt(a) * (m / (2 * math.pi)) ** (dim / 2) * torch.exp(-0.5 * m * e)


def _module(name, **attrs):
    m = types.ModuleType(name)
    m.__dict__.update(attrs)
    return m


def _system(c, seed, tau_value=TAU):
    from bolt_amd.physical_system import physical_system
    import bolt_amd.src.nonrelativistic_boltzmann.advection_terms as advection
    import bolt_amd.src.nonrelativistic_boltzmann.collision_operator as collisions
    import bolt_amd.src.nonrelativistic_boltzmann.moments as moments
    S, dim, two_d = c["species"], _p_dim(c), c["q2"] > 1
    r = _uniforms(seed, 16)

    def ends(n):
        top = [_p_max(c, s) if n > 1 else 0.5 for s in range(S)]
        return [-x for x in top], top

    (a1, b1), (a2, b2), (a3, b3) = ends(c["p1"]), ends(c["p2"]), ends(c["p3"])
    domain = _module("domain", q1_start=0.0, q1_end=1.0, N_q1=c["q1"], q2_start=0.0, q2_end=1.0,
                     N_q2=c["q2"], p1_start=a1, p1_end=b1, N_p1=c["p1"], p2_start=a2, p2_end=b2,
                     N_p2=c["p2"], p3_start=a3, p3_end=b3, N_p3=c["p3"], N_ghost=3)
    side = "mirror" if c["walls"] else "periodic"
    bc = _module("boundary_conditions", in_q1_left=side, in_q1_right=side,
                 in_q2_bottom="periodic", in_q2_top="periodic")

    def tau(q1, q2, p1, p2, p3):
        return tau_value * (q1 * 0 + 1) * (p1 * 0 + 1)

    params = _module(
        "params", fields_enabled=c["fields"] != "off", source_enabled=True,
        fields_type="electrodynamic" if c["fields"] == "em" else "electrostatic",
        fields_solver="fdtd" if c["fields"] == "em" else "fft",
        fields_initialize="user-defined" if c["fields"] == "em" else "fft",
        solver_method_in_q="FVM", solver_method_in_p="FVM",
        reconstruction_method_in_q=c["recon_q"], reconstruction_method_in_p=c["recon_p"],
        riemann_solver_in_q=c["riemann"], riemann_solver_in_p=c["riemann"], p_dim=dim,
        num_devices=1, mass=list(MASSES[:S]), charge=list(CHARGES[:S]), boltzmann_constant=1,
        instantaneous_collisions=False, hybrid_model_enabled=False, eps=1, mu=1, tau=tau,
        time_stepper_fvm=c["stepper"], precision=c["precision"])

    def initialize_f(q1, q2, p1, p2, p3, params):
        n = _density(q1, q2, r, two_d)
        return _drifting(p1, p2, p3, n, r, params.mass, dim)

    def initialize_E(q1, q2, params):
        return _field(q1, q2, r, 8)

    def initialize_B(q1, q2, params):
        b1_, b2_, b3_ = _field(q1, q2, r, 11)
        return (b1_, b2_, 0.5 + b3_)

    init = _module("initialize", initialize_f=initialize_f, initialize_E=initialize_E,
                   initialize_B=initialize_B)
    return physical_system(domain, bc, params, init, advection, collisions.BGK, moments)


def _field(q1, q2, r, k):
    """A uniform initial field from the seed; the currents make it vary."""
    return tuple(0.05 * (r[k + j] - 0.5) + 0.0 * q1 for j in range(3))


def _members(c):
    """The ensemble's uneven members: (N_q1, N_p) each, from the case alone."""
    r = _uniforms(c["sizes"] + 101, 2 * c["members"])
    return [(ENSEMBLE_Q[int(4 * r[2 * i])], ENSEMBLE_P[int(4 * r[2 * i + 1])])
            for i in range(c["members"])]


def _member_case(c, nq, n):
    return _unnamed((nq, 1), (n, n, 1), ("weno5", "weno5"), "SSP-RK3", precision=c["precision"])


def _member_tau(seed, i):
    return 10.0 ** (-3.0 + 3.0 * _uniforms(seed * 1009 + i, 1)[0])


def _member_dt(nq, n):
    return 0.4 / (nq * (P_MAX[2] * (1.0 - 1.0 / n)))


def _adjoint_case(c):
    return _unnamed((c["q1"], c["q2"]), (c["p1"], c["p2"], 1), ("weno5", "weno5"), "SSP-RK3")


def _weights(v1, v2, q1, q2, r):
    """The gradient of a smooth objective with respect to the final state."""
    g = 1.0 + 0.1 * v1 + 0.05 * (v1 ** 2 - 0.5 * v2 ** 2)
    return g * (1.0 + 0.3 * torch.cos(2 * math.pi * (q1 + q2 + r[9])))


# ---------------------------------------------------------------------------
# What a user's program has in hand, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    from bolt_amd.nonlinear_solver import nonlinear_solver
    kind = case["kind"]
    if kind == "ensemble":
        from bolt_amd.ensemble import Ensemble
        members = _members(case)
        solvers = [nonlinear_solver(_system(_member_case(case, nq, n), seed * 1009 + i,
                                            _member_tau(seed, i)))
                   for i, (nq, n) in enumerate(members)]
        ens = Ensemble(solvers, [_member_dt(nq, n) for nq, n in members], tuning_cache=False)
        return {"case": case, "ensemble": ens}
    if kind == "adjoint":
        c = _adjoint_case(case)
        s = nonlinear_solver(_system(c, seed))
        P = c["p1"] * c["p2"]
        v1, v2 = s.p1_center.reshape(P, 1, 1), s.p2_center.reshape(P, 1, 1)
        g = s.N_ghost
        q1 = s.q1_center[0, :, g:-g, g:-g]
        q2 = s.q2_center[0, :, g:-g, g:-g]
        f0 = s.f[:, 0, g:-g, g:-g].contiguous().requires_grad_(True)
        tau = torch.tensor(TAU, dtype=F64, device=f0.device, requires_grad=True)
        return {"case": case, "solver": s, "f0": f0, "tau": tau,
                "weights": _weights(v1, v2, q1, q2, _uniforms(seed, 16)).contiguous(),
                "dt": _dt(c)}
    s = nonlinear_solver(_system(case, seed))
    if kind == "replay":
        s.capture(1, _dt(case))
    return {"case": case, "solver": s, "dt": _dt(case)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        ens = state["ensemble"]
        ens.step(case["steps"])
        return {"f": ens.f}
    if kind == "adjoint":
        from bolt_amd import adjoint
        f = adjoint.evolve(state["solver"], state["f0"], state["tau"], case["steps"], state["dt"],
                           case["every"])
        g_f0, g_tau = torch.autograd.grad(f, [state["f0"], state["tau"]], state["weights"])
        return {"f": f.detach(), "g_f0": g_f0, "g_tau": g_tau}
    s = state["solver"]
    if kind == "replay":
        s.replay()
    else:
        s.strang_timestep(state["dt"])
    # the state's own buffers, as views (q2, q1, p), and the moments a program watches
    out = {"f": [sp.f if s._layout == 0 else sp.f.transpose(1, 2) for sp in s._spc],
           "moments": [sp.mom[:5] for sp in s._spc]}
    if case["fields"] == "em":
        out["yee"] = s.fields_solver._yee
    return out


# ---------------------------------------------------------------------------
# The same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _pad(f, dim, wall=None):
    """f with three cells more on each side of ``dim``: its periodic images, or the
    images a reflecting wall gives (``wall``: the velocity axis that is reversed)."""
    n = f.shape[dim]
    if wall is None:
        return torch.cat([f.narrow(dim, n - 3, 3), f, f.narrow(dim, 0, 3)], dim)
    lo = f.narrow(dim, 0, 3).flip(dim).flip(wall)
    hi = f.narrow(dim, n - 3, 3).flip(dim).flip(wall)
    return torch.cat([lo, f, hi], dim)


def _beta(a, b, c):
    """weno5.py:58-71."""
    s = 4 / 3 * a * a - 19 / 3 * a * b + 25 / 3 * b * b + 11 / 3 * a * c - 31 / 3 * b * c \
        + 10 / 3 * c * c
    return s + 1e-17 * (1.0 + a.abs() + b.abs() + c.abs())


def _states(y, recon):
    """(left, right) face states of the centre cell of the five-cell window y."""
    y0, y1, y2, y3, y4 = y
    if recon == "minmod":  # minmod.py:4-71
        x, c, z = 2 * (y2 - y1), 0.5 * (y3 - y1), 2 * (y3 - y2)
        m = torch.minimum(torch.minimum(x.abs(), c.abs()), z.abs())

        def sign(t):
            return torch.where(t < 0, -1.0, 1.0).to(F64)
        s = 0.25 * (sign(x) + sign(c)).abs() * (sign(x) + sign(z)) * m
        return y2 - 0.5 * s, y2 + 0.5 * s
    if recon == "ppm":  # ppm.py:57-98
        def slope(a, b, c):
            d, e, m = 0.5 * (c - a), 2 * (b - a), 2 * (c - b)
            low = torch.minimum(d.abs(), torch.minimum(e.abs(), m.abs()))
            return torch.where(e * m <= 0, torch.zeros_like(a), torch.where(d > 0, low, -low))
        s1, s2, s3 = slope(y0, y1, y2), slope(y1, y2, y3), slope(y2, y3, y4)
        lo, hi = 0.5 * (y2 + y1) - (s2 - s1) / 6, 0.5 * (y3 + y2) - (s3 - s2) / 6
        flat = (hi - y2) * (y2 - lo) <= 0
        d, e = hi - lo, 6 * (y2 - 0.5 * (hi + lo))
        over, under = d * (d - e) < 0, d * (d + e) < 0
        lo, hi = torch.where(flat, y2, lo), torch.where(flat, y2, hi)
        lo1 = torch.where(over, 3 * y2 - 2 * hi, lo)
        return lo1, torch.where(under & ~over, 3 * y2 - 2 * lo1, hi)
    b1, b2, b3 = _beta(y0, y1, y2), _beta(y1, y2, y3), _beta(y2, y3, y4)  # weno5.py:57-98
    k1, k2, k3 = 1 / (16 * b1 ** 2), 5 / (8 * b2 ** 2), 1 / (16 * b3 ** 2)
    left = (5 * k1 * (-y0 / 8 + 3 * y1 / 4 + 3 * y2 / 8) + k2 * (3 * y1 / 8 + 3 * y2 / 4 - y3 / 8)
            + k3 * (15 * y2 / 8 - 5 * y3 / 4 + 3 * y4 / 8)) / (5 * k1 + k2 + k3)
    right = (k1 * (3 * y0 / 8 - 5 * y1 / 4 + 15 * y2 / 8) + k2 * (-y1 / 8 + 3 * y2 / 4 + 3 * y3 / 8)
             + 5 * k3 * (3 * y2 / 8 + 3 * y3 / 4 - y4 / 8)) / (k1 + k2 + 5 * k3)
    return left, right


def _faces(f, dim, C, recon, wall=None):
    """Upwind states of the n + 1 faces along ``dim`` (riemann.py:46-49; for this linear
    flux the local Lax-Friedrichs flux is the same)."""
    n = f.shape[dim]
    p = _pad(f, dim, wall)
    lo, hi = _states([p.narrow(dim, k, n + 2) for k in range(5)], recon)
    return torch.where(C > 0, hi.narrow(dim, 0, n + 1), lo.narrow(dim, 1, n + 1))


class _Exact:
    """One species on its grid; f is (q2, q1, p3, p2, p1)."""

    def __init__(self, c, s, tau, dim):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.c, self.dim, self.tau, self.dev = c, dim, tau, dev
        self.m, self.e = MASSES[s], CHARGES[s]
        self.v, self.dp = [], []
        for a, n in enumerate((c["p1"], c["p2"], c["p3"])):
            top = _p_max(c, s) if n > 1 else 0.5
            d = 2 * top / n
            x = -top + (0.5 + torch.arange(n, dtype=F64, device=dev)) * d
            self.v.append(x.reshape([1, 1, 1, 1, 1][:4 - a] + [n] + [1] * a))
            self.dp.append(d)
        self.dV = self.dp[0] * self.dp[1] * self.dp[2]
        self.wall = 4 if c["walls"] else None

    def initial(self, r):
        c = self.c
        q2 = ((0.5 + torch.arange(c["q2"], dtype=F64, device=self.dev)) / c["q2"]).reshape(-1, 1)
        q1 = ((0.5 + torch.arange(c["q1"], dtype=F64, device=self.dev)) / c["q1"]).reshape(1, -1)
        n = _density(q1 + 0 * q2, q2 + 0 * q1, r, c["q2"] > 1).reshape(c["q2"], c["q1"], 1, 1, 1)
        f = _drifting(*self.v, n, r, self.m, self.dim)
        return f.expand(c["q2"], c["q1"], c["p3"], c["p2"], c["p1"]).contiguous()

    def moment(self, f, w):
        return (f * w).sum((2, 3, 4)) * self.dV

    def moments(self, f):
        v1, v2, v3 = self.v
        e = 0.5 * (v1 ** 2 + v2 ** 2 + v3 ** 2)
        return torch.stack([self.moment(f, w).reshape(-1)
                            for w in (torch.ones_like(v1), v1, v2, v3, e)])

    def maxwellian(self, f):
        """collision_operator.py:15-116."""
        n, a, b, c, E = (x.reshape(f.shape[0], f.shape[1], 1, 1, 1) for x in self.moments(f))
        m = self.m
        u = [x / (n + 1e-30) for x in (a, b, c)]
        T = (1.0 / self.dim) * (2 * (E * m) - n * m * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)) \
            / (n + 1e-30) + 1e-30
        out = n * (m / (2 * math.pi * T)) ** (self.dim / 2)
        for k in range(self.dim):
            out = out * torch.exp(-m * (self.v[k] - u[k]) ** 2 / (2 * T))
        return out

    def currents(self, f):
        s1 = _faces(f, 1, self.v[0], self.c["recon_q"]).narrow(1, 0, f.shape[1])
        s2 = _faces(f, 0, self.v[1], self.c["recon_q"]).narrow(0, 0, f.shape[0])
        return torch.stack([self.e * self.moment(s, v).reshape(-1)
                            for s, v in zip((s1, s2, f), self.v)])

    def rhs(self, f, fields=None):
        """df_dt_fvm.py:56-97, 251-323."""
        c, (v1, v2, v3) = self.c, self.v

        def along(dim, C, recon, d, wall=None):
            F = C * _faces(f, dim, C, recon, wall)
            n = f.shape[dim]
            return (F.narrow(dim, 1, n) - F.narrow(dim, 0, n)) / d
        out = (self.maxwellian(f) - f) / self.tau
        if c["q1"] > 1:
            out = out - along(1, v1, c["recon_q"], 1.0 / c["q1"], self.wall)
        if c["q2"] > 1:
            out = out - along(0, v2, c["recon_q"], 1.0 / c["q2"])
        if fields is not None:
            E1, E2, E3, B1, B2, B3 = (x.reshape(f.shape[0], f.shape[1], 1, 1, 1) for x in fields)
            k = self.e / self.m
            for a, n, C in ((0, c["p1"], k * (E1 + v2 * B3 - v3 * B2)),
                            (1, c["p2"], k * (E2 + v3 * B1 - v1 * B3)),
                            (2, c["p3"], k * (E3 + v1 * B2 - v2 * B1))):
                if n > 1:
                    out = out - along(4 - a, C, c["recon_p"], self.dp[a])
        return out


def _poisson(c, rho):
    """electrostatic/fft.py:9-78: cell-centred fields of the charge density."""
    r = rho.reshape(c["q2"], c["q1"])
    k1 = torch.fft.fftfreq(c["q1"], 1.0 / c["q1"], dtype=F64, device=r.device).reshape(1, -1)
    k2 = torch.fft.fftfreq(c["q2"], 1.0 / c["q2"], dtype=F64, device=r.device).reshape(-1, 1)
    den = 4 * math.pi ** 2 * (k1 ** 2 + k2 ** 2)
    den[0, 0] = 1.0
    phi = torch.fft.fft2(r - r.mean()) / den
    phi[0, 0] = 0
    E = [torch.fft.ifft2(-2j * math.pi * k * phi).real.reshape(-1) for k in (k1, k2)]
    z = torch.zeros_like(E[0])
    return [E[0], E[1], z, z, z, z]


def _yee_start(c, r, dev):
    """The Yee grid's initial fields at the points the reference evaluates them."""
    l2 = (torch.arange(c["q2"], dtype=F64, device=dev) / c["q2"]).reshape(-1, 1)
    l1 = (torch.arange(c["q1"], dtype=F64, device=dev) / c["q1"]).reshape(1, -1)
    l1, l2 = l1 + 0 * l2, l2 + 0 * l1
    m1, m2 = l1 + 0.5 / c["q1"], l2 + 0.5 / c["q2"]
    E = [_field(a, b, r, 8)[k] for k, (a, b) in enumerate(((l1, l2), (m1, l2), (m1, m2)))]
    B = [_field(a, b, r, 11)[k] for k, (a, b) in enumerate(((m1, l2), (l1, l2), (l1, l2)))]
    return E + [B[0], B[1], B[2] + 0.5]


def _n1(x):
    return torch.roll(x, -1, 1)


def _n2(x):
    return torch.roll(x, -1, 0)


def _centred(y):
    """fields.py:527-557."""
    E1, E2, E3, B1, B2, B3 = y
    return [0.5 * (E1 + _n1(E1)), 0.5 * (E2 + _n2(E2)), E3, 0.5 * (B1 + _n2(B1)),
            0.5 * (B2 + _n1(B2)), 0.25 * (B3 + _n2(B3) + _n1(B3) + _n1(_n2(B3)))]


def _leapfrog(c, y, J, dt):
    """fdtd_explicit.py:141-177 with unit permittivity and permeability."""
    E1, E2, E3, B1, B2, B3 = y
    J1, J2, J3 = (x.reshape(c["q2"], c["q1"]) for x in J)
    i1, i2 = float(c["q1"]), float(c["q2"])
    E1, E2, E3 = (E1 + dt * ((_n2(B3) - B3) * i2 - J1), E2 + dt * (-(_n1(B3) - B3) * i1 - J2),
                  E3 + dt * ((_n1(B2) - B2) * i1 - (_n2(B1) - B1) * i2 - J3))

    def d1(x):
        return (x - torch.roll(x, 1, 1)) * i1

    def d2(x):
        return (x - torch.roll(x, 1, 0)) * i2
    return [E1, E2, E3, B1 - dt * d2(E3), B2 + dt * d1(E3), B3 - dt * (d1(E2) - d2(E1))]


def _exact_step(c, species, fs, dt, yee=None):
    """One step of every species (fvm_operator.py:6-50); the Yee grid goes once per
    step from the currents of the first two stages."""
    def es(us):
        return _poisson(c, sum(x.e * x.moments(u)[0] for x, u in zip(species, us)))

    def all_rhs(us, fields):
        return [x.rhs(u, fields) for x, u in zip(species, us)]

    def fields_of(us):
        return es(us) if c["fields"] == "es" else None
    if c["stepper"] == "RK2":
        half = [f + 0.5 * dt * k for f, k in zip(fs, all_rhs(fs, fields_of(fs)))]
        return [f + dt * k for f, k in zip(fs, all_rhs(half, fields_of(half)))], yee
    F1 = F2 = F3 = None
    if yee is not None:
        F1 = _centred(yee)
    elif c["fields"] == "es":
        F1 = es(fs)
    u1 = [f + dt * k for f, k in zip(fs, all_rhs(fs, F1))]
    if yee is not None:
        J = 0.5 * sum(x.currents(f) + x.currents(u) for x, f, u in zip(species, fs, u1))
        yee = _leapfrog(c, yee, J, dt)
        new = _centred(yee)
        F2 = new[:3] + [0.5 * (a + b) for a, b in zip(F1[3:], new[3:])]
        F3 = [0.5 * (a + b) for a, b in zip(F1[:3], new[:3])] + F1[3:]
    elif c["fields"] == "es":
        F2 = es(u1)
    u2 = [0.75 * f + 0.25 * (u + dt * k) for f, u, k in zip(fs, u1, all_rhs(u1, F2))]
    if yee is None and c["fields"] == "es":
        F3 = es(u2)
    return [f / 3 + 2 / 3 * (u + dt * k) for f, u, k in zip(fs, u2, all_rhs(u2, F3))], yee


def exact(case, seed):
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    if case["kind"] == "ensemble":
        out = []
        for i, (nq, n) in enumerate(_members(case)):
            c = _member_case(case, nq, n)
            x = _Exact(c, 0, _member_tau(seed, i), 2)
            f = [x.initial(_uniforms(seed * 1009 + i, 16))]
            for _ in range(case["steps"]):
                f, _ = _exact_step(c, [x], f, _member_dt(nq, n))
            out.append(f[0].reshape(nq, n * n).t().reshape(-1))
        return {"f": torch.cat(out)}
    r = _uniforms(seed, 16)
    species = [_Exact(case, s, TAU, _p_dim(case)) for s in range(case["species"])]
    fs = [x.initial(r) for x in species]
    yee = _yee_start(case, r, species[0].dev) if case["fields"] == "em" else None
    fs, yee = _exact_step(case, species, fs, _dt(case), yee)
    out = {"f": [f.reshape(case["q2"], case["q1"], -1) for f in fs],
           "moments": [x.moments(f) for x, f in zip(species, fs)]}
    if yee is not None:
        out["yee"] = torch.stack([y.reshape(-1) for y in yee])
    return out


def _exact_adjoint(case, seed):
    from torch.utils.checkpoint import checkpoint
    c, r = _adjoint_case(case), _uniforms(seed, 16)
    x = _Exact(c, 0, TAU, 2)
    f0 = x.initial(r).requires_grad_(True)
    tau = torch.tensor(TAU, dtype=F64, device=f0.device, requires_grad=True)
    dt = _dt(c)

    def step(f, t):
        x.tau = t
        return _exact_step(c, [x], [f], dt)[0][0]
    f = f0
    for _ in range(case["steps"]):
        f = checkpoint(step, f, tau, use_reentrant=False)
    P, q = c["p1"] * c["p2"], (c["q2"], c["q1"])
    v1, v2 = (v.expand(1, 1, 1, c["p2"], c["p1"]).reshape(1, 1, P) for v in x.v[:2])
    q2 = ((0.5 + torch.arange(q[0], dtype=F64, device=f0.device)) / q[0]).reshape(-1, 1, 1)
    q1 = ((0.5 + torch.arange(q[1], dtype=F64, device=f0.device)) / q[1]).reshape(1, -1, 1)
    w = _weights(v1, v2, q1, q2, r).reshape(f.shape)
    g_f0, g_tau = torch.autograd.grad(f, [f0, tau], w)
    return {"f": f.detach().reshape(*q, P).permute(2, 1, 0),
            "g_f0": g_f0.reshape(*q, P).permute(2, 1, 0), "g_tau": g_tau}


# ---------------------------------------------------------------------------
# What one pass cannot do without
# ---------------------------------------------------------------------------
# Operations of one face of a cell along one axis: indicator or slopes, state, flux difference.
FACE = {"minmod": 18, "ppm": 45, "weno5": 50}


def _step_work(c):
    """A stage needs the moments of its whole input, so its output is written and read
    again: every stage reads its inputs once and writes its output once (RK2: 5 passes
    over f, SSP-RK3: 8)."""
    cells = c["q1"] * c["q2"] * c["p1"] * c["p2"] * c["p3"] * c["species"]
    stages, passes = (2, 5) if c["stepper"] == "RK2" else (3, 8)
    per = 22 + FACE[c["recon_q"]] * ((c["q1"] > 1) + (c["q2"] > 1))
    if c["fields"] != "off":
        per += FACE[c["recon_p"]] * ((c["p1"] > 1) + (c["p2"] > 1) + (c["p3"] > 1))
    size = 8 if c["precision"] == "fp64" else 4
    return passes * cells * size, stages * cells * per


def work(case):
    if case["kind"] == "ensemble":
        parts = [_step_work(_member_case(case, nq, n)) for nq, n in _members(case)]
        return {"bytes": case["steps"] * sum(p[0] for p in parts),
                "flops": case["steps"] * sum(p[1] for p in parts)}
    if case["kind"] == "adjoint":
        # forward, the stages again from the checkpoints, and the stage adjoints, which read
        # the state, the adjoint and its bases and cost about three forward stages
        b, f = _step_work(_adjoint_case(case))
        return {"bytes": case["steps"] * (2 * b + 11 * b // 8), "flops": case["steps"] * 5 * f}
    b, f = _step_work(case)
    return {"bytes": b, "flops": f}
