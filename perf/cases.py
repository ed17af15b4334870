"""Measured cases of the ensemble membrane solver: what a program that uses the package does.

A case is a tube wall (``ntheta`` x ``nz`` nodes, the workloads' aspect ratios), an ensemble of
``samples`` log-normal modulus fields (10 % coefficient of variation) and one ``kind`` of call:

* ``solve``    one coupled time step through the drop-in ``GPUSolidSolver`` (pressure from the fluid
               side, then ``Solve``): the loop of a coupled run, where every step is a call;
* ``step``     a run of ``steps`` time steps in one call, stored or matrix-free operator;
* ``updated``  the same with the stiffness and the pressure load re-formed on the moved geometry
               every ``interval`` steps;
* ``gradient`` misfit loss of a run and its gradient with respect to every element's log modulus;
* ``batch``    many uneven meshes advanced together, 99 steps in one replayed graph;
* ``stress``   per-element stresses of the current displacement;
* ``reform``   new modulus samples into an assembled system and one stiffness product with them.

``prepare`` holds what such a program holds before the call (the assembled system, the load tables,
the start state); ``run`` is the call.  Time steps follow the explicit stability bound of the mesh.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch
import torch.utils.checkpoint

DENSITY, NU, E0, COV, THICKNESS = 1.0, 0.5, 7.0e6, 0.10, 0.07
KSHEAR = 5.0 / 6.0
P_MEAN, P_AMP = 1.33e4, 0.1
BATCH_TABLE = 1 << 21       # load-table entries of a batched ensemble (its step index only grows)


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one step of a coupled run on the smallest workload mesh: a call per step, latency only
        {"name": "solve-2k-s16", "kind": "solve", "ntheta": 64, "nz": 32, "samples": 16},
        # a single deterministic wall (one sample) over a short run, no stored matrix
        {"name": "matfree-2.5k-s1", "kind": "step", "ntheta": 45, "nz": 57, "samples": 1,
         "method": "matfree", "steps": 50, "beta": 0.0, "damped": True, "tuned": False,
         "thickness_samples": False},
        # a large ensemble on a coarse wall whose thickness is sampled too; 500 is no multiple of a
        # wavefront
        {"name": "stored-2.5k-s500", "kind": "step", "ntheta": 45, "nz": 57, "samples": 500,
         "method": "stored", "steps": 20, "beta": 1.0e-7, "damped": True, "tuned": False,
         "thickness_samples": True},
        # the forward runs of the differentiation workload
        {"name": "stored-49k-s32", "kind": "step", "ntheta": 192, "nz": 256, "samples": 32,
         "method": "stored", "steps": 10, "beta": 0.0, "damped": False, "tuned": False,
         "thickness_samples": False},
        # the throughput workload, set up as the drop-in solver sets it up (timed visiting order
        # and occupancy)
        {"name": "stored-102k-s128", "kind": "step", "ntheta": 256, "nz": 400, "samples": 128,
         "method": "stored", "steps": 4, "beta": 1.0e-4, "damped": False, "tuned": True,
         "thickness_samples": False},
        # the same wall without the stored matrix
        {"name": "matfree-102k-s128", "kind": "step", "ntheta": 256, "nz": 400, "samples": 128,
         "method": "matfree", "steps": 4, "beta": 1.0e-4, "damped": False, "tuned": True,
         "thickness_samples": False},
        # the reference solver's own mode and largest published size: K(X + u) every step, 200 samples
        {"name": "updated-66k-s200", "kind": "updated", "ntheta": 206, "nz": 320, "samples": 200,
         "steps": 2, "interval": 1, "beta": 0.0, "damped": True},
        # an inverse problem's loss and gradient with the stored operator
        {"name": "gradient-49k-s32", "kind": "gradient", "ntheta": 192, "nz": 256, "samples": 32,
         "method": "stored", "steps": 40, "every": 10, "observations": 4, "beta": 0.0, "block": 0},
        # the same without a stored matrix, damped, the reverse sweep by blocks of 64 samples
        {"name": "gradient-33k-s128", "kind": "gradient", "ntheta": 128, "nz": 256, "samples": 128,
         "method": "matfree", "steps": 24, "every": 8, "observations": 3, "beta": 1.0e-6, "block": 64},
        # an uneven ensemble of walls in one launch per step
        {"name": "batch-10-uneven", "kind": "batch", "meshes": 10, "mesh_seed": 3, "max_ntheta": 256,
         "max_nz": 200, "max_samples": 256, "steps": 99},
        # stress output of a finished run
        {"name": "stress-66k-s100", "kind": "stress", "ntheta": 206, "nz": 320, "samples": 100},
        # one iteration of a sampler or optimiser: new moduli into the stored matrix, one product
        {"name": "reform-33k-s128", "kind": "reform", "ntheta": 128, "nz": 256, "samples": 128},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mesh(rng, most):
    """A wall and a sample count, over the logarithm of their ranges, N * S at most ``most``."""
    n = _log_int(rng, 600, 102400)
    ntheta = max(12, min(512, int(round(math.sqrt(n * rng.uniform(0.4, 1.6))))))
    nz = max(8, min(1000, int(round(n / ntheta))))
    s = _log_int(rng, 1, 512)
    return {"ntheta": ntheta, "nz": nz, "samples": max(1, min(s, most // (ntheta * nz)))}


def draw(rng):
    kind = rng.choice(["solve", "step", "step", "step", "updated", "gradient", "batch", "stress", "reform"])
    if kind == "solve":
        return {"kind": kind, **_mesh(rng, 1 << 20)}
    if kind == "step":
        c = {"kind": kind, **_mesh(rng, 13_000_000)}
        size = c["ntheta"] * c["nz"] * c["samples"]
        c["method"] = rng.choice(["stored", "matfree"])
        c["steps"] = max(2, min(60, 50_000_000 // size))
        c["beta"] = rng.choice([0.0, 1.0e-7, 1.0e-6])
        c["damped"] = rng.random() < 0.5
        c["tuned"] = rng.random() < 0.5
        c["thickness_samples"] = rng.random() < 0.25
        return c
    if kind == "updated":
        c = {"kind": kind, **_mesh(rng, 10_000_000)}
        c["steps"] = max(2, min(40, 26_000_000 // (c["ntheta"] * c["nz"] * c["samples"])))
        c["interval"] = rng.choice([1, 1, 5])
        c["beta"] = rng.choice([0.0, 1.0e-7])
        c["damped"] = True
        return c
    if kind == "gradient":
        c = {"kind": kind, **_mesh(rng, 4_000_000)}
        c["method"] = rng.choice(["stored", "matfree"])
        c["every"] = rng.choice([4, 6, 8])
        c["steps"] = c["every"] * rng.choice([3, 4])
        c["observations"] = rng.choice([1, 2, 3])
        c["beta"] = rng.choice([0.0, 1.0e-6])
        c["block"] = 64 if c["method"] == "matfree" and c["samples"] > 64 else 0
        return c
    if kind == "batch":
        return {"kind": kind, "meshes": rng.randint(3, 12), "mesh_seed": rng.randrange(1 << 20),
                "max_ntheta": rng.randint(32, 200), "max_nz": rng.randint(48, 200),
                "max_samples": rng.randint(8, 256), "steps": 99}
    return {"kind": kind, **_mesh(rng, 6_500_000)}


# ------------------------------------------------------------------------------- inputs of a case
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _tube(ntheta, nz, radius=0.5):
    """Nodes [N,3], triangles [E,3] and the two fixed end rings of a straight wall."""
    from cvfes_amd.mesh import tube_geometry
    return tube_geometry(ntheta, nz, radius, 12.0 * radius)


def _batch_meshes(case):
    rng = np.random.default_rng(case["mesh_seed"])
    m = case["meshes"]
    nth = rng.integers(min(32, case["max_ntheta"]), case["max_ntheta"] + 1, m)
    nzs = rng.integers(min(48, case["max_nz"]), case["max_nz"] + 1, m)
    smp = rng.integers(min(8, case["max_samples"]), case["max_samples"] + 1, m)
    return [(int(a), int(b), int(s)) for a, b, s in zip(nth, nzs, smp)]


def _inputs(case, seed):
    """The wall, its modulus samples, thickness, start displacement, time step and pressures."""
    dev = _device()
    nodes, el, bdy = _tube(case["ntheta"], case["nz"])
    n, S = nodes.shape[0], case["samples"]
    gen = torch.Generator(device=dev).manual_seed(1000 + seed)
    var = math.log(1.0 + COV * COV)
    z = torch.randn((el.shape[0], S), generator=gen, dtype=torch.float64, device=dev)
    E = E0 * torch.exp(math.sqrt(var) * z - 0.5 * var)
    rng = np.random.default_rng(seed)
    if case.get("thickness_samples"):
        thick = THICKNESS * rng.uniform(0.9, 1.1, (n, S))
    else:
        thick = np.full(n, THICKNESS)
    # a smooth start displacement: a few radial and axial modes, a thousandth of the radius
    theta = np.arctan2(nodes[:, 1], nodes[:, 0])
    along = nodes[:, 2] / nodes[:, 2].max()
    amp = 1.0e-3 * 0.5 * rng.uniform(0.5, 1.0)
    radial = amp * np.sin(math.pi * along) * (1.0 + 0.3 * np.cos(rng.integers(1, 5) * theta + rng.uniform(0, 6)))
    u0 = np.stack([radial * np.cos(theta), radial * np.sin(theta),
                   0.2 * amp * np.sin(2.0 * math.pi * along + rng.uniform(0, 6)) * np.sin(math.pi * along)], 1)
    # largest eigenvalue of M^-1 K of these walls, about 22 (c/h)^2 with the CPU lumping, and a
    # third more for the stiffest element
    h = min(2.0 * math.pi * 0.5 / case["ntheta"], 6.0 / (case["nz"] - 1))
    lam = 30.0 * E0 / (DENSITY * (1.0 - NU * NU)) / (h * h)
    beta = float(case.get("beta", 0.0))
    dt = 0.5 * (-beta + math.sqrt(beta * beta + 4.0 / lam))
    damp = 0.0
    if case.get("damped"):
        area = 2.0 * math.pi * 0.5 * 6.0 / n
        damp = 0.02 * DENSITY * THICKNESS * area / 3.0 / dt
    steps = int(case.get("steps", 1))
    p = P_MEAN * (1.0 + P_AMP * np.sin(2.0 * math.pi * np.arange(max(steps, 1)) / 37.0 + rng.uniform(0, 6)))
    return SimpleNamespace(nodes=nodes, el=el, bdy=bdy, n=n, S=S, E=E, thick=thick, u0=u0.reshape(-1),
                           dt=dt, beta=beta, damp=damp, p=p, steps=steps, gen=gen, rng=rng)


def _system(x, store):
    from cvfes_amd.system import MembraneSystem
    return MembraneSystem(x.nodes, x.el, x.bdy, x.S, vthickness=x.thick, elmE=x.E.cpu().numpy(),
                          density=DENSITY, nu=NU, store_values=store)


def _batch_inputs(case, seed):
    out = []
    for i, (a, b, s) in enumerate(_batch_meshes(case)):
        out.append(_inputs({"ntheta": a, "nz": b, "samples": s, "steps": case["steps"]}, 64 * seed + i))
    k = torch.arange(BATCH_TABLE, dtype=torch.float64, device=_device())
    return out, P_MEAN * (1.0 + P_AMP * torch.sin(2.0 * math.pi * k / 37.0))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        from cvfes_amd.batch import BatchedEnsemble
        xs, table = _batch_inputs(case, seed)
        systems = [_system(x, False) for x in xs]
        loads = [s.loads(table) for s in systems]
        ens = BatchedEnsemble(systems, loads, dts=[x.dt for x in xs], methods="matfree")
        ens.initial_state(u0s=[x.u0 for x in xs])
        ens.autotune()
        ens.initial_state(u0s=[x.u0 for x in xs])
        return {"case": case, "ens": ens}
    x = _inputs(case, seed)
    state = {"case": case, "x": x}
    zero = np.zeros(3 * x.n)
    if kind == "solve":
        from cvfes_amd.mesh import SolidMesh
        from cvfes_amd.physicsSolver import FluidSolver, SerialComm
        from cvfes_amd.physicsSolverSDampGPUs import GPUSolidSolver
        mesh = SolidMesh(x.nodes, x.el, x.bdy, x.S, thickness=THICKNESS, density=DENSITY, E=E0, v=NU,
                         elmE=x.E.cpu().numpy(), iniU=x.u0)
        config = SimpleNamespace(dt=x.dt, nSmp=x.S, time=0.0, constant_pressure=P_MEAN,
                                 pressure_waveform="sine", pressure_mean=P_MEAN,
                                 pressure_amplitude=P_AMP, pressure_period=0.8)
        comm = SerialComm()
        state["fluid"] = FluidSolver(comm, mesh, config)
        state["solid"] = GPUSolidSolver(comm, mesh, config)
        return state
    if kind == "gradient":
        from cvfes_amd.adjoint import AdjointProblem
        s = _system(x, case["method"] == "stored")
        every = x.steps // case["observations"]
        obs = list(range(every, x.steps + 1, every))
        u_obs = _observations(x, obs)
        state["problem"] = AdjointProblem(s, s.loads(x.p), x.steps, x.dt, beta=x.beta, method=case["method"],
                                          obs_steps=obs, u_obs=u_obs, checkpoint_every=case["every"],
                                          u0=x.u0, sample_block=case["block"] or None)
        state["theta"] = torch.log(x.E)
        return state
    if kind in ("stress", "reform"):
        s = _system(x, kind == "reform")
        state["u"] = _field(x)
        state["system"] = s
        if kind == "reform":
            state["theta"] = torch.log(x.E.flip(1)).contiguous()
        return state
    s = _system(x, kind == "step" and case["method"] == "stored")
    method = case.get("method", "matfree")
    if case.get("tuned"):
        tune = s.loads(np.full(40, 1.0))
        s.autotune_occupancy(tune, x.dt, beta=x.beta, damp=x.damp, method=method, steps=6)
        if method == "stored":
            s.autotune_row_order(tune, x.dt, beta=x.beta, damp=x.damp, method=method, steps=6)
    state["system"], state["load"], state["method"] = s, s.loads(x.p), method
    s.initial_state(x.u0, zero, state["load"], x.dt, beta=x.beta, damp=x.damp, method=method)
    return state


def _observations(x, obs):
    """Observed displacements: the start shape scaled along the run, with noise of each sample."""
    base = torch.as_tensor(x.u0, device=_device()).reshape(x.n, 3, 1)
    out = torch.empty((len(obs), x.n, 3, x.S), dtype=torch.float64, device=_device())
    for i, k in enumerate(obs):
        noise = torch.randn((1, 1, x.S), generator=x.gen, dtype=torch.float64, device=_device())
        out[i] = base * (1.0 - 0.05 * k / x.steps + 0.05 * noise)
    return out


def _field(x):
    """A displacement field [N,3,S]: the start shape with an amplitude and a ripple per sample."""
    dev = _device()
    base = torch.as_tensor(x.u0, device=dev).reshape(x.n, 3, 1)
    a = torch.rand((1, 1, x.S), generator=x.gen, dtype=torch.float64, device=dev)
    ripple = torch.randn((x.n, 3, x.S), generator=x.gen, dtype=torch.float64, device=dev)
    return (base * (0.5 + a) + 1.0e-5 * ripple).contiguous()


# ----------------------------------------------------------------------------------------- a pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        fluid, solid = state["fluid"], state["solid"]
        fluid.Solve(0.05, solid.dt)
        solid.RefreshContext(fluid)
        solid.Solve(0.05, solid.dt)
        return solid.system.u, solid.system.up
    if kind == "batch":
        state["ens"].run(case["steps"])
        return [s.u for s in state["ens"].systems]
    if kind == "gradient":
        from cvfes_amd.adjoint import EnsembleLoss
        theta = state["theta"].detach().requires_grad_(True)
        loss = EnsembleLoss.apply(theta, state["problem"])
        loss.sum().backward()
        return loss.detach(), theta.grad
    s = state["system"]
    if kind == "stress":
        return s.element_stress(u=state["u"])
    if kind == "reform":
        s.set_log_modulus(state["theta"])
        return s.coef, s.spmv(state["u"])
    x = state["x"]
    if kind == "updated":
        s.step_updated(state["load"], x.dt, case["interval"], beta=x.beta, damp=x.damp)
    else:
        s.step(state["load"], x.dt, beta=x.beta, damp=x.damp, method=state["method"])
    return s.u, s.up


# ------------------------------------------------------------------------- what a pass cannot avoid
def work(case):
    """Bytes: per step the operator once (upper blocks of the stored matrix, or the coefficients),
    two states in and one out, the masses; operations of the products and updates."""
    if case["kind"] == "batch":
        parts = [_step_work(a, b, s, "matfree", 0.0, False) for a, b, s in _batch_meshes(case)]
        return {"bytes": case["steps"] * sum(p[0] for p in parts), "flops": case["steps"] * sum(p[1] for p in parts)}
    a, b, S = case["ntheta"], case["nz"], case["samples"]
    n, e = a * b, 2 * a * (b - 1)
    upper = n + a * (3 * b - 2)
    state = 24.0 * n * S
    if case["kind"] == "stress":
        return {"bytes": state + 48.0 * e * S + 12.0 * e + 24.0 * n, "flops": 230.0 * e * S}
    if case["kind"] == "reform":
        return {"bytes": 2.0 * 8.0 * e * S + 2.0 * 72.0 * upper * S + 648.0 * e + 2.0 * state,
                "flops": 162.0 * e * S + 18.0 * (2 * upper - n) * S}
    if case["kind"] == "updated":
        # unique state traffic of a step; the re-formed product per element and sample
        return {"bytes": case["steps"] * (3.0 * state + 8.0 * e * S + 12.0 * e + 24.0 * n),
                "flops": case["steps"] * (3 * 150.0 * e + 20.0 * n) * S}
    steps = case.get("steps", 1)
    method = case.get("method", "stored")
    by, fl = _step_work(a, b, S, method, case.get("beta", 0.0), case.get("thickness_samples", False))
    if case["kind"] != "gradient":
        return {"bytes": steps * by, "flops": steps * fl}
    # forward run, then per step an adjoint step (the recomputed step shares its operator read) and
    # the gradient term: mu, the state and the coefficients in, the gradient in and out
    grad = 2.0 * state + 24.0 * e * S + 648.0 * e
    return {"bytes": steps * (2.0 * by + 3.0 * state + grad) + (8.0 * e + 72.0 * upper) * S,
            "flops": steps * (3.0 * fl + 190.0 * e * S)}


def _step_work(a, b, S, method, beta, thick):
    n, e = a * b, 2 * a * (b - 1)
    upper = n + a * (3 * b - 2)
    by = 72.0 * n * S + (8.0 * n * S if thick else 8.0 * n) + 25.0 * n
    if method == "stored":
        by += 72.0 * upper * S + 4.0 * (2 * upper - n)
        fl = 18.0 * (2 * upper - n) * S
    else:
        by += 8.0 * e * S + 648.0 * e + 12.0 * e
        fl = 24.0 * 9.0 * e * S
    return by, fl + (20.0 + (9.0 if beta else 0.0)) * n * S


# --------------------------------------------------------------------- the same in plain torch, 64 bits
class _Model:
    """Unit element matrices, masses, loads and products of one wall, formula by formula."""

    def __init__(self, x, E):
        dev = _device()
        t = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
        self.x, self.el = x, torch.as_tensor(x.el, device=dev)
        self.X = t(x.nodes)
        self.T, self.b, self.c, self.A = _frames(self.X[self.el].unbind(1))
        kh = _blocks(self.b, self.c, self.A)
        e = self.el.shape[0]
        full = torch.zeros((e, 9, 9), dtype=torch.float64, device=dev)
        for p in range(3):
            for q in range(3):
                full[:, 3 * p:3 * p + 3, 3 * q:3 * q + 3] = self.T.transpose(1, 2) @ kh[p][q] @ self.T
        self.khat = full
        th = t(x.thick)
        th = th[:, None] if th.ndim == 1 else th
        h = th[self.el]
        self.coef = h.mean(1) * E
        m = torch.zeros((x.n, h.shape[2]), dtype=torch.float64, device=dev)
        for p in range(3):
            w = 0.5 * h[:, p] + 0.25 * h[:, (p + 1) % 3] + 0.25 * h[:, (p + 2) % 3]
            m.index_add_(0, self.el[:, p], self.A[:, None] * w)
        self.m = (DENSITY / 9.0 * m)[:, None, :]
        f = torch.zeros((x.n, 3), dtype=torch.float64, device=dev)
        for p in range(3):
            f.index_add_(0, self.el[:, p], self.A[:, None] * self.T[:, 2] / 3.0)
        self.f1 = f[:, :, None]
        self.fixed = torch.as_tensor(x.bdy, device=dev)
        self.dof = (3 * self.el[:, :, None] + torch.arange(3, device=dev)).reshape(-1)

    def product(self, v, coef=None):
        """K v for v [N,3,S]."""
        coef = self.coef if coef is None else coef
        e = self.el.shape[0]
        ve = v[self.el].reshape(e, 9, -1)
        y = (self.khat @ ve) * coef[:, None, :]
        out = torch.zeros((3 * self.x.n, y.shape[2]), dtype=torch.float64, device=v.device)
        return out.index_add(0, self.dof, y.reshape(9 * e, -1)).reshape(v.shape)

    def start(self, p0, damp, coef=None):
        x = self.x
        S = x.S
        u = torch.as_tensor(x.u0, device=self.X.device).reshape(x.n, 3, 1).expand(x.n, 3, S).contiguous()
        a = (p0 * self.f1 - self.product(u, coef)) / self.m
        return u, u + 0.5 * x.dt * x.dt * a

    def advance(self, u, up, kx, load, damp):
        x = self.x
        force = load - kx - (damp / x.dt) * (u - up)
        new = (x.dt * x.dt * force + self.m * (2.0 * u - up)) / self.m
        return new.index_fill(0, self.fixed, 0.0)

    def step(self, u, up, p, damp, coef=None):
        kx = self.product(u + (self.x.beta / self.x.dt) * (u - up), coef)
        return self.advance(u, up, kx, p * self.f1, damp), u


def _frames(X):
    """Rows e1, e2, e3 of the element frames, b, c and areas from three corner points (last axes:
    3, or 3 x S with the components on axis 1)."""
    unit = lambda v: v / v.norm(dim=1, keepdim=True)  # noqa: E731
    e1 = unit(X[2] - X[1])
    d = X[0] - X[2]
    e2 = unit(d - (d * e1).sum(1, keepdim=True) * e1)
    e3 = torch.cross(e1, e2, dim=1)
    rel = [v - X[0] for v in X]
    lx = [(r * e1).sum(1) for r in rel]
    ly = [(r * e2).sum(1) for r in rel]
    b = [ly[1] - ly[2], ly[2] - ly[0], ly[0] - ly[1]]
    c = [lx[2] - lx[1], lx[0] - lx[2], lx[1] - lx[0]]
    A = 0.5 * (lx[1] * ly[2] - lx[2] * ly[1])
    return torch.stack([e1, e2, e3], 1), b, c, A


def _blocks(b, c, A):
    g, gk = 0.5 * (1.0 - NU), 0.5 * KSHEAR * (1.0 - NU)
    z = torch.zeros_like(A)
    scale = 1.0 / (4.0 * A * (1.0 - NU * NU))
    out = []
    for p in range(3):
        row = []
        for q in range(3):
            k = [b[p] * b[q] + g * c[p] * c[q], NU * b[p] * c[q] + g * c[p] * b[q], z,
                 NU * c[p] * b[q] + g * b[p] * c[q], c[p] * c[q] + g * b[p] * b[q], z,
                 z, z, gk * (b[p] * b[q] + c[p] * c[q])]
            row.append((torch.stack(k, 1) * scale[:, None]).reshape(-1, 3, 3))
        out.append(row)
    return out


def _moved(m, u, x):
    """(K(X + u) x, unit-pressure load on X + u) of every sample, in slices of the samples."""
    el, n = m.el, m.x.n
    kx, fl = torch.zeros_like(x), torch.zeros_like(x)
    g, gk = 0.5 * (1.0 - NU), 0.5 * KSHEAR * (1.0 - NU)
    for s in range(0, x.shape[2], 50):
        at = slice(s, s + 50)
        T, b, c, A = _frames([m.X[el[:, p]][:, :, None] + u[:, :, at][el[:, p]] for p in range(3)])
        scale = m.coef[:, at] / (4.0 * A * (1.0 - NU * NU))
        loc = [(T * x[:, :, at][el[:, q]][:, None]).sum(2) for q in range(3)]
        part, load = torch.zeros_like(x[:, :, at]), torch.zeros_like(x[:, :, at])
        for p in range(3):
            L = 0.0
            for q in range(3):
                v = loc[q]
                L = L + torch.stack([
                    (b[p] * b[q] + g * c[p] * c[q]) * v[:, 0] + (NU * b[p] * c[q] + g * c[p] * b[q]) * v[:, 1],
                    (NU * c[p] * b[q] + g * b[p] * c[q]) * v[:, 0] + (c[p] * c[q] + g * b[p] * b[q]) * v[:, 1],
                    gk * (b[p] * b[q] + c[p] * c[q]) * v[:, 2]], 1)
            part.index_add_(0, el[:, p], scale[:, None] * (T * L[:, :, None]).sum(1))
            load.index_add_(0, el[:, p], A[:, None] / 3.0 * T[:, 2])
        kx[:, :, at], fl[:, :, at] = part, load
    return kx, fl


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        xs, table = _batch_inputs(case, seed)
        p = table[:case["steps"]].tolist()
        out = []
        for x in xs:
            m = _Model(x, x.E)
            u, up = m.start(p[0], 0.0)
            for k in range(case["steps"]):
                u, up = m.step(u, up, p[k], 0.0)
            out.append(u)
        return out
    x = _inputs(case, seed)
    if kind == "solve":
        m = _Model(x, x.E)
        wave = lambda t: P_MEAN * (1.0 + P_AMP * math.sin(2.0 * math.pi * t / 0.8))  # noqa: E731
        u, up = m.start(wave(0.0), 0.0)
        return m.step(u, up, wave(0.05), 0.0)
    if kind == "stress":
        m = _Model(x, x.E)
        u = _field(x)
        loc = [(m.T[..., None] * u[m.el[:, q]][:, None]).sum(2) for q in range(3)]
        eps = [0.0] * 5
        for q in range(3):
            b, c, v = m.b[q][:, None], m.c[q][:, None], loc[q]
            for i, term in enumerate((b * v[:, 0], c * v[:, 1], c * v[:, 0] + b * v[:, 1], b * v[:, 2], c * v[:, 2])):
                eps[i] = eps[i] + term
        f = x.E / (1.0 - NU * NU) / (2.0 * m.A[:, None])
        g, gk = 0.5 * (1.0 - NU), 0.5 * KSHEAR * (1.0 - NU)
        z = torch.zeros_like(f)
        s = [f * (eps[0] + NU * eps[1]), f * (NU * eps[0] + eps[1]), f * g * eps[2], f * gk * eps[3], f * gk * eps[4]]
        L = torch.stack([s[0], s[2], s[3], s[2], s[1], s[4], s[3], s[4], z], 1).reshape(-1, 3, 3, x.S)
        G = torch.einsum("eki,ekls,elj->eijs", m.T, L, m.T)
        return torch.stack([G[:, 0, 0], G[:, 1, 1], G[:, 0, 1], G[:, 0, 2], G[:, 1, 2]], 1)
    if kind == "reform":
        m = _Model(x, x.E.flip(1))
        return m.coef, m.product(_field(x))
    if kind == "gradient":
        theta = torch.log(x.E).requires_grad_(True)
        every = x.steps // case["observations"]
        obs = list(range(every, x.steps + 1, every))
        u_obs = _observations(x, obs)
        m = _Model(x, x.E)
        coef = THICKNESS * torch.exp(theta)
        u, up = m.start(float(x.p[0]), 0.0, coef)
        loss = 0.0
        for k in range(x.steps):
            u, up = torch.utils.checkpoint.checkpoint(m.step, u, up, float(x.p[k]), 0.0, coef, use_reentrant=False)
            if k + 1 in obs:
                loss = loss + 0.5 * (u - u_obs[obs.index(k + 1)]).square().sum((0, 1))
        loss.sum().backward()
        return loss.detach(), theta.grad
    m = _Model(x, x.E)
    u, up = m.start(float(x.p[0]), x.damp)
    count, geometry = 0, None
    for k in range(x.steps):
        if kind == "step":
            u, up = m.step(u, up, float(x.p[k]), x.damp)
            continue
        if count >= case["interval"]:
            geometry, count = u, 1
        else:
            count += 1
        v = u + (x.beta / x.dt) * (u - up)
        kx, fl = _moved(m, torch.zeros_like(u) if geometry is None else geometry, v)
        u, up = m.advance(u, up, kx, float(x.p[k]) * fl, x.damp), u
    return u, up
