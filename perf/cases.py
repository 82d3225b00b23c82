"""The work that a user of this framework has it do, as cases to be timed.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)`
one more of the same ranges; `prepare` makes what a user's program holds before
the call (grids on the GPU, solver handles, tolerances), `run` is one pass
through the public entry points, `work` says what such a pass has to read,
write and compute at least, `tolerance` how far another correct implementation
at the same precision may be off, and `exact` gives the result in 64 bits by
plain torch: the constant-coefficient Poisson problem is solved directly in the
eigenvectors of its second differences, everything else is written out.

Kinds:
  poisson  Sol_MultigridPressure3DDevice<T> / Sol_MultigridPressureMixed3DDeviceD:
           the pressure equation, from a zero guess to a relative residual.
  pcg      Sol_PCGPressure3DDevice<T>: variable coefficient, multigrid
           preconditioner.
  ns       Eqn_IncompressibleNS3D<T>: stable time step, then one step.
  grad     AdvectProjectProblem: loss and its gradient (forward and backward).
  scalar   Eqn_ScalarAdvection3D<T>: one step of a scalar in a fixed flow.
"""
import ctypes as C
import math

import numpy as np
import torch

from opencurrent_amd import _lib, adjoint, solvers
from opencurrent_amd import _types as T
from opencurrent_amd._types import BC, BCSet, Grid3DDesc, HostGrid
from opencurrent_amd.device import DeviceGrid

NP = {"f32": np.float32, "f64": np.float64}
SCHEMES = {"upwind": T.IT_FIRST_ORDER_UPWIND, "centred": T.IT_SECOND_ORDER_CENTERED,
           "upwind2": T.IT_SECOND_ORDER_UPWIND}
STEPPERS = {"euler": T.TS_FORWARD_EULER, "ab2": T.TS_ADAMS_BASHFORD2}
# share of the stable step that is taken: that rule is forward Euler's, and
# Adams-Bashforth is stable for diffusion up to half of it
STEP_SHARE = {"euler": 1.0, "ab2": .4}
# relative residual a pressure solve is asked for, by precision
REL_RESIDUAL = {"f32": 1e-5, "f64": 1e-8, "mixed": 1e-10}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: a tracer step on a small odd grid, where
        # launches and latency count
        {"name": "scalar_f32_101x67x45", "kind": "scalar", "precision": "f32", "nx": 101, "ny": 67, "nz": 45,
         "scheme": "upwind"},
        # a small pressure solve (closed box), bound by latency at every level
        {"name": "poisson_f64_64", "kind": "poisson", "precision": "f64", "nx": 64, "ny": 64, "nz": 64,
         "faces": "closed"},
        # single precision and unequal sides, fixed potential on two plates
        {"name": "poisson_f32_96x80x112", "kind": "poisson", "precision": "f32", "nx": 96, "ny": 80, "nz": 112,
         "faces": "plates"},
        # the framework's headline solve: FP32 V-cycles in FP64 refinement
        {"name": "poisson_mixed_256", "kind": "poisson", "precision": "mixed", "nx": 256, "ny": 256, "nz": 256,
         "faces": "closed"},
        # and a large plain FP64 solve (full multigrid)
        {"name": "poisson_f64_256", "kind": "poisson", "precision": "f64", "nx": 256, "ny": 256, "nz": 256,
         "faces": "plates"},
        # variable density: conjugate gradients preconditioned by multigrid
        {"name": "pcg_f64_64", "kind": "pcg", "precision": "f64", "nx": 64, "ny": 64, "nz": 64},
        # Rayleigh-Benard convection (periodic sides, no-slip plates),
        # second-order upwind, with each of the two projections
        {"name": "convection_mixed_128", "kind": "ns", "flow": "convection", "precision": "mixed", "nx": 128,
         "ny": 128, "nz": 128, "scheme": "upwind2", "stepper": "euler"},
        {"name": "convection_f64_128", "kind": "ns", "flow": "convection", "precision": "f64", "nx": 128, "ny": 128,
         "nz": 128, "scheme": "upwind2", "stepper": "euler"},
        # lock exchange in a closed no-slip box at production size,
        # anisotropic cells
        {"name": "lockex_mixed_512x512x256", "kind": "ns", "flow": "lockex", "precision": "mixed", "nx": 512,
         "ny": 512, "nz": 256, "scheme": "upwind", "stepper": "euler"},
        # a small single-precision run with the Adams-Bashforth stepper
        {"name": "lockex_f32_96x64x48", "kind": "ns", "flow": "lockex", "precision": "f32", "nx": 96, "ny": 64,
         "nz": 48, "scheme": "upwind", "stepper": "ab2"},
        # gradient of a tracer-matching loss w.r.t. the initial velocity:
        # forward and backward with checkpoints, single precision
        {"name": "grad_f32_128", "kind": "grad", "precision": "f32", "nx": 128, "ny": 128, "nz": 128, "steps": 20,
         "walls": False},
        # and in double precision in a closed box of unequal sides
        {"name": "grad_f64_80x48x64", "kind": "grad", "precision": "f64", "nx": 80, "ny": 48, "nz": 64, "steps": 6,
         "walls": True},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _sides(rng, lo, hi, most):
    """sides for a multigrid problem: a common power of two times small
    factors, as a user who wants the grid to coarsen picks them"""
    while True:
        base = 2 ** rng.randint(2, 5)
        n = [base * max(2, round(_log_uniform(rng, lo, hi) / base)) for _ in range(3)]
        # the coarsest level stays small: no factor beyond 8 is left uncoarsened
        if all(lo <= v <= hi for v in n) and max(v // base for v in n) <= 8 and n[0] * n[1] * n[2] <= most:
            return n


def draw(rng):
    kind = rng.choice(["scalar", "poisson", "poisson", "pcg", "ns", "ns", "grad"])
    if kind == "scalar":
        n = [int(_log_uniform(rng, 24, 200)) for _ in range(3)]
        return {"kind": kind, "precision": rng.choice(["f32", "f64"]), "nx": n[0], "ny": n[1], "nz": n[2],
                "scheme": rng.choice(["upwind", "centred", "upwind2"])}
    if kind == "poisson":
        n = _sides(rng, 32, 256, 256 ** 3)
        return {"kind": kind, "precision": rng.choice(["f32", "f64", "mixed"]), "nx": n[0], "ny": n[1], "nz": n[2],
                "faces": rng.choice(["closed", "plates"])}
    if kind == "pcg":
        n = _sides(rng, 32, 128, 96 ** 3)
        return {"kind": kind, "precision": "f64", "nx": n[0], "ny": n[1], "nz": n[2]}
    if kind == "ns":
        n = _sides(rng, 32, 256, 160 ** 3)
        flow = rng.choice(["convection", "lockex"])
        return {"kind": kind, "flow": flow, "precision": rng.choice(["f32", "f64", "mixed"]), "nx": n[0], "ny": n[1],
                "nz": n[2], "scheme": rng.choice(["upwind", "upwind2"]), "stepper": rng.choice(["euler", "ab2"])}
    n = _sides(rng, 32, 160, 128 ** 3)
    return {"kind": kind, "precision": rng.choice(["f32", "f64"]), "nx": n[0], "ny": n[1], "nz": n[2],
            "steps": rng.randint(4, 20), "walls": rng.random() < .5}


# ---------------------------------------------------------------- inputs

def _n(case):
    return case["nx"], case["ny"], case["nz"]


def _spacing(case):
    """cells of a unit cube's edge along the longest side; the lock exchange
    has cells half as high as wide"""
    h = 1.0 / max(_n(case))
    if case.get("flow") == "lockex":
        return 1.0, 1.0, .5
    return h, h, h


def _uniform(shape, gen):
    return 2 * torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64) - 1


def _random_mac(n, gen):
    nx, ny, nz = n
    return _uniform((nx + 1, ny, nz), gen), _uniform((nx, ny + 1, nz), gen), _uniform((nx, ny, nz + 1), gen)


def _div(u, v, w, h):
    return (u[1:] - u[:-1]) / h[0] + (v[:, 1:] - v[:, :-1]) / h[1] + (w[:, :, 1:] - w[:, :, :-1]) / h[2]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _modes(n, gen, periodic, count=4):
    """a smooth random field at the points of `n` fractions per axis: a few
    low modes; along a non-periodic axis they vanish at 0 and 1"""
    field = torch.zeros((), dtype=torch.float64, device="cuda")
    p = torch.rand((count, 7), generator=gen, device="cuda", dtype=torch.float64).cpu().numpy()
    for q in range(count):
        f = torch.full((1, 1, 1), 2 * float(p[q, 6]) - 1, dtype=torch.float64, device="cuda")
        for a in range(3):
            x = n[a].reshape([-1 if b == a else 1 for b in range(3)])
            m = 1 + int(3 * p[q, a])
            f = f * (torch.sin(2 * math.pi * (m * x + float(p[q, 3 + a]))) if periodic[a]
                     else torch.sin(math.pi * m * x))
        field = field + f
    return field


def _at(n, a, face):
    """fractions of the side at the faces (n+1) or centres (n) of axis a"""
    k = torch.arange(n[a] + 1 if face else n[a], device="cuda", dtype=torch.float64)
    return (k if face else k + .5) / n[a]


def _solenoidal(n, h, gen, periodic, speed):
    """a smooth MAC velocity with zero discrete divergence (the curl of edge
    potentials along y and z), no flow through the walls, max |u| = speed"""
    az = _modes([_at(n, 0, True), _at(n, 1, True), _at(n, 2, False)], gen, periodic)
    ay = _modes([_at(n, 0, True), _at(n, 1, False), _at(n, 2, True)], gen, (periodic[0], True, periodic[2]))
    u = (az[:, 1:] - az[:, :-1]) / h[1] - (ay[:, :, 1:] - ay[:, :, :-1]) / h[2]
    v = -(az[1:] - az[:-1]) / h[0]
    w = (ay[1:] - ay[:-1]) / h[0]
    s = speed / max(float(x.abs().max()) for x in (u, v, w))
    return u * s, v * s, w * s


def _host(x, pads, dtype):
    g = HostGrid(*x.shape, 1, 1, 1, *pads, dtype=dtype)
    g.interior()[:] = x.to(torch.float64 if dtype == np.float64 else torch.float32).cpu().numpy()
    return g


def _mac_host(u, v, w, t, dtype):
    return (_host(u, (0, 1, 1), dtype), _host(v, (1, 0, 1), dtype), _host(w, (1, 1, 0), dtype),
            _host(t, (1, 1, 1), dtype))


class _Memory:
    """a device grid's allocation; holds the solver that owns it"""

    def __init__(self, desc, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(desc.allocated),), "data": (int(desc.base), False),
                                         "typestr": "<f8" if desc.dtype == T.OCU_F64 else "<f4", "version": 2}


def _view(desc, owner):
    """a solver-owned device grid's cells as a torch tensor (no copy); the
    solver lives as long as the tensor"""
    flat = torch.as_tensor(_Memory(desc, owner), device="cuda")
    full = flat[16 - desc.gz:].view(desc.pnx, desc.pny, desc.pnz)
    cells = full[desc.gx:desc.gx + desc.nx, desc.gy:desc.gy + desc.ny, desc.gz:desc.gz + desc.nz]
    cells.owner = owner
    return cells


def _faces(case):
    b = BCSet.uniform(T.BC_NEUMANN)
    if case["faces"] == "plates":
        b.zneg = BC(T.BC_DIRICHELET, 0.0, 0.0)
        b.zpos = BC(T.BC_DIRICHELET, 0.0, 0.0)
    return b


def _poisson_rhs(case, seed):
    """the divergence of a random velocity, mean removed"""
    h = _spacing(case)
    b = _div(*_random_mac(_n(case), _generator(seed)), h)
    return b - b.mean()


def _pcg_inputs(case, seed):
    n, gen = _n(case), _generator(seed)
    b = _uniform(n, gen)
    c = [_at(n, a, False) for a in range(3)]
    coeff = 1.0 + .4 * torch.tanh(_modes(c, gen, (True, True, True)))
    return b - b.mean(), coeff


def _ns_params(case):
    p = _lib.NSParams()
    p.nx, p.ny, p.nz = _n(case)
    p.hx, p.hy, p.hz = _spacing(case)
    wall = BC(T.BC_FORCED_INFLOW_VARIABLE_SLIP, 0.0, 1.0)
    if case["flow"] == "convection":
        fb, tb = BCSet.uniform(T.BC_PERIODIC), BCSet.uniform(T.BC_PERIODIC)
        fb.zneg, fb.zpos = wall, wall
        tb.zneg, tb.zpos = BC(T.BC_DIRICHELET, 1.0, 0.0), BC(T.BC_DIRICHELET, 0.0, 0.0)
        p.vertical_direction = T.DIR_ZPOS
        p.gravity, p.bouyancy, p.viscosity, p.thermal_diffusion = -1.0, 1e5 * .71, .71, 1.0
        p.max_divergence = 1e-8 if case["precision"] != "f32" else .5
    else:
        fb = BCSet.uniform(T.BC_FORCED_INFLOW_VARIABLE_SLIP)
        for f in BCSet.FACES:
            setattr(fb, f, wall)
        tb = BCSet.uniform(T.BC_NEUMANN)
        p.vertical_direction = T.DIR_YPOS
        p.gravity, p.bouyancy, p.viscosity, p.thermal_diffusion = -1.0, 1.0, .1, .1
        p.max_divergence = 1e-8 if case["precision"] != "f32" else 1e-3
    p.cfl_factor = 1.0 if case["scheme"] == "upwind" else .5
    p.flow_bc, p.temp_bc = fb, tb
    p.advection_scheme, p.time_step = SCHEMES[case["scheme"]], STEPPERS[case["stepper"]]
    p.mixed_projection = int(case["precision"] == "mixed")
    return p


def _ns_fields(case, seed):
    """a flow in progress: a smooth divergence-free velocity and the
    temperature (convection: linear profile plus plumes and noise; lock
    exchange: heavy and light fluid with a noisy interface)"""
    n, h, gen = _n(case), _spacing(case), _generator(seed)
    centres = [_at(n, a, False) for a in range(3)]
    noise = _uniform(n, gen)
    if case["flow"] == "convection":
        periodic = (True, True, False)
        u, v, w = _solenoidal(n, h, gen, periodic, 20.0)
        t = (1 - centres[2])[None, None, :] + .1 * _modes(centres, gen, periodic) + 1e-3 * noise
    else:
        u, v, w = _solenoidal(n, h, gen, (False, False, False), .5)
        t = torch.where(centres[0] < .5, -1.0, 1.0)[:, None, None] + 1e-3 * noise
    return u, v, w, t


def _grad_inputs(case, seed):
    n, gen = _n(case), _generator(seed)
    x = [_at(n, a, False).reshape([-1 if b == a else 1 for b in range(3)]) for a in range(3)]
    c = torch.rand((2, 3), generator=gen, device="cuda", dtype=torch.float64).cpu().numpy() * .2
    blob = [sum((x[a] - .4 - float(c[q, a])) ** 2 for a in range(3)) for q in range(2)]
    phi0, target = torch.exp(-blob[0] / .02), torch.exp(-blob[1] / .02)
    return phi0, target, [m[:n[0], :n[1], :n[2]] for m in _random_mac(n, gen)]


def _grad_bcs(case):
    if not case["walls"]:
        return None, None
    wall = BCSet.uniform(T.BC_FORCED_INFLOW_VARIABLE_SLIP)
    for f in BCSet.FACES:
        setattr(wall, f, BC(T.BC_FORCED_INFLOW_VARIABLE_SLIP, 0.0, 1.0))
    return wall, BCSet.uniform(T.BC_NEUMANN)


def _grad_dt(case):
    return .25 / max(_n(case))


def _scalar_fields(case, seed):
    n, h, gen = _n(case), _spacing(case), _generator(seed)
    u, v, w = _solenoidal(n, h, gen, (True, True, True), 1.0)
    phi = .5 + .25 * _modes([_at(n, a, False) for a in range(3)], gen, (True, True, True)) + .1 * _uniform(n, gen)
    return u, v, w, phi


def prepare(case, seed):
    n, h = _n(case), _spacing(case)
    kind, prec = case["kind"], case["precision"]
    dtype = NP["f32" if prec == "f32" else "f64"]
    s = {"kind": kind}
    if kind == "poisson":
        b = _poisson_rhs(case, seed)
        rhs = DeviceGrid(*n, dtype=dtype)
        rhs.interior().copy_(b)
        make = solvers.MultigridPressureMixed3D if prec == "mixed" else solvers.MultigridPressure3D
        s["solver"] = make(rhs, *h, _faces(case))
        s["desc"] = s["solver"].pressure_desc()
        s["pressure"] = _view(s["desc"], s["solver"])
        s["tol"] = REL_RESIDUAL[prec] * float(b.square().mean().sqrt())
    elif kind == "pcg":
        b, coeff = _pcg_inputs(case, seed)
        rhs, c = DeviceGrid(*n, dtype=dtype), DeviceGrid(*n, dtype=dtype)
        rhs.interior().copy_(b)
        c.interior().copy_(coeff)
        s["solver"] = solvers.PCGPressure3D(rhs, c, *h, BCSet.uniform(T.BC_NEUMANN),
                                            preconditioner=solvers.PCGPressure3D.MULTIGRID)
        s["desc"] = s["solver"].pressure_desc()
        s["pressure"] = _view(s["desc"], s["solver"])
        s["tol"] = 1e-8 * float(b.square().sum().sqrt()) * min(h)
    elif kind == "ns":
        s["solver"] = solvers.IncompressibleNS3D(_ns_params(case), *_mac_host(*_ns_fields(case, seed), dtype))
        s["share"] = STEP_SHARE[case["stepper"]]
        s["cap"] = .1 if case["flow"] == "lockex" else math.inf
        s["views"] = {}
    elif kind == "grad":
        phi0, target, vel = _grad_inputs(case, seed)
        flow, phi_bc = _grad_bcs(case)
        p = adjoint.AdvectProjectProblem(*n, *h, dt=_grad_dt(case), steps=case["steps"], dtype=dtype,
                                         checkpoint_every=5, flow_bc=flow, phi_bc=phi_bc)
        p.set_scalars(phi0, target)
        s["problem"], s["velocity"] = p, []
        for g, m, x in zip((p.u, p.v, p.w), p.masks, vel):
            t = torch.zeros_like(g.tensor)
            _cells(t, g.desc)[:n[0], :n[1], :n[2]] = x
            t[~m] = 0
            s["velocity"].append(t)
    else:
        p = _lib.ScalarParams()
        p.nx, p.ny, p.nz = n
        p.hx, p.hy, p.hz = h
        p.bc = BCSet.uniform(T.BC_PERIODIC)
        p.advection_scheme = SCHEMES[case["scheme"]]
        s["solver"] = solvers.ScalarAdvection3D(p, *_mac_host(*_scalar_fields(case, seed), dtype))
        s["dt"] = .25 * s["solver"].get_max_stable_timestep()
        d = Grid3DDesc()
        _lib.check(_lib.host().ocu_scalar_field(s["solver"].h, 3, C.byref(d)), "field")
        s["phi"] = _view(d, s["solver"])
    return s


def _cells(flat, desc):
    return flat[16 - desc.gz:].view(desc.pnx, desc.pny, desc.pnz)[desc.gx:desc.gx + desc.nx,
                                                                  desc.gy:desc.gy + desc.ny,
                                                                  desc.gz:desc.gz + desc.nz]


# ---------------------------------------------------------------- one pass

def run(s):
    kind = s["kind"]
    if kind in ("poisson", "pcg"):
        _lib.check(_lib.hip().ocu_grid_clear(C.byref(s["desc"]), 0.0, _lib.host().ocu_get_compute_stream()), "clear")
        ok, _ = s["solver"].solve(s["tol"], 40)
        if not ok:
            raise RuntimeError("the solve did not converge")
        return s["pressure"]
    if kind == "ns":
        ns, out = s["solver"], []
        dt = min(s["share"] * ns.get_max_stable_timestep(), s["cap"])
        if not ns.advance_one_step(dt):
            raise RuntimeError("the step failed")
        for which in range(4):  # u, v, w, temperature; the step alternates between two sets of buffers
            d = ns.field_desc(which)
            if d.base not in s["views"]:
                s["views"][d.base] = _view(d, ns)
            out.append(s["views"][d.base])
        return out
    if kind == "grad":
        p = s["problem"]
        loss = p.forward(*s["velocity"])
        gu, gv, gw, gphi = p.backward()
        n = p.n
        grads = [_cells(g, x.desc)[:n[0], :n[1], :n[2]] for g, x in zip((gu, gv, gw), (p.u, p.v, p.w))]
        return [loss, *grads, gphi]
    if not s["solver"].advance_one_step(s["dt"]):
        raise RuntimeError("the step failed")
    return s["phi"]


# ---------------------------------------------------------------- least work

def work(case):
    """each input read once, each output written once; the operations of one
    application of every operator on the path (for a solve: of one residual)"""
    cells = case["nx"] * case["ny"] * case["nz"]
    kind, width = case["kind"], 4 if case["precision"] == "f32" else 8
    if kind == "poisson":
        return {"bytes": 2 * width * cells, "flops": 10 * cells}
    if kind == "pcg":
        return {"bytes": 3 * width * cells, "flops": 25 * cells}
    if kind == "ns":
        more = 8 if case["stepper"] == "ab2" else 0
        return {"bytes": (8 + more) * width * cells, "flops": 180 * cells}
    if kind == "grad":
        # the velocity, the two scalars and the four gradients; per step one
        # application of the advection and of its adjoint
        return {"bytes": 9 * width * cells, "flops": 60 * case["steps"] * cells}
    return {"bytes": 5 * width * cells, "flops": 22 * cells}


def tolerance(case):
    """about four times what the path itself is seen to be off `exact`: a
    pressure solve by the residual it was asked for, the gradient in single
    precision by its two projections' stopping rule"""
    kind, prec = case["kind"], case["precision"]
    if kind == "poisson":
        return {"rel": {"f32": 2e-4, "f64": 6e-6, "mixed": 2e-7}[prec]}
    if kind == "pcg":
        return {"rel": 1e-7}
    if kind == "ns":
        return {"rel": 2e-3 if prec == "f32" else 2e-6}
    if kind == "grad":
        return {"rel": 2e-2 if prec == "f32" else 1e-9}
    return {"rel": 2e-7 if prec == "f32" else 1e-15}


# ---------------------------------------------------------------- 64 bits

def _basis(n, kind):
    """orthonormal eigenvectors (columns) of the second difference on n cells
    and its eigenvalues times -h^2: cell-centred homogeneous Neumann or
    Dirichlet faces, or periodic"""
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    x = k[:, None] + .5
    if kind == "neumann":
        q, e = torch.cos(math.pi * x * k / n), 2 - 2 * torch.cos(math.pi * k / n)
    elif kind == "dirichlet":
        q, e = torch.sin(math.pi * x * (k + 1) / n), 2 - 2 * torch.cos(math.pi * (k + 1) / n)
    else:
        m = (k + 1) // 2  # 0, 1, 1, 2, 2, ...: cosines and sines in turn
        even = (k % 2 == 0) & (k > 0)
        q = torch.where(even, torch.sin(2 * math.pi * x * m / n), torch.cos(2 * math.pi * x * m / n))
        if n % 2 == 0:  # the highest mode: alternating signs (its cosine vanishes at the centres)
            q[:, -1] = 1 - 2 * (k % 2)
        e = 2 - 2 * torch.cos(2 * math.pi * m / n)
    return q / q.square().sum(0).sqrt(), e


def _along(q, f, axis):
    return torch.movedim(torch.tensordot(q, f, dims=([1], [axis])), 0, axis)


def _poisson(b, h, kinds):
    """p with lap p = b, mean-free where the problem is singular"""
    bases = [_basis(b.shape[a], kinds[a]) for a in range(3)]
    f = b
    for a in range(3):
        f = _along(bases[a][0].T.contiguous(), f, a)
    lam = 0
    for a in range(3):
        lam = lam - (bases[a][1] / h[a] ** 2).reshape([-1 if c == a else 1 for c in range(3)])
    singular = all(k != "dirichlet" for k in kinds)
    if singular:
        lam = lam.clone()
        lam[0, 0, 0] = 1
    f = f / lam
    if singular:
        f = f.clone()
        f[0, 0, 0] = 0
    for a in range(3):
        f = _along(bases[a][0].contiguous(), f, a)
    return f


def _take(x, a, lo, hi):
    return x.narrow(a, lo, hi - lo)


def _project(u, v, w, h, periodic):
    """the projection of a MAC velocity given at faces 0 .. n-1 of each axis
    (walls: no flow through them); returned at the same faces"""
    vel = []
    for a, x in enumerate((u, v, w)):
        if not periodic[a]:  # no flow through the low wall
            x = torch.cat([torch.zeros_like(_take(x, a, 0, 1)), _take(x, a, 1, x.shape[a])], a)
        vel.append(x)

    def high(x, a):
        first = _take(x, a, 0, 1)
        return torch.cat([_take(x, a, 1, x.shape[a]), first if periodic[a] else torch.zeros_like(first)], a)

    d = sum((high(x, a) - x) / h[a] for a, x in enumerate(vel))
    p = _poisson(d, h, ["periodic" if q else "neumann" for q in periodic])
    out = []
    for a, x in enumerate(vel):
        first = _take(p, a, p.shape[a] - 1, p.shape[a]) if periodic[a] else _take(p, a, 0, 1)
        below = torch.cat([first, _take(p, a, 0, p.shape[a] - 1)], a)
        out.append(x - (p - below) / h[a])
    return out


def _with_high(x, a, periodic):
    """append face n: the periodic copy of face 0, or the closed wall"""
    first = _take(x, a, 0, 1)
    return torch.cat([x, first if periodic else torch.zeros_like(first)], a)


def _pad(x, a, lo, hi):
    return torch.cat([lo, x, hi], a)


def _mac_ghosts(vel, periodic):
    """each component at faces 0 .. n along its own axis, with one ghost
    layer: periodic copies, or no-slip walls (tangential components change
    sign, the normal one is zero)"""
    out = []
    for c, x in enumerate(vel):
        x = _with_high(x, c, periodic[c])
        for a in range(3):
            n = x.shape[a] - (1 if a == c else 0)
            if periodic[a]:
                lo = _take(x, a, n - 1, n)
                hi = _take(x, a, 1, 2) if a == c else _take(x, a, 0, 1)
            elif a == c:
                lo = hi = torch.zeros_like(_take(x, a, 0, 1))
            else:
                lo, hi = -_take(x, a, 0, 1), -_take(x, a, n - 1, n)
            x = _pad(x, a, lo, hi)
        out.append(x)
    return out


def _cell_ghosts(t, periodic, values):
    """one ghost layer of a cell-centred field: periodic, Dirichlet (values
    per axis: low and high) or homogeneous Neumann"""
    for a in range(3):
        n = t.shape[a]
        first, last = _take(t, a, 0, 1), _take(t, a, n - 1, n)
        if periodic[a]:
            t = _pad(t, a, last, first)
        elif values[a] is not None:
            t = _pad(t, a, 2 * values[a][0] - first, 2 * values[a][1] - last)
        else:
            t = _pad(t, a, first, last)
    return t


def _face_flux(x, a, n, vel_hi, vel_lo, periodic, scheme):
    """vel_hi * (value at the high face) - vel_lo * (value at the low face)
    along axis a for the cells 0 .. n-1; x starts with one ghost layer"""
    def cells(x):  # the n cells of the other two axes
        for b in range(3):
            if b != a:
                x = x.narrow(b, 1, n[b])
        return x

    x = cells(x)
    m = n[a]
    xm, x0, xp = (_take(x, a, k, k + m) for k in (0, 1, 2))
    if scheme == "centred":
        return vel_hi * (.5 * (x0 + xp)) - vel_lo * (.5 * (xm + x0))
    if scheme == "upwind":
        return vel_hi * torch.where(vel_hi < 0, xp, x0) - vel_lo * torch.where(vel_lo < 0, x0, xm)
    # second upstream samples; past the ghost layer they wrap, or are missing
    one = _take(x, a, 0, 1)
    has_lo = torch.ones_like(x0, dtype=torch.bool)
    has_hi = torch.ones_like(x0, dtype=torch.bool)
    xmm = torch.cat([_take(x, a, m - 1, m) if periodic else one, _take(x, a, 0, m - 1)], a)
    if not periodic:
        has_lo.narrow(a, 0, 1).fill_(False)
    if x.shape[a] >= m + 3:  # the component normal to the axis: its ghost layer reaches n+1
        xpp = _take(x, a, 3, m + 3)
    else:
        xpp = torch.cat([_take(x, a, 3, m + 2), _take(x, a, 2, 3) if periodic else one], a)
        if not periodic:
            has_hi.narrow(a, m - 1, 1).fill_(False)
    hi = torch.where(vel_hi < 0, torch.where(has_hi, xp + .5 * (xp - xpp), xp), x0 + .5 * (x0 - xm))
    lo = torch.where(vel_lo < 0, x0 + .5 * (x0 - xp), torch.where(has_lo, xm + .5 * (xm - xmm), xm))
    return vel_hi * hi - vel_lo * lo


def _shifted(x, n, off):
    """x at the cells 0 .. n-1 displaced by `off`; x starts with one ghost layer"""
    return x[tuple(slice(1 + o, 1 + o + m) for o, m in zip(off, n))]


def _unit(a):
    return tuple(int(b == a) for b in range(3))


def _minus(off, a):
    return tuple(o - int(b == a) for b, o in enumerate(off))


def _laplacian(x, n, h):
    c = _shifted(x, n, (0, 0, 0))
    return sum((_shifted(x, n, _unit(a)) + _shifted(x, n, _minus((0, 0, 0), a)) - 2 * c) / h[a] ** 2 for a in range(3))


def _self_advection(vel, n, h, periodic, scheme):
    """-div(u u) at the low faces of the cells; vel with ghosts"""
    out = []
    for c in range(3):
        d = 0
        for a in range(3):
            # the advecting component at the two faces along a of the
            # control volume around this component's sample
            va = vel[a]
            lo = .5 * (_shifted(va, n, (0, 0, 0)) + _shifted(va, n, _minus((0, 0, 0), c)))
            hi = .5 * (_shifted(va, n, _unit(a)) + _shifted(va, n, _minus(_unit(a), c)))
            d = d - _face_flux(vel[c], a, n, hi, lo, periodic[a], scheme) / h[a]
        out.append(d)
    return out


def _passive_advection(vel, phi, n, h, periodic, scheme):
    """-div(u phi); vel with ghosts"""
    d = 0
    for a in range(3):
        hi, lo = _shifted(vel[a], n, _unit(a)), _shifted(vel[a], n, (0, 0, 0))
        d = d - _face_flux(phi, a, n, hi, lo, periodic[a], scheme) / h[a]
    return d


def _as_given(fields, case):
    """what the framework was handed: rounded to single precision where the
    case runs in it"""
    if case["precision"] != "f32":
        return list(fields)
    return [x.float().double() for x in fields]


def _low_faces(vel, n):
    return [x[:n[0], :n[1], :n[2]] for x in vel]


def _exact_ns(case, seed):
    n, h, p = _n(case), _spacing(case), _ns_params(case)
    u, v, w, t = _as_given(_ns_fields(case, seed), case)
    scheme = case["scheme"]
    if case["flow"] == "convection":
        periodic, values, vertical = (True, True, False), (None, None, (1.0, 0.0)), 2
    else:
        periodic, values, vertical = (False,) * 3, (None,) * 3, 1
    vel = _mac_ghosts(_low_faces((u, v, w), n), periodic)
    tg = _cell_ghosts(t, periodic, values)
    step = p.cfl_factor * min(h[a] / float(_inner(vel[a], n, a).abs().max()) for a in range(3))
    hm = min(h)
    step = min(step, hm * hm / (6 * p.thermal_diffusion), hm * hm / (6 * p.viscosity))
    step *= STEP_SHARE[case["stepper"]]
    dt = min(step, .1) if case["flow"] == "lockex" else step
    dvel = _self_advection(vel, n, h, periodic, scheme)
    for c in range(3):
        dvel[c] = dvel[c] + p.viscosity * _laplacian(vel[c], n, h)
    coef = -p.gravity * p.bouyancy
    dvel[vertical] = dvel[vertical] + .5 * coef * (t + _shifted(tg, n, _minus((0, 0, 0), vertical)))
    dt_t = _passive_advection(vel, tg, n, h, periodic, scheme) + p.thermal_diffusion * _laplacian(tg, n, h)
    t_new = t + dt * dt_t
    star = [_shifted(vel[c], n, (0, 0, 0)) + dt * dvel[c] for c in range(3)]
    del dvel, vel, tg, dt_t
    new = _project(*star, h, periodic)
    return [_with_high(x, a, periodic[a]) for a, x in enumerate(new)] + [t_new]


def _inner(x, n, a):
    """a component's own faces 0 .. n without its ghosts"""
    return x[tuple(slice(1, 1 + n[b] + int(b == a)) for b in range(3))]


def _exact_grad(case, seed):
    n, h, dt = _n(case), _spacing(case), _grad_dt(case)
    phi0, target, vel = _grad_inputs(case, seed)
    phi0, target, *vel = _as_given([phi0, target, *vel], case)
    periodic = (not case["walls"],) * 3
    phi0 = phi0.clone().requires_grad_(True)
    vel = [x.clone().requires_grad_(True) for x in vel]
    faces = [_with_high(x, a, periodic[a]) for a, x in enumerate(_project(*vel, h, periodic))]
    phi = phi0
    for _ in range(case["steps"]):
        pg = _cell_ghosts(phi, periodic, (None,) * 3)
        d = 0
        for a in range(3):
            up, lo = _take(faces[a], a, 1, n[a] + 1), _take(faces[a], a, 0, n[a])
            d = d - _face_flux(pg, a, n, up, lo, periodic[a], "centred") / h[a]
        phi = phi + dt * d
    loss = .5 * (phi - target).square().sum()
    loss.backward()
    return [float(loss.detach()), *[x.grad for x in vel], phi0.grad]


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        if case["precision"] != "mixed" and case["faces"] == "closed":
            return None  # the pressure is defined up to a constant, and only the mixed solver removes it
        b, = _as_given([_poisson_rhs(case, seed)], case)
        kinds = ["neumann", "neumann", "dirichlet" if case["faces"] == "plates" else "neumann"]
        return _poisson(b, _spacing(case), kinds)
    if kind == "pcg":
        return None  # defined up to a constant
    if kind == "ns":
        return _exact_ns(case, seed)
    if kind == "grad":
        return _exact_grad(case, seed)
    n, h = _n(case), _spacing(case)
    u, v, w, phi = _as_given(_scalar_fields(case, seed), case)
    dt = .25 * min(h[a] / float(x.abs().max()) for a, x in enumerate((u, v, w)))
    d = 0
    pg = _cell_ghosts(phi, (True,) * 3, (None,) * 3)
    for a, x in enumerate((u, v, w)):
        up, lo = _take(x, a, 1, n[a] + 1), _take(x, a, 0, n[a])
        d = d - _face_flux(pg, a, n, up, lo, True, case["scheme"]) / h[a]
    return phi + dt * d
