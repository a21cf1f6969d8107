"""What a user of this engine has it do, as cases whose passes can be timed.

Every case is a run: an initial state on a mesh is advanced a few RK4 steps
through `Solver.rk4_integrate` (or `Solver.dt_from_cfl` + `Solver.rk4_step`,
or `Batch.rk4`), as the benchmark, the tests and a program that replaces the
reference's `RK_integration` do it.  A pass first copies the initial state
into the state it advances, so that every pass does the same work.

`listed()` holds the benchmark's own workloads (Sod tube, vortex, shock-bubble
in its plain, sensor-gated and learned forms, the 1D ensemble) and the sizes
and options beside them: a small grid where launches count, grids whose sides
no tile divides, a mesh read from a Gmsh file, orders 1 and 3, the Rusanov
flux, the stiffened gas.  `draw()` gives more of the same ranges.

`exact()` is the same scheme in plain 64-bit torch on the tensor-product grid:
nodes [..., y element, x element, y node, x node], written from the equations
alone.  It covers the runs without a sensor or indicator (those decide by
thresholds and have no closed value); nothing of it uses the engine.
"""
from __future__ import annotations

import functools
import math
import os
import random
import tempfile

import numpy as np
import torch

import dg_amd
from dg_amd import Batch, Config, Indicator, Mesh, Solver

PHYSICS = {"single": 0, "two-fluid": 1, "passive": 2, "stiffened": 3}
FLUX = {"rusanov": 0, "roe": 1}
LIMITER = {"none": 0, "hr": 1, "hri": 3, "learned": 8}
PERIODIC, FARFIELD, REFLECTIVE = dg_amd.PERIODIC, dg_amd.FARFIELD, dg_amd.REFLECTIVE
THRESHOLDS = [0.01, 0.01, 0.01]  # the sensor's contact, shock and interface thresholds
GAMMA = 1.4


def _case(name, problem, nx, ny=1, order=2, physics="single", flux="roe", limiter="none", control="fixed", cfl=0.4,
          steps=4, precision="fp64", source="built"):
    c = dict(problem=problem, nx=nx, ny=ny, order=order, physics=physics, flux=flux, limiter=limiter, control=control,
             cfl=cfl, steps=steps, precision=precision, source=source)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: a 1D shock tube to which the launches of a step are everything
        _case("sod_1000_p2", "tube", 1000, flux="rusanov", limiter="hr", control="cfl", steps=20),
        # a 1D two-fluid tube of high order; no tile width divides its element count
        _case("tube_4001_p3_twofluid", "tube", 4001, order=3, physics="two-fluid", limiter="hr", control="cfl", steps=10),
        # a small 2D run driven step by step by the user's own loop
        _case("vortex_64_p2_loop", "vortex", 64, 64, control="loop", cfl=0.3, steps=10),
        # smooth flow at the benchmark's size, no limiter
        _case("vortex_512_p2", "vortex", 512, 512, cfl=0.3),
        # the same with a round number of elements that the tiles do not divide, CFL steps, the cheaper flux
        _case("vortex_500_p2_rusanov", "vortex", 500, 500, flux="rusanov", control="cfl", cfl=0.3),
        # third order in 2D
        _case("vortex_256_p3", "vortex", 256, 256, order=3, cfl=0.3),
        # the shock-bubble benchmark in its plain form: the largest ordinary run
        _case("bubble_1024x512_p2_hr", "bubble", 1024, 512, physics="two-fluid", limiter="hr"),
        # and as bench.py runs it by default: FP32 contractions, limiting where the trained indicator flags
        _case("bubble_1024x512_p2_learned", "bubble", 1024, 512, physics="two-fluid", limiter="learned",
              precision="fp32mfma"),
        # and gated by the reference's sensor
        _case("bubble_1024x512_p2_hri", "bubble", 1024, 512, physics="two-fluid", limiter="hri"),
        # first order on a mesh from a Gmsh file, the reference's own mesh input
        _case("bubble_450x225_p1_gmsh", "bubble", 450, 225, order=1, physics="two-fluid", limiter="hr", control="cfl",
              source="gmsh"),
        # the widest state (6 fields) of the stiffened gas, limited
        _case("stiffened_512x256_p2_hr", "wave", 512, 256, physics="stiffened", limiter="hr", control="cfl"),
        # the ensemble: nx problems with ny elements at most, orders 1 to 3
        _case("ensemble_256", "ensemble", 256, 4000, order=0, physics="two-fluid", limiter="hr", control="cfl", steps=10),
    ]


def draw(rng):
    def size(lo, hi):  # uniform in the logarithm; multiples of the tiles and ragged ones alike
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return max(lo, n // 8 * 8) if rng.random() < 0.4 else n

    kind = rng.choice(["tube", "tube", "vortex", "vortex", "bubble", "bubble", "bubble", "wave", "ensemble"])
    order, flux = rng.choice([1, 2, 2, 3]), rng.choice(["roe", "rusanov"])
    steps = rng.randrange(3, 7)
    if kind == "tube":
        return _case(None, "tube", size(100, 16000), 1, order, rng.choice(["single", "two-fluid", "passive", "stiffened"]), flux,
                     "hr", "cfl", 0.4, 3 * steps)
    if kind == "vortex":
        return _case(None, "vortex", size(32, 448), size(32, 448), order, "single", flux, "none",
                     rng.choice(["fixed", "cfl", "loop"]), 0.3, steps)
    if kind == "bubble":
        nx = size(64, 640)
        ny = max(32, nx // 2 + rng.choice([0, 0, 1, 3]))
        lim = rng.choice(["hr", "hr", "hri"])
        return _case(None, "bubble", nx, ny, order, "two-fluid", flux, lim, rng.choice(["fixed", "cfl"]), 0.4, steps)
    if kind == "wave":
        return _case(None, "wave", size(48, 384), size(48, 384), order, rng.choice(["two-fluid", "passive", "stiffened"]),
                     flux, rng.choice(["hr", "none"]), "cfl", 0.3, steps)
    return _case(None, "ensemble", rng.randrange(16, 193), size(400, 4000), 0, "two-fluid", "roe", "hr", "cfl", 0.4,
                 2 * steps)


# ------------------------------------------------------------------ geometry
def _lattice_1d(p):
    """Lattice positions of the 1D element's nodes: the ends, then the interior."""
    return [0, p] + list(range(1, p))


def _lattice_2d(p):
    """Lattice positions (x, y) of the 2D element's nodes in Gmsh order."""
    def quad(lo, hi):
        if lo == hi:
            return [(lo, lo)]
        out = [(lo, lo), (hi, lo), (hi, hi), (lo, hi)]
        m = hi - lo
        for (x0, y0), (x1, y1) in ((out[0], out[1]), (out[1], out[2]), (out[2], out[3]), (out[3], out[0])):
            out += [(x0 + i * (x1 - x0) // m, y0 + i * (y1 - y0) // m) for i in range(1, m)]
        return out + (quad(lo + 1, hi - 1) if m > 1 else [])
    return quad(0, p)


def _flat_nodes(case, order):
    if case["problem"] in ("tube", "ensemble"):
        return _lattice_1d(order)
    return [y * (order + 1) + x for x, y in _lattice_2d(order)]


def _pack(fields, nodes):
    """[F, ey, ex, b, a] -> the engine's U[(e*N_F + f)*N_s + i]."""
    f = fields.shape[0]
    u = fields.reshape(f, fields.shape[1] * fields.shape[2], -1)[:, :, nodes]
    return u.permute(1, 0, 2).contiguous().reshape(-1)


def _unpack(u, n_f, ey, ex, order, nodes):
    v = u.reshape(ey * ex, n_f, len(nodes)).permute(1, 0, 2)
    out = torch.empty_like(v)
    out[:, :, nodes] = v
    one_d = len(nodes) == order + 1
    return out.reshape(n_f, ey, ex, 1 if one_d else order + 1, order + 1)


def _box(case):
    """(x0, x1, y0, y1) and the boundary tags (left, right, bottom, top)."""
    if case["problem"] in ("tube", "ensemble"):
        return (-1.0, 1.0, 0.0, 0.0), (FARFIELD, FARFIELD)
    if case["problem"] == "vortex":
        return (0.0, 10.0, 0.0, 10.0), (PERIODIC,) * 4
    if case["problem"] == "wave":
        return (0.0, 2.0, 0.0, 1.0), (PERIODIC,) * 4
    return (0.0, 2.0, 0.0, 1.0), (FARFIELD, FARFIELD, REFLECTIVE, REFLECTIVE)


def _cell(case):
    (x0, x1, y0, y1), _ = _box(case)
    hx = (x1 - x0) / case["nx"]
    return hx, (y1 - y0) / case["ny"] if y1 > y0 else hx


def _node_coordinates(case, dev):
    p, (x0, _, y0, _) = case["order"], _box(case)[0]
    hx, hy = _cell(case)
    one_d = case["problem"] == "tube"
    k = torch.arange(p + 1, device=dev, dtype=torch.float64)
    ix = torch.arange(case["nx"], device=dev, dtype=torch.float64)
    iy = torch.arange(case["ny"], device=dev, dtype=torch.float64)
    x = (x0 + (ix[:, None] * p + k[None]) * (hx / p))[None, :, None, :]
    y = torch.zeros(1, 1, 1, 1, device=dev, dtype=torch.float64) if one_d else \
        (y0 + (iy[:, None] * p + k[None]) * (hy / p))[:, None, :, None]
    return torch.broadcast_tensors(x, y)


# ------------------------------------------------------------- initial states
def _conserved(physics, rho, vel, p, gamma, extra):
    """[F, ...] of the physics from primitive values; extra: pinf, or (phic, phinc)."""
    ke = 0.5 * rho * sum(v * v for v in vel)
    head = [rho] + [rho * v for v in vel]
    if physics == "stiffened":
        beta = gamma * extra / (gamma - 1)
        tail = [p / (gamma - 1) + beta + ke, 1 / (gamma - 1), beta]
    elif physics == "two-fluid":
        tail = [p / (gamma - 1) + ke, 1 / (gamma - 1)]
    elif physics == "passive":
        tail = [p / (gamma - 1) + ke, rho * extra[0], extra[1]]
    else:
        tail = [p / (gamma - 1) + ke]
    return torch.stack(torch.broadcast_tensors(*(head + tail)))


def _two_sides(case, rng, left):
    """A shock tube of moderate strength: one state on each side of the diaphragm."""
    one = torch.ones(left.shape, dtype=torch.float64, device=left.device)

    def side(lo, hi, *right):
        return torch.where(left, rng.uniform(lo, hi) * one, rng.uniform(*(right or (lo, hi))) * one)
    rho, p = side(0.8, 1.2, 0.125, 0.3), side(0.8, 1.2, 0.1, 0.3)
    u = side(-0.2, 0.2)
    gamma = side(1.2, 1.67) if case["physics"] in ("two-fluid", "stiffened") else torch.full_like(rho, GAMMA)
    extra = side(0.0, 1.0) if case["physics"] == "stiffened" else (side(0.0, 1.0), side(0.0, 1.0))
    return _conserved(case["physics"], rho, [u], p, gamma, extra)


def _initial(case, seed, dev):
    """[F, ey, ex, b, a] of the case's problem, varied by the seed."""
    rng = random.Random(seed)
    x, y = _node_coordinates(case, dev)
    if case["problem"] == "tube":  # the side is chosen by the element's first node
        return _two_sides(case, rng, (x[..., :1] < rng.uniform(-0.1, 0.1)).expand_as(x))
    if case["problem"] == "vortex":  # isentropic vortex in a (1, 1) stream
        b, xc, yc = rng.uniform(4.0, 5.0), rng.uniform(4.0, 6.0), rng.uniform(4.0, 6.0)
        dx, dy = torch.remainder(x - xc + 5.0, 10.0) - 5.0, torch.remainder(y - yc + 5.0, 10.0) - 5.0
        ex = torch.exp(0.5 * (1.0 - dx * dx - dy * dy))
        t = 1.0 - (GAMMA - 1) * b * b / (8 * GAMMA * math.pi ** 2) * ex * ex
        rho = t ** (1.0 / (GAMMA - 1))
        return _conserved("single", rho, [1.0 - b / (2 * math.pi) * ex * dy, 1.0 + b / (2 * math.pi) * ex * dx], rho ** GAMMA,
                          GAMMA, None)
    if case["problem"] == "bubble":  # a planar shock moving into a light gas bubble, by element centre
        xm, ym = 0.5 * (x[..., :1] + x[..., -1:]).expand_as(x), 0.5 * (y[..., :1, :] + y[..., -1:, :]).expand_as(y)
        m2 = rng.uniform(1.2, 1.3) ** 2
        xs, rb, rho_b = rng.uniform(0.08, 0.22), rng.uniform(0.22, 0.27), rng.uniform(0.138, 0.2)
        p2, rho2 = 1.0 + 2 * GAMMA / (GAMMA + 1) * (m2 - 1), (GAMMA + 1) * m2 / ((GAMMA - 1) * m2 + 2)
        shocked = xm < xs
        bubble = ((xm - 0.5) ** 2 + (ym - 0.5) ** 2 < rb * rb) & ~shocked
        one = torch.ones_like(x)
        rho = torch.where(shocked, rho2 * one, torch.where(bubble, rho_b * one, one))
        u = torch.where(shocked, math.sqrt(m2 * GAMMA) * (1 - 1 / rho2) * one, 0 * one)
        return _conserved("two-fluid", rho, [u, 0 * one], torch.where(shocked, p2 * one, one),
                          torch.where(bubble, 1.667 * one, GAMMA * one), None)

    def wave():  # "wave": smooth flow in which every field varies
        a, b, c, d = (rng.uniform(-1, 1) for _ in range(4))
        return a * torch.sin(math.pi * x + 2 * math.pi * c) + b * torch.cos(2 * math.pi * y + 2 * math.pi * d) + \
            0.3 * torch.sin(2 * math.pi * (x + y))
    rho, p = 1.0 + 0.15 * wave(), 1.0 + 0.15 * wave()
    u, v = 0.1 * wave() + rng.uniform(-0.3, 0.3), 0.1 * wave() + rng.uniform(-0.3, 0.3)
    gamma = 1.4 + 0.1 * (1 + torch.tanh(wave())) if case["physics"] in ("two-fluid", "stiffened") else torch.full_like(x, GAMMA)
    extra = 0.5 + 0.1 * wave() if case["physics"] == "stiffened" else (0.5 + 0.1 * wave(), 0.5 + 0.1 * wave())
    return _conserved(case["physics"], rho, [u, v], p, gamma, extra)


def _ensemble_spec(case):
    """Element counts uniform in [max/20, max], orders uniform in 1..3: the same for every seed."""
    rng = random.Random(20261202)
    ne = [rng.randint(max(2, case["ny"] // 20), case["ny"]) for _ in range(case["nx"])]
    return ne, [rng.randint(1, 3) for _ in range(case["nx"])]


def _ensemble_state(case, k, ne, p, seed, dev):
    one = dict(case, problem="tube", nx=ne, ny=1, order=p)
    x, _ = _node_coordinates(one, dev)
    return _two_sides(one, random.Random(seed * 1000 + k), (x[..., :1] < 1e-12).expand_as(x))


# ------------------------------------------------------------------ the engine
@functools.lru_cache(maxsize=4)
def _mesh(nx, ny, order, n_f, box, bc, source):
    """A user's program builds or reads its mesh once; it does not depend on the seed."""
    mesh = Mesh(1 if len(bc) == 2 else 2, order, nx, ny, *box, bc=bc, nfields=n_f)
    if source == "gmsh":
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "mesh.msh")
            mesh.write_gmsh(path)
            mesh = Mesh.from_gmsh(path, nfields=n_f)
    return mesh


def _solver(case):
    box, bc = _box(case)
    cfg = Config(1 if len(bc) == 2 else 2, case["order"], PHYSICS[case["physics"]], FLUX[case["flux"]])
    solver = Solver(cfg, _mesh(case["nx"], case["ny"], case["order"], cfg.nfields, box, bc, case["source"]))
    if case["limiter"] in ("hri", "learned"):
        solver.set_sensor_thresholds(THRESHOLDS)
    if case["limiter"] == "learned":
        solver.set_indicator(*_indicator())
    if case["precision"] == "fp32mfma":
        solver.set_precision(1)
    return solver


@functools.lru_cache(maxsize=1)
def _indicator():
    """The trained network and its threshold: features of 64 shock-bubble and
    smooth states, labelled by the sensor, learned once and kept, as a user
    keeps trained weights."""
    small = _case(None, "bubble", 96, 48, physics="two-fluid", limiter="hri")
    solver, net = _solver(small), Indicator(seed=3)
    solver.set_indicator(net, 0.0)
    n = small["nx"] * small["ny"]
    xs, ys = [], []
    for k in range(64):
        c = dict(small, problem="wave") if k % 4 == 3 else small
        u = _pack(_initial(c, 7000 + k, "cuda"), _flat_nodes(c, 2))
        x = torch.zeros(n, 64, dtype=torch.float32, device="cuda")
        s = torch.zeros(n, dtype=torch.int32, device="cuda")
        solver.features(u, x)
        solver.sensing(u, s)
        xs.append(x)
        ys.append((s != 0).float())
    x, y = torch.cat(xs), torch.cat(ys)
    net.train(x, y, epochs=30, batch=1024, lr=2e-3, pos_weight=float((y.numel() - y.sum()) / y.sum()), seed=3)
    torch.cuda.synchronize()
    return net, 0.0  # the network's own decision; the shock guard holds every shock cell


def _cfl_length(case):
    return case["cfl"] * min(_cell(case)) / (2 * case["order"] + 1)


def prepare(case, seed):
    dev = "cuda"
    if case["problem"] == "ensemble":
        ne, orders = _ensemble_spec(case)
        batch = Batch(Config(1, 1, PHYSICS[case["physics"]], FLUX[case["flux"]]), ne, orders)
        batch.set_block_sizes([128])  # what autotune() chooses for ensembles of these sizes
        u0 = torch.cat([_pack(_ensemble_state(case, k, n, p, seed, dev), _lattice_1d(p)) for k, (n, p) in enumerate(zip(ne, orders))])
        return {"case": case, "batch": batch, "U0": u0, "U": torch.empty_like(u0),
                "T": torch.zeros(len(ne), dtype=torch.float64, device=dev),
                "status": torch.zeros(len(ne), dtype=torch.int32, device=dev)}
    solver = _solver(case)
    u0 = _pack(_initial(case, seed, dev), _flat_nodes(case, case["order"]))
    state = {"case": case, "solver": solver, "U0": u0, "U": torch.empty_like(u0), "cfl": _cfl_length(case),
             "limiter": LIMITER[case["limiter"]], "dt_dev": torch.zeros(1, dtype=torch.float64, device=dev)}
    if case["control"] == "fixed":  # the step of the initial state, kept for the run
        solver.dt_from_cfl(u0, state["cfl"], state["dt_dev"])
        torch.cuda.synchronize()
        state["dt"] = float(state["dt_dev"].item())
    return state


def run(state):
    case, u = state["case"], state["U"]
    stream = torch.cuda.current_stream()
    u.copy_(state["U0"])
    if case["problem"] == "ensemble":
        state["T"].zero_()
        state["status"].zero_()
        state["batch"].rk4(u, case["cfl"], case["steps"], state["T"], state["status"], limiter=LIMITER[case["limiter"]],
                           stream=stream)
        return {"U": u, "T": state["T"], "status": state["status"]}
    solver = state["solver"]
    if case["control"] == "loop":
        for _ in range(case["steps"]):
            solver.dt_from_cfl(u, state["cfl"], state["dt_dev"], stream=stream)
            solver.rk4_step(u, state["dt_dev"], state["limiter"], stream=stream)
        return {"U": u, "dt": state["dt_dev"]}
    if case["control"] == "cfl":
        steps, t = solver.rk4_integrate(u, 1, state["cfl"], nsteps=case["steps"], tf=1e30, limiter=state["limiter"], stream=stream)
    else:
        steps, t = solver.rk4_integrate(u, 0, state["dt"], nsteps=case["steps"], limiter=state["limiter"], stream=stream)
    return {"U": u, "steps": steps, "time": t}


def work(case):
    """Per RK4 stage the state it starts from is read and its result written
    once (a limiter can be part of either); the operations are those of the
    tensor-product scheme: values at the quadrature points, fluxes, test
    integrals, Riemann problems and the element's mass matrix."""
    if case["problem"] == "ensemble":
        ne, orders = _ensemble_spec(case)
        parts = [work(dict(case, problem="tube", nx=n, ny=1, order=p)) for n, p in zip(ne, orders)]
        return {k: sum(q[k] for q in parts) for k in ("bytes", "flops")}
    one_d = case["problem"] == "tube"
    d = 1 if one_d else 2
    f = 2 + d + {"single": 0, "two-fluid": 1, "passive": 2, "stiffened": 2}[case["physics"]]
    p = case["order"]
    n_s, n_q = (p + 1) ** d, (p + 1 if one_d else _volume_points(p)) ** d
    q1, n1 = round(n_q ** (1 / d)), p + 1
    faces, n_face = d, (1 if one_d else p + 1)
    apply_2d = 2 * (q1 * n1 * n1 + q1 * q1 * n1)  # one tensor-product transform of one field
    volume = f * (1 + d) * (apply_2d if d == 2 else 2 * q1 * n1) + n_q * (30 + 10 * d * f)
    surface = faces * n_face * (120 + 8 * f * n1)
    mass = f * (2 * d * n1 * n_s)
    elements = case["nx"] * case["ny"]
    limit = 0 if case["limiter"] in ("none", "hri", "learned") else f * d * (p + 1) ** (d - 1) * (4 * n1 * n1 + 20 * p)
    stages = 4 * case["steps"]
    return {"bytes": float(stages * 16 * elements * f * n_s), "flops": float(stages * elements * (volume + surface + mass + limit + 4 * f * n_s))}


# ----------------------------------------------------- the scheme in plain torch
def _volume_points(p):
    """Volume Gauss points per direction of the 2D element."""
    return 2 if p == 1 else p + 2


def _lagrange(nodes, x):
    """Values and derivatives of the Lagrange polynomials on `nodes` at x: [len(x), len(nodes)]."""
    v, d = np.zeros((len(x), len(nodes))), np.zeros((len(x), len(nodes)))
    for i in range(len(nodes)):
        poly = np.poly1d([1.0])
        for m in range(len(nodes)):
            if m != i:
                poly = poly * np.poly1d([1.0, -nodes[m]]) / (nodes[i] - nodes[m])
        v[:, i], d[:, i] = poly(x), poly.deriv()(x)
    return v, d


class _Grid:
    """Rows of elements; `count`: elements of each row (the rest of a row is
    padding) where the rows are separate problems; hx, hy broadcast over rows."""

    def __init__(self, case, dev, hx, hy, bc, count=None):
        def at(a):
            return torch.tensor(a, dtype=torch.float64, device=dev)
        self.physics, self.flux, self.p = case["physics"], case["flux"], case["order"]
        self.bc, self.hx, self.hy, self.d = bc, hx, hy, len(bc) // 2
        p, d = self.p, self.d
        nodes = np.linspace(-1, 1, p + 1)
        gx, gw = np.polynomial.legendre.leggauss(p + 1 if d == 1 else _volume_points(p))
        v, dv = _lagrange(nodes, gx)
        self.V, self.DV, self.w = at(v), at(dv), at(gw)
        fx, fw = np.polynomial.legendre.leggauss(p + 1)
        fv, _ = _lagrange(nodes, fx)
        self.FV, self.fw = at(fv), at(fw)
        mx, mw = np.polynomial.legendre.leggauss(p + 1)
        mv, _ = _lagrange(nodes, mx)
        self.Minv = at(np.linalg.inv(mv.T @ np.diag(mw) @ mv))
        taylor = np.zeros((p + 1, p + 1))  # derivatives at 0 of the Lagrange polynomials
        for i in range(p + 1):
            poly = np.poly1d([1.0])
            for m in range(p + 1):
                if m != i:
                    poly = poly * np.poly1d([1.0, -nodes[m]]) / (nodes[i] - nodes[m])
            for k in range(p + 1):
                taylor[k, i] = poly(0.0)
                poly = poly.deriv()
        self.L2T, self.T2L = at(taylor), at(np.linalg.inv(taylor))
        self.count = count

    def _last(self, ex, dev):
        """Row mask of the element at the right end of each row, [1, rows, ex]."""
        i = torch.arange(ex, device=dev)
        return (i[None] == (ex - 1 if self.count is None else (self.count - 1)[:, None]))[None]

    # -- pointwise physics; q[0..F-1], vel and normal as lists over directions
    def prim(self, q):
        d = self.d
        rho, vel, e = q[0], [q[1 + k] / q[0] for k in range(d)], q[d + 1]
        beta = q[d + 3] if self.physics == "stiffened" else torch.zeros_like(rho)
        alpha = q[d + 2] if self.physics in ("two-fluid", "stiffened") else torch.full_like(rho, 1 / (GAMMA - 1))
        p = (e - beta - 0.5 * rho * sum(v * v for v in vel)) / alpha
        return rho, vel, e, alpha, beta, p

    def speed(self, q):
        """Sound speed."""
        rho, vel, e, alpha, beta, p = self.prim(q)
        gamma = 1 + 1 / alpha
        return torch.sqrt(gamma * (p + (1 - 1 / gamma) * beta) / rho)

    def nonconservative(self):
        """First field that is not in conservation form (all after it are not either)."""
        return {"single": 2 + self.d, "two-fluid": 2 + self.d, "passive": 3 + self.d, "stiffened": 2 + self.d}[self.physics]

    def volume_flux(self, q, k):
        rho, vel, e, _, _, p = self.prim(q)
        f = [rho * vel[k]] + [rho * vel[k] * vel[j] + (p if j == k else 0) for j in range(self.d)] + [(e + p) * vel[k]]
        if self.physics == "passive":
            f.append(q[self.d + 2] * vel[k])
        return f + [torch.zeros_like(rho)] * (len(q) - len(f))

    def riemann(self, a, b, k):
        """Flux and non-conservative terms [F, ...] across a face normal to direction k, a to b."""
        d, nc0 = self.d, self.nonconservative()
        fa, fb = self.volume_flux(a, k), self.volume_flux(b, k)
        ra, va, ea, la, _, pa = self.prim(a)
        rb, vb, eb, lb, _, pb = self.prim(b)
        nc = [torch.zeros_like(ra) for _ in range(nc0)]
        if self.flux == "rusanov":
            s = torch.maximum(va[k].abs() + self.speed(a), vb[k].abs() + self.speed(b))
            f = [0.5 * (x + y) - 0.5 * s * (v - u) for x, y, u, v in zip(fa, fb, a, b)]
            nc += [-0.25 * (va[k] + vb[k]) * (v - u) for u, v in zip(a[nc0:], b[nc0:])]
            return torch.stack(f), torch.stack(nc)
        rt = torch.sqrt(rb / ra)

        def mean(x, y):
            return (x + rt * y) / (1 + rt)
        vel = [mean(x, y) for x, y in zip(va, vb)]
        rho, h, alpha = rt * ra, mean((ea + pa) / ra, (eb + pb) / rb), mean(la, lb)
        c = torch.sqrt((h - 0.5 * sum(v * v for v in vel)) / alpha)
        i = mean(pa * la, pb * lb)
        p = i / alpha
        dp = (alpha * (pb * lb - pa * la) - i * (lb - la)) / alpha ** 2 if self.physics in ("two-fluid", "stiffened") else pb - pa
        drho, dvn, vn = rb - ra, vb[k] - va[k], vel[k]
        w0 = (vn - c).abs() * (dp - rho * c * dvn) / (2 * c * c)
        w2 = vn.abs() * (drho - dp / (c * c))
        w3 = (vn + c).abs() * (dp + rho * c * dvn) / (2 * c * c)
        density = w0 + w2 + w3
        jump = [density]
        energy = w0 * (h - vn * c) + w2 * 0.5 * sum(v * v for v in vel) + w3 * (h + vn * c)
        for j in range(d):
            if j == k:
                jump.append(w0 * (vn - c) + w2 * vn + w3 * (vn + c))
            else:  # the shear wave
                shear = vn.abs() * rho * (vb[j] - va[j])
                jump.append(vel[j] * density + shear)
                energy = energy + shear * vel[j]
        if self.physics in ("two-fluid", "stiffened"):
            energy = energy + vn.abs() * (lb - la) * p
        if self.physics == "stiffened":
            energy = energy + vn.abs() * (b[d + 3] - a[d + 3])
        jump.append(energy)
        if self.physics == "passive":
            jump += [density, density]
        else:
            jump += [vn.abs() * (v - u) for u, v in zip(a[nc0:], b[nc0:])]
        nc += [-0.5 * vn * (v - u) for u, v in zip(a[nc0:], b[nc0:])]
        return torch.stack([0.5 * (x + y) - 0.5 * j for x, y, j in zip(fa, fb, jump)]), torch.stack(nc)

    # -- right-hand side: U[F, ey, ex, b, a]
    def rhs(self, U):
        d, V, DV, w, FV, fw = self.d, self.V, self.DV, self.w, self.FV, self.fw
        e = torch.einsum
        if d == 1:
            ug = e("fyxba,ga->fyxbg", U, V)
        else:
            ug = e("fyxba,hb,ga->fyxhg", U, V, V)
        q, nc0 = list(ug), self.nonconservative()
        wy = torch.ones(1, dtype=U.dtype, device=U.device) if d == 1 else w
        Vy = torch.ones(1, 1, dtype=U.dtype, device=U.device) if d == 1 else V
        half = [self.hx / 2, self.hy / 2 if d == 2 else 1.0]
        fx = torch.stack(self.volume_flux(q, 0)) * half[1]
        out = e("fyxhg,h,g,hb,ga->fyxba", fx, wy, w, Vy, DV)
        if d == 2:
            fy = torch.stack(self.volume_flux(q, 1)) * half[0]
            out = out + e("fyxhg,h,g,hb,ga->fyxba", fy, wy, w, DV, V)
        if nc0 < len(q):
            _, vel, *_ = self.prim(q)
            src = -vel[0] * e("fyxba,hb,ga->fyxhg", U[nc0:], Vy, DV) / half[0]
            if d == 2:
                src = src - vel[1] * e("fyxba,hb,ga->fyxhg", U[nc0:], DV, V) / half[1]
            out[nc0:] += e("fyxhg,h,g,hb,ga->fyxba", src * (half[0] * half[1]), wy, w, Vy, V)
        # faces normal to x: the trace of every element's right end against its right neighbour
        def reflect(t, k):
            t = t.clone()
            t[1 + k] = -t[1 + k]
            return t

        def sweep(left_end, right_end, k, tags, last):
            """left_end/right_end: traces [F, ..., n, ...] with the sweep's elements in dimension `dim`."""
            dim = 2 if k == 0 else 1
            nxt = torch.roll(left_end, -1, dim)
            if tags[1] != PERIODIC:
                ghost = reflect(right_end, k) if tags[1] == REFLECTIVE else right_end
                nxt = torch.where(last, ghost, nxt)
            F, N = self.riemann(list(right_end), list(nxt), k)
            to_right, to_left = -F + N, torch.roll(F + N, 1, dim)
            if tags[0] != PERIODIC:
                first = torch.zeros_like(last)
                first.select(dim, 0)[...] = True
                ghost = reflect(left_end, k) if tags[0] == REFLECTIVE else left_end
                Fg, Ng = self.riemann(list(ghost), list(left_end), k)
                to_left = torch.where(first, Fg + Ng, to_left)
            return to_right, to_left

        ey, ex = U.shape[1], U.shape[2]
        FVy = torch.ones(1, 1, dtype=U.dtype, device=U.device) if d == 1 else FV
        fwy = torch.ones(1, dtype=U.dtype, device=U.device) if d == 1 else fw
        L, R = e("fyxb,hb->fyxh", U[..., 0], FVy), e("fyxb,hb->fyxh", U[..., -1], FVy)
        last = self._last(ex, U.device)[..., None].expand(1, ey, ex, 1)
        r, l = sweep(L, R, 0, self.bc[:2], last)
        jf = half[1] if d == 2 else 1.0
        out[..., -1] += e("fyxh,h,hb->fyxb", r * jf, fwy, FVy)
        out[..., 0] += e("fyxh,h,hb->fyxb", l * jf, fwy, FVy)
        if d == 2:
            B, T = e("fyxa,ga->fyxg", U[..., 0, :], FV), e("fyxa,ga->fyxg", U[..., -1, :], FV)
            top = (torch.arange(ey, device=U.device) == ey - 1)[None, :, None, None].expand(1, ey, ex, 1)
            r, l = sweep(B, T, 1, self.bc[2:], top)
            out[..., -1, :] += e("fyxg,g,ga->fyxa", r * half[0], fw, FV)
            out[..., 0, :] += e("fyxg,g,ga->fyxa", l * half[0], fw, FV)
        # mass matrix
        if d == 1:
            return e("fyxba,ca->fyxbc", out, self.Minv) / half[0]
        return e("fyxba,db,ca->fyxdc", out, self.Minv, self.Minv) / (half[0] * half[1])

    # -- hierarchical reconstruction along one direction at a time
    def limit_along(self, U, k):
        dim, axis = (2, 4) if k == 0 else (1, 3)
        n = self.p
        A = torch.movedim(torch.movedim(U, axis, -1) @ self.L2T.T, -1, 0)  # [coefficient, F, ey, ex, other node]
        AL, AR = torch.roll(A, 1, dim + 1), torch.roll(A, -1, dim + 1)
        lim = [None] * (n + 1)
        avg_c = None
        for m in range(n, 0, -1):
            dl = dc = dr = rl = rc = rr = 0.0
            for j in range(m - 1, n + 1):
                e = j - m + 2
                inner = (1.0 - (-1.0) ** e) / math.factorial(e)
                dl, dc, dr = dl + AL[j] * inner, dc + A[j] * inner, dr + AR[j] * inner
                if j > m:
                    rl = rl + lim[j] * (((-1.0) ** e - (-3.0) ** e) / math.factorial(e))
                    rc = rc + lim[j] * inner
                    rr = rr + lim[j] * ((3.0 ** e - 1.0) / math.factorial(e))
            avg_c = 0.5 * (dc - rc)
            c1, c2 = 0.5 * (avg_c - 0.5 * (dl - rl)), 0.5 * (0.5 * (dr - rr) - avg_c)
            lim[m] = torch.where(c1 * c2 > 0, torch.sign(c1) * torch.minimum(c1.abs(), c2.abs()), torch.zeros_like(c1))
        lim[0] = avg_c
        lim = torch.stack(lim)
        tags = self.bc[2 * k:2 * k + 2]
        if tags[0] != PERIODIC:  # the end elements keep their mean; at a wall the normal momentum stays as it is
            mean = sum(A[j] * ((1.0 - (-1.0) ** (j + 1)) / math.factorial(j + 1)) for j in range(n + 1)) * 0.5
            flat = torch.cat([mean[None], torch.zeros_like(A[1:])])
            ends = self._last(U.shape[2], U.device)[..., None].expand(1, U.shape[1], U.shape[2], 1).clone() if k == 0 else \
                torch.zeros(1, U.shape[1], U.shape[2], 1, dtype=torch.bool, device=U.device)
            if k == 0:
                ends[:, :, 0] = True
            else:
                ends[:, 0] = True
                ends[:, -1] = True
            if tags[0] == REFLECTIVE:
                flat[:, 1 + k] = A[:, 1 + k]
            lim = torch.where(ends, flat, lim)
        return torch.movedim(torch.movedim(lim, 0, -1) @ self.T2L.T, -1, axis).contiguous()

    def limit(self, U, limiter):
        if limiter == "none":
            return U
        U = self.limit_along(U, 0)
        return self.limit_along(U, 1) if self.d == 2 else U

    def dt(self, U, cfl):
        q = list(U)
        c = self.speed(q)
        s = torch.stack([v.abs() + c for v in self.prim(q)[1]]).amax(0)
        if self.count is None:
            return cfl / s.max()
        used = torch.arange(U.shape[2], device=U.device)[None] < self.count[:, None]
        return (cfl / torch.where(used[..., None, None], s, torch.zeros_like(s)).amax((1, 2, 3)))[:, None, None, None]

    def step(self, U, dt, limiter):
        acc, stage = U, U
        for k, (nxt, g) in enumerate(((0.5, 1 / 6), (0.5, 1 / 3), (1.0, 1 / 3), (0.0, 1 / 6))):
            du = dt * self.rhs(self.limit(stage, limiter) if k else stage)
            acc, stage = acc + g * du, U + nxt * du
        return self.limit(acc, limiter)


def exact(case, seed):
    if case["limiter"] in ("hri", "learned") or case["precision"] != "fp64":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["problem"] == "ensemble":
        return _exact_ensemble(case, seed, dev)
    hx, hy = _cell(case)
    grid = _Grid(case, dev, hx, hy, _box(case)[1])
    U, cfl, lim = _initial(case, seed, dev), _cfl_length(case), case["limiter"]
    dt, t = grid.dt(U, cfl), 0.0
    if case["control"] == "cfl":
        U = grid.limit(U, lim)
    for _ in range(case["steps"]):
        if case["control"] != "fixed":
            dt = grid.dt(U, cfl)
        U = grid.step(U, dt, lim)
        t = t + float(dt)
    packed = _pack(U, _flat_nodes(case, case["order"]))
    if case["control"] == "loop":
        return {"U": packed, "dt": dt.reshape(1)}
    return {"U": packed, "steps": case["steps"], "time": t}


def _exact_ensemble(case, seed, dev):
    """The problems of one order as rows of one grid, padded to the longest."""
    ne, orders = _ensemble_spec(case)
    parts, times = [None] * len(ne), torch.zeros(len(ne), dtype=torch.float64, device=dev)
    for p in (1, 2, 3):
        ids = [k for k in range(len(ne)) if orders[k] == p]
        if not ids:
            continue
        states = [_ensemble_state(case, k, ne[k], p, seed, dev) for k in ids]
        longest = max(ne[k] for k in ids)
        U = torch.cat([torch.cat([s, s[:, :, -1:].expand(-1, -1, longest - s.shape[2], -1, -1)], 2) for s in states], 1)
        count = torch.tensor([ne[k] for k in ids], device=dev)
        hx = (2.0 / count.double())[:, None, None, None]
        grid = _Grid(dict(case, order=p), dev, hx, 1.0, (FARFIELD, FARFIELD), count)
        cfl = case["cfl"] * hx.reshape(-1) / (2 * p + 1)
        U = grid.limit(U, case["limiter"])
        t = 0
        for _ in range(case["steps"]):
            dt = grid.dt(U, cfl)
            U = grid.step(U, dt, case["limiter"])
            t = t + dt.reshape(-1)
        for i, k in enumerate(ids):
            parts[k] = _pack(U[:, i:i + 1, :ne[k]].contiguous(), _lattice_1d(p))
            times[k] = t[i]
    return {"U": torch.cat(parts), "T": times, "status": None}
