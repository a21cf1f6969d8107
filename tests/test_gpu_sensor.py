"""The troubled-cell sensor where its kernels decide by bounds and walk chains.

The tests of a pair run only where a bound of their measures passes a
threshold, and each element settles by itself which earlier elements flagged
it.  Flags are compared with the oracle's sequential loop, every flag equal: on
ramps whose jump per cell lies within a tenth of a threshold on either side (a
whole row points at its next element, so the chains are as long as the mesh),
on random walks, for thresholds from 0 to past the measures' largest value
1/2, with near-vacuum, negative and NaN cells, and on meshes two elements wide,
where a periodic neighbour counts twice.  The averages that an RK stage leaves
for the sensor give the run of the kernels that form them from the state.
"""
import numpy as np
import pytest
import torch

import oracle
from dg_amd import (FARFIELD, LIMIT_HRI, LIMIT_M2I, LIMIT_P0I, LIMIT_PRI, MULTIFLUID, PASSIVE, PERIODIC, REFLECTIVE, ROE,
                    STIFFENED, Config, Mesh, Solver, nfields, problems)
from tests.helpers import per_field_rel

pytestmark = pytest.mark.gpu


def _state(mesh, d, order, ph, kind, size, seed, spoil=False):
    """Nodal state whose cells step by `size` in the logarithm of density,
    pressure and 1/(gamma-1), along the element numbers or in a random walk."""
    rng = np.random.default_rng(seed)
    n, nf, ns = mesh.sizes["N_E"], nfields(d, ph), (order + 1) ** d

    def levels():
        step = np.ones(n) if kind == "ramp" else rng.choice([-1.0, 0.0, 1.0], n)
        walk = np.cumsum(step * size * rng.uniform(0.9, 1.1, n))
        return np.exp(np.clip(walk - walk.mean(), -6, 6)) if rng.random() < 0.7 else np.ones(n)

    rho, p = levels(), levels()
    alpha = 2.5 * levels() if ph in (MULTIFLUID, STIFFENED) else np.full(n, 2.5)
    beta = np.full(n, 0.7) if ph == STIFFENED else np.zeros(n)
    u, v = 0.3 * np.sin(np.arange(n) * size), rng.normal(0, 0.01, n)
    U = np.zeros((n, nf))
    U[:, 0], U[:, 1] = rho, rho * u
    if d == 2:
        U[:, 2] = rho * v
    U[:, d + 1] = p * alpha + beta + 0.5 * rho * (u * u + (v * v if d == 2 else 0.0))
    U[:, d + 2] = alpha if ph in (MULTIFLUID, STIFFENED) else rho
    if ph == STIFFENED:
        U[:, d + 3] = beta
    if spoil:
        pick = rng.permutation(n)[:8]
        U[pick[:2], 0] *= -1.0
        U[pick[2:4], d + 1] *= -1.0
        U[pick[4:6], 0] = 1e-300
        U[pick[6], 0] = np.nan
        U[pick[7], d + 1] = np.inf
    nodal = np.repeat(U[:, :, None], ns, axis=2)
    return np.ascontiguousarray((nodal * (1.0 + 1e-9 * rng.normal(size=nodal.shape))).reshape(-1))


@pytest.mark.parametrize("ph", [MULTIFLUID, PASSIVE, STIFFENED])
@pytest.mark.parametrize("d,n,bc", [
    (1, (1500,), (PERIODIC, PERIODIC)), (1, (2,), (PERIODIC, PERIODIC)), (1, (300,), (FARFIELD, REFLECTIVE)),
    (2, (257, 3), (PERIODIC,) * 4), (2, (2, 9), (PERIODIC,) * 4),
    (2, (33, 16), (FARFIELD, REFLECTIVE, PERIODIC, PERIODIC)),
])
def test_flags_of_chains_and_thresholds(device, ph, d, n, bc):
    order = 1
    # 1D meshes are numbered along x, 2D ones row by row
    mesh = (Mesh(1, order, n[0], bc=bc, nfields=nfields(1, ph)) if d == 1 else
            Mesh(2, order, n[0], n[1], 0.0, 1.0, 0.0, 0.5, bc=bc, nfields=nfields(2, ph)))
    prob = oracle.Problem(mesh.tables(), ph, ROE)
    solver = Solver(Config(d, order, ph, ROE), mesh)
    flagged = 0
    for k, th in enumerate([1e-5, 1e-3, 0.02, 0.2, 0.45, 0.0, 0.5, 0.7, -1.0]):
        for kind in ("ramp", "walk"):
            for on in ((th,), (th, th), (2.0, th, th), (th, 2.0, 2.0), (2.0, 2.0, th)):
                size = min(max(th, 1e-7), 0.5) * (6 if on[:2] == (2.0, 2.0) else 1)  # gamma moves less than 1/(gamma-1)
                U = _state(mesh, d, order, ph, kind, size, 100 * k + len(on), spoil=mesh.sizes["N_E"] > 100 and k % 3 == 2)
                with np.errstate(all="ignore"):
                    ref, uavg = prob.sensing(U, on)
                Ud = torch.from_numpy(U).to(device)
                sd = torch.full((prob.cfg.N_E,), -7, dtype=torch.int32, device=device)
                ua = torch.zeros(prob.cfg.N_E * prob.nf, dtype=torch.float64, device=device)
                solver.set_sensor_thresholds(on)
                solver.sensing(Ud, sd, ua)
                torch.cuda.synchronize()
                assert np.array_equal(ua.cpu().numpy(), uavg, equal_nan=True)
                assert np.array_equal(sd.cpu().numpy(), ref), (th, kind, on)
                flagged += int((ref != 0).sum())
    assert flagged


@pytest.mark.parametrize("order,n", [(2, (16, 8)), (2, (19, 6)), (3, (9, 7)), (3, (8, 4))])
@pytest.mark.parametrize("ph,limiter", [(MULTIFLUID, LIMIT_HRI), (MULTIFLUID, LIMIT_M2I), (MULTIFLUID, LIMIT_PRI),
                                        (MULTIFLUID, LIMIT_P0I), (PASSIVE, LIMIT_HRI), (STIFFENED, LIMIT_HRI)])
def test_averages_of_the_stage(device, order, n, ph, limiter):
    """Limited steps against the oracle (1e-11, as the other limited runs):
    each stage's averages decide the flags of the limiter after it."""
    mesh = Mesh(2, order, n[0], n[1], 0.0, 1.2, 0.0, 0.7, bc=(FARFIELD, FARFIELD, PERIODIC, PERIODIC),
                nfields=nfields(2, ph))
    prob = oracle.Problem(mesh.tables(), ph, ROE)
    solver = Solver(Config(2, order, ph, ROE), mesh)
    U0 = problems.oblique_riemann_state(mesh, ph, seed=11)
    th = (0.01, 0.01, 0.01)
    solver.set_sensor_thresholds(th)
    dt = 0.3 * prob.dt_from_cfl(U0, mesh.dx / (2 * order + 1))
    U_ref, _, _, _ = prob.rk4(U0, 0, dt, nsteps=4, limiter=limiter, thresholds=th)
    Ud = torch.from_numpy(U0).to(device)
    solver.rk4_integrate(Ud, 0, dt, nsteps=4, limiter=limiter)
    torch.cuda.synchronize()
    for l2, li in per_field_rel(Ud.cpu().numpy(), U_ref, prob.nf, prob.cfg.N_s):
        assert l2 < 1e-11 and li < 1e-11, (l2, li)
