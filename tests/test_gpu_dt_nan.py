"""Dt of states that hold NaN: the reference's idamax passes over a NaN that is
not the first value, so Dt comes from the largest finite |u|+a, wherever in a
wave, a block or the mesh the NaN lie; a NaN in the first node is Dt itself.
Bit for bit the oracle's Dt, and CFL runs with the time control on the device
and on the host give the same steps, times and states."""
import numpy as np
import pytest
import torch

import oracle
from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, ROE, SINGLEFLUID, Config, DgxError, Mesh, Solver, nfields, problems)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,order,ph", [(1, (64,), 1, SINGLEFLUID), (1, (1000,), 3, MULTIFLUID), (2, (24, 20), 2, MULTIFLUID),
                                          (2, (9, 5), 1, SINGLEFLUID)])
def test_dt_passes_over_nan(device, d, n, order, ph):
    nf, ns = nfields(d, ph), (order + 1) ** d
    mesh = (Mesh(1, order, n[0], 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=nf) if d == 1 else
            Mesh(2, order, n[0], n[1], 0.0, 1.2, 0.0, 0.7, bc=(FARFIELD,) * 4, nfields=nf))
    prob = oracle.Problem(mesh.tables(), ph, ROE)
    solver = Solver(Config(d, order, ph, ROE), mesh)
    base = problems.smooth_random_state(mesh, ph, seed=7)
    nodes = mesh.sizes["N_E"] * ns
    cfl = 0.3 * mesh.dx / (2 * order + 1)
    rng = np.random.default_rng(5)
    picks = [[k] for k in (1, 16, 32, 48, 63)] + [[64] if nodes > 64 else [2], [0], [0, 5], list(range(1, nodes, 2)), list(range(1, nodes))]
    picks += [rng.permutation(nodes - 1)[:k] + 1 for k in (3, nodes // 10, nodes // 3)]
    dt = torch.zeros(1, dtype=torch.float64, device=device)
    for pick in picks:
        U0 = base.copy()
        U0.reshape(-1, nf, ns)[np.asarray(pick) // ns, 0, np.asarray(pick) % ns] = np.nan
        with np.errstate(all="ignore"):
            ref = prob.dt_from_cfl(U0, cfl)
        solver.dt_from_cfl(torch.from_numpy(U0).to(device), cfl, dt)
        torch.cuda.synchronize()
        assert np.array_equal(dt.cpu().numpy(), [ref], equal_nan=True), (list(pick)[:5], float(dt), ref)
        assert np.isnan(ref) == (pick[0] == 0)
        if len(pick) > 3 or np.isnan(ref):
            continue
        for limiter in (0, LIMIT_HR):
            out = []
            for on in (True, False):
                solver.set_device_time(on)
                U = torch.from_numpy(U0).to(device)
                try:
                    run = solver.rk4_integrate(U, 1, cfl, nsteps=2, tf=1e30, limiter=limiter)
                except DgxError as e:  # the first step carried the NaN to the first node
                    run = str(e)
                torch.cuda.synchronize()
                out.append((run, U.cpu().numpy()))
            assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1], equal_nan=True)
