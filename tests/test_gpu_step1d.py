"""The 1D whole-step kernel (k_step1d: one launch per RK4 step) where its
windows can go wrong: meshes of one window and one element more or less,
fewer elements than the halo on a periodic mesh, both domain ends, and the
element counts at which the launch shape changes.

Every case runs a few CFL steps and a fixed-Dt run against the oracle (1e-11
relative L2 and Linf per field, the bar of every RK4 trajectory here), the
device's time control against the per-step host loop (the same bits: the
same kernel, with Dt from its own maxima or from k_upa_max), and the face +
element kernels (1e-11 again).
"""
import numpy as np
import pytest
import torch

import oracle
from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, PASSIVE, PATH_GENERAL, PERIODIC, REFLECTIVE, ROE, RUSANOV,
                    SINGLEFLUID, STIFFENED, Config, Mesh, Solver, nfields, problems)
from tests.helpers import per_field_rel

pytestmark = pytest.mark.gpu


def _check(device, n, order, ph, flux, bc, limiter, steps):
    mesh = Mesh(1, order, n, 1, -1.0, 1.0, bc=bc, nfields=nfields(1, ph))
    prob = oracle.Problem(mesh.tables(), ph, flux)
    U0 = problems.smooth_random_state(mesh, ph, seed=n + order)
    cfl = 0.3 * mesh.dx / (2 * order + 1)
    solver = Solver(Config(1, order, ph, flux), mesh)
    U_ref, n_ref, T_ref, _ = prob.rk4(U0, 1, cfl, nsteps=steps, tf=1e30, limiter=limiter)
    out = []
    for on in (True, False):
        solver.set_device_time(on)
        U = torch.from_numpy(U0).to(device)
        k, T = solver.rk4_integrate(U, 1, cfl, nsteps=steps, tf=1e30, limiter=limiter)
        assert k == n_ref and abs(T - T_ref) <= 1e-12 * T_ref
        torch.cuda.synchronize()
        out.append((U.cpu().numpy(), T))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    dt = prob.dt_from_cfl(U0, cfl)
    F_ref, _, _, _ = prob.rk4(U0, 0, dt, nsteps=steps, limiter=limiter)
    runs = [(out[0][0], U_ref)]
    for path in (0, PATH_GENERAL):
        solver.set_path(path)
        U = torch.from_numpy(U0).to(device)
        solver.rk4_integrate(U, 0, dt, nsteps=steps, limiter=limiter)
        torch.cuda.synchronize()
        runs.append((U.cpu().numpy(), F_ref))
    for U, ref in runs:
        for l2, li in per_field_rel(U, ref, prob.nf, prob.cfg.N_s):
            assert l2 < 1e-11 and li < 1e-11, (n, order, ph, bc, limiter, l2, li)


@pytest.mark.parametrize("limiter", [0, LIMIT_HR])
@pytest.mark.parametrize("bc", [(FARFIELD, REFLECTIVE), (PERIODIC, PERIODIC)])
@pytest.mark.parametrize("order,sizes", [(1, (2, 48, 49, 64, 65)), (2, (3, 26, 27, 42, 43)), (3, (5, 16, 17, 32, 33))])
def test_window_edges(device, order, sizes, bc, limiter):
    """Windows of 64, 42 and 32 elements that own 48, 26 and 16 of them."""
    for k, n in enumerate(sizes):
        ph = (SINGLEFLUID, MULTIFLUID, PASSIVE, STIFFENED)[k % 4]
        _check(device, n, order, ph, ROE if k % 2 else RUSANOV, bc, limiter, 3)


@pytest.mark.parametrize("n", [8192, 8193, 73728, 73729])
def test_launch_shapes(device, n):
    """p = 3: the last mesh of the two narrow launch shapes and the first of
    the next (512 blocks of 16 elements, 1536 of 48)."""
    _check(device, n, 3, MULTIFLUID, ROE, (FARFIELD, FARFIELD), LIMIT_HR, 2)
