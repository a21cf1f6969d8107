"""The 1D whole-step kernel in its widest launch shape, two elements a lane,
and past the block count (2048) from which the maxima of |u|+a are reduced by a
launch of their own before the step.

Device time control against the per-step host loop (the same bits, state and
time), against the face + element kernels (1e-11 per field, the bar of every
RK4 trajectory here), and a NaN in the mesh's first node, which alone decides
the time step then: the run stops before its first step and leaves the state.
"""
import numpy as np
import pytest
import torch

from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, PATH_GENERAL, ROE, RUSANOV, SINGLEFLUID, Config, Mesh, Solver,
                    nfields, problems)
from tests.helpers import per_field_rel

pytestmark = pytest.mark.gpu

# two elements a lane (windows of 256, 170 and 128 elements that own 16 fewer
# with the limiter, 8 without): the first size is past 1536 blocks of one
# element a lane, the second past 2048 blocks of two
CASES = [(1, 172033, LIMIT_HR), (1, 491521, LIMIT_HR), (2, 105985, LIMIT_HR), (2, 315393, LIMIT_HR), (3, 229377, LIMIT_HR),
         (3, 245761, 0)]


@pytest.mark.parametrize("order,n,limiter", CASES)
def test_wide_launch_and_own_reduction(device, order, n, limiter):
    ph, flux = (MULTIFLUID, ROE) if order == 3 else (SINGLEFLUID, RUSANOV)
    mesh = Mesh(1, order, n, 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=nfields(1, ph))
    solver = Solver(Config(1, order, ph, flux), mesh)
    U0 = problems.smooth_random_state(mesh, ph, seed=order)
    cfl = 0.3 * mesh.dx / (2 * order + 1)
    runs = []
    for path, on in ((0, True), (0, False), (PATH_GENERAL, False)):
        solver.set_path(path)
        solver.set_device_time(on)
        U = torch.from_numpy(U0).to(device)
        k, T = solver.rk4_integrate(U, 1, cfl, nsteps=3, tf=1e30, limiter=limiter)
        torch.cuda.synchronize()
        assert k == 3
        runs.append((U.cpu().numpy(), T))
    assert np.array_equal(runs[0][0], runs[1][0]) and runs[0][1] == runs[1][1]
    assert abs(runs[0][1] - runs[2][1]) <= 1e-12 * runs[2][1]
    for l2, li in per_field_rel(runs[0][0], runs[2][0], nfields(1, ph), order + 1):
        assert l2 < 1e-11 and li < 1e-11, (order, n, l2, li)
    assert not np.array_equal(runs[0][0], U0)


@pytest.mark.parametrize("n", [300, 245761])
def test_nan_in_the_first_node_stops_the_run(device, n):
    mesh = Mesh(1, 3, n, 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=4)
    solver = Solver(Config(1, 3, MULTIFLUID, ROE), mesh)
    U0 = problems.smooth_random_state(mesh, MULTIFLUID, seed=1)
    U0[0] = np.nan
    U = torch.from_numpy(U0).to(device)
    with pytest.raises(Exception, match="too small or NaN"):
        solver.rk4_integrate(U, 1, 0.3 * mesh.dx / 7, nsteps=5, tf=1e30, limiter=0)
    torch.cuda.synchronize()
    assert np.array_equal(U.cpu().numpy(), U0, equal_nan=True)
