"""The tile kernel and the one-launch HR limiter on 2D grids whose sides are
not whole tiles (8 x 4 and 8 x 8 elements), built or read from a Gmsh file:
one element less, one more, a single row or column, odd and even row lengths
(paired loads and stores need whole pairs).

Against the oracle: the right-hand side to 1e-12 of its largest value (FMA
contraction only) and limited RK4 runs to 1e-11 relative L2 and Linf per
field, the bars of the whole-tile grids.  The one-launch limiter gives the
bits of the two in-place sweeps.
"""
import numpy as np
import pytest
import torch

import oracle
from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, PASSIVE, PATH_GENERAL, PERIODIC, REFLECTIVE, ROE, RUSANOV,
                    SINGLEFLUID, STIFFENED, Config, Mesh, Solver, nfields, problems)
from tests.helpers import per_field_rel

pytestmark = pytest.mark.gpu

BCS = [(PERIODIC,) * 4, (FARFIELD, FARFIELD, REFLECTIVE, REFLECTIVE), (REFLECTIVE, FARFIELD, PERIODIC, PERIODIC)]
SIZES = [(7, 3), (9, 5), (16, 9), (2, 6), (23, 1), (1, 4), (10, 4)]


def _run(device, mesh, order, ph, flux, seed):
    prob = oracle.Problem(mesh.tables(), ph, flux)
    U0 = problems.smooth_random_state(mesh, ph, seed=seed)
    solver = Solver(Config(2, order, ph, flux), mesh)
    assert solver.path == PATH_GENERAL  # the reported path: whole tiles only
    Ud = torch.from_numpy(U0).to(device)
    f = torch.full_like(Ud, float("nan"))
    solver.rhs(Ud, f)
    torch.cuda.synchronize()
    ref = prob.rhs(U0)
    assert np.abs(f.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    dt = 0.3 * prob.dt_from_cfl(U0, mesh.dx / (2 * order + 1))
    for limiter in (0, LIMIT_HR):
        U_ref, _, _, _ = prob.rk4(U0, 0, dt, nsteps=3, limiter=limiter)
        Ud = torch.from_numpy(U0).to(device)
        solver.rk4_integrate(Ud, 0, dt, nsteps=3, limiter=limiter)
        torch.cuda.synchronize()
        for l2, li in per_field_rel(Ud.cpu().numpy(), U_ref, prob.nf, prob.cfg.N_s):
            assert l2 < 1e-11 and li < 1e-11, (mesh.sizes["nx"], mesh.sizes["ny"], order, ph, limiter, l2, li)
    out = torch.full_like(Ud, float("nan"))
    solver.limit_into(LIMIT_HR, Ud, out)
    solver.limit(LIMIT_HR, Ud)
    torch.cuda.synchronize()
    assert torch.equal(out, Ud)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("ph", [SINGLEFLUID, MULTIFLUID, PASSIVE, STIFFENED])
def test_ragged_grids(device, order, ph):
    for k, (nx, ny) in enumerate(SIZES):
        mesh = Mesh(2, order, nx, ny, 0.0, 1.2, 0.0, 0.7, bc=BCS[k % 3], nfields=nfields(2, ph))
        _run(device, mesh, order, ph, ROE if k % 2 else RUSANOV, 10 * order + k)


@pytest.mark.parametrize("order,n,bc", [(1, (9, 6), BCS[1]), (2, (16, 8), BCS[0]), (2, (11, 7), BCS[2]), (3, (8, 5), BCS[1])])
def test_gmsh_grid(device, tmp_path, order, n, bc):
    """A file in grid order takes the same kernels, whole tiles or not."""
    m = Mesh(2, order, n[0], n[1], 0.0, 1.2, 0.0, 0.7, bc=bc, nfields=5)
    m.write_gmsh(tmp_path / "m.msh")
    _run(device, Mesh.from_gmsh(tmp_path / "m.msh", nfields=5), order, MULTIFLUID, ROE, 3)


def test_state_not_16_byte_aligned(device):
    """The paired instance needs aligned states; others take single loads and
    stores and give the same bits."""
    mesh = Mesh(2, 2, 18, 7, 0.0, 1.2, 0.0, 0.7, bc=BCS[1], nfields=5)
    solver = Solver(Config(2, 2, MULTIFLUID, ROE), mesh)
    U0 = problems.smooth_random_state(mesh, MULTIFLUID, seed=2)
    out = []
    for shift in (0, 1):
        big = torch.zeros(U0.size + shift, dtype=torch.float64, device=device)
        U = big[shift:]
        U.copy_(torch.from_numpy(U0))
        solver.rk4_integrate(U, 0, 1e-3, nsteps=2, limiter=LIMIT_HR)
        torch.cuda.synchronize()
        out.append(U.cpu().numpy())
    assert np.array_equal(out[0], out[1])
