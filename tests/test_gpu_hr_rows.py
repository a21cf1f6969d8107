"""The one-launch 2D HR limiter on grids with many rows, where a block marches
up its strip of 256 (element, field) columns: the bits of the two in-place
sweeps, for rows of one column less and more than a strip, a last strip narrower
than an element, a single strip, row counts that leave a remainder, and every
boundary kind at the ends (walls and far fields limit without neighbours)."""
import numpy as np
import pytest
import torch

from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, PASSIVE, PERIODIC, REFLECTIVE, ROE, SINGLEFLUID, STIFFENED, Config,
                    Mesh, Solver, nfields, problems)

pytestmark = pytest.mark.gpu

BCS = [(PERIODIC,) * 4, (FARFIELD, FARFIELD, REFLECTIVE, REFLECTIVE), (REFLECTIVE, FARFIELD, PERIODIC, PERIODIC),
       (PERIODIC, PERIODIC, FARFIELD, REFLECTIVE)]
CASES = [(SINGLEFLUID, (64, 1541)), (SINGLEFLUID, (65, 770)), (MULTIFLUID, (51, 1537)), (MULTIFLUID, (52, 801)),
         (MULTIFLUID, (103, 523)), (PASSIVE, (205, 311)), (STIFFENED, (43, 790)), (STIFFENED, (42, 1540))]


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("ph,n", CASES)
def test_rows_equal_two_sweeps(device, order, ph, n):
    for k, bc in enumerate(BCS):
        mesh = Mesh(2, order, n[0], n[1], 0.0, 1.0, 0.0, 2.0, bc=bc, nfields=nfields(2, ph))
        solver = Solver(Config(2, order, ph, ROE), mesh)
        assert solver.hr_one_launch
        U = problems.oblique_riemann_state(mesh, ph, seed=k)
        U *= 1.0 + 0.02 * np.sin(0.37 * np.arange(U.size))  # no column smooth enough to pass unlimited
        Ud = torch.from_numpy(U).to(device)
        buf = torch.full((U.size + 1,), float("nan"), dtype=torch.float64, device=device)
        out = buf[k % 2:U.size + k % 2]  # 16-byte aligned, then not
        solver.limit_into(LIMIT_HR, Ud, out)
        torch.cuda.synchronize()
        assert np.array_equal(Ud.cpu().numpy(), U)
        solver.limit(LIMIT_HR, Ud)
        torch.cuda.synchronize()
        assert torch.equal(out, Ud), (order, ph, n, bc)
        assert not np.array_equal(Ud.cpu().numpy(), U)
