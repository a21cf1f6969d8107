"""Which kernels a run launches, from the solver's own launch counts: the tile
kernel on every 2D grid, whole tiles or ragged, built or read from a file in
grid order; one launch a step on 1D grids; the face + element kernels where
they are asked for and on file meshes whose elements are in another order."""
import pytest
import torch

from dg_amd import (FARFIELD, LIMIT_HR, MULTIFLUID, PATH_GENERAL, PATH_TILED, REFLECTIVE, ROE, Config, Mesh, Solver, problems)

pytestmark = pytest.mark.gpu
BC = (FARFIELD, FARFIELD, REFLECTIVE, REFLECTIVE)


def _launches(device, mesh, d, order, path, limiter):
    solver = Solver(Config(d, order, MULTIFLUID, ROE), mesh)
    if path is not None:
        solver.set_path(path)
    U = torch.from_numpy(problems.smooth_random_state(mesh, MULTIFLUID, seed=1)).to(device)
    solver.profile(True)
    solver.rk4_integrate(U, 0, 1e-4, nsteps=2, limiter=limiter)
    torch.cuda.synchronize()
    return solver, {k: solver.profile_read(k)[1] for k in ("stage", "face", "elem")}


TILE = {"stage": 8, "face": 0, "elem": 0}
GENERAL = {"stage": 0, "face": 8, "elem": 8}


@pytest.mark.parametrize("limiter", [0, LIMIT_HR])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("n", [(16, 8), (11, 7)])
def test_2d_grids(device, tmp_path, order, n, limiter):
    built = Mesh(2, order, n[0], n[1], 0.0, 1.2, 0.0, 0.7, bc=BC, nfields=5)
    built.write_gmsh(tmp_path / "m.msh")
    for mesh, whole in ((built, n[0] % 8 == 0), (Mesh.from_gmsh(tmp_path / "m.msh", nfields=5), False)):
        solver, count = _launches(device, mesh, 2, order, None, limiter)
        assert count == TILE, (order, n, whole)
        assert solver.path == (PATH_TILED if whole else PATH_GENERAL)
        assert solver.hr_one_launch == (order <= 2)
        assert _launches(device, mesh, 2, order, PATH_GENERAL, limiter)[1] == GENERAL


def test_file_in_another_order(device, tmp_path):
    """The same elements, one pair swapped in the file: no grid."""
    Mesh(2, 2, 8, 4, 0.0, 1.2, 0.0, 0.7, bc=BC, nfields=5).write_gmsh(tmp_path / "m.msh")
    lines = (tmp_path / "m.msh").read_text().split("\n")
    quads = [i for i, s in enumerate(lines) if len(s.split()) > 9 and s.split()[1] == "10"]
    assert len(quads) == 32
    a, b = quads[3], quads[12]
    lines[a], lines[b] = lines[b], lines[a]
    (tmp_path / "m.msh").write_text("\n".join(lines))
    mesh = Mesh.from_gmsh(tmp_path / "m.msh", nfields=5)
    assert _launches(device, mesh, 2, 2, None, 0)[1] == GENERAL


@pytest.mark.parametrize("limiter", [0, LIMIT_HR])
def test_1d_grids(device, limiter):
    mesh = Mesh(1, 2, 101, 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=4)
    assert _launches(device, mesh, 1, 2, None, limiter)[1] == {"stage": 2, "face": 0, "elem": 0}
    assert _launches(device, mesh, 1, 2, PATH_GENERAL, limiter)[1] == GENERAL
