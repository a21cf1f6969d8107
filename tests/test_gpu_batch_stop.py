"""Ensemble problems that stop while cut into several segments.

A stop is one decision of all workgroups of a problem: two gas halves that
part fast enough to leave a vacuum lose positivity after a few steps, with the
middle segments turning NaN first.  Such a problem gets status 1, keeps the
state and time of its last step however many steps follow, in one call or two,
and gives the bits of the same problem on one workgroup.  A problem that
enters with a status of its own is left alone, and the others run on as if they
were by themselves.
"""
import numpy as np
import pytest
import torch

from dg_amd import FARFIELD, MULTIFLUID, ROE, Batch, Config, Mesh, problems

pytestmark = pytest.mark.gpu

N_E, CFL = 300, 0.4


def _parting(mesh, speed):
    """rho = 1, p = 0.1 on both sides, moving apart at `speed`."""
    x, _ = problems.node_xy(mesh)
    left = (x[:, :1] < 1e-12) & np.ones_like(x, dtype=bool)
    v, p = np.where(left, -speed, speed), np.full_like(x, 0.1)
    return np.stack([np.ones_like(x), v, p / 0.4 + 0.5 * v * v, np.full_like(x, 2.5)], axis=1).reshape(-1)


@pytest.mark.parametrize("block", [64, 128, 256, 1024])
def test_cut_problem_stops(device, block):
    orders = [1, 2, 3, 1, 2, 3, 2]
    speeds = [1.0, 1.0, 1.0, 0.1, 0.1, 0.1, 1.0]  # the last one is never started
    n, bad, good, off = 7, [0, 1, 2], [3, 4, 5], 6
    cfg = Config(1, 1, MULTIFLUID, ROE)
    meshes = [Mesh(1, p, N_E, 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=4) for p in orders]
    states = [_parting(m, s) for m, s in zip(meshes, speeds)]

    def run(ids, min_chunk, calls):
        batch = Batch(cfg, [N_E] * len(ids), [orders[k] for k in ids])
        batch.set_min_chunk(min_chunk)
        batch.set_block_sizes([block])
        cut = batch.block_sizes[2]
        U = torch.from_numpy(batch.pack([states[k] for k in ids])).to(device)
        T = torch.zeros(len(ids), dtype=torch.float64, device=device)
        st = torch.tensor([5 if k == off else 0 for k in ids], dtype=torch.int32, device=device)
        for c, steps in enumerate(calls):
            batch.rk4(U, CFL, steps, T, st, limit_initial=c == 0)
        torch.cuda.synchronize()
        return batch.unpack(U.cpu().numpy()), T.cpu().numpy(), st.cpu().numpy(), cut

    everyone = list(range(n))
    U, T, st, cut = run(everyone, 16, [24])
    assert cut >= (n if block <= 256 else 0)
    assert list(st) == [1, 1, 1, 0, 0, 0, 5]
    assert (T[bad] > 0).all() and T[off] == 0.0
    assert np.array_equal(U[off], states[off])
    for min_chunk, calls in ((16, [25]), (16, [40]), (16, [13, 18]), (0, [24])):
        V, S, s2, _ = run(everyone, min_chunk, calls)
        assert list(s2) == list(st)
        for k in bad + [off]:
            assert S[k] == T[k] and np.array_equal(V[k], U[k], equal_nan=True), (k, min_chunk, calls)
        if sum(calls) == 24:
            assert np.array_equal(S, T) and all(np.array_equal(V[k], U[k]) for k in good)
    V, S, s2, _ = run(good, 16, [24])
    assert not s2.any() and np.array_equal(S, T[good])
    assert all(np.array_equal(V[i], U[k]) and np.isfinite(U[k]).all() for i, k in enumerate(good))
