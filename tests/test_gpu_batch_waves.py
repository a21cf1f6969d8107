"""Ensembles on both sides of the line from which workgroups of up to 128
threads run two to a SIMD (1024 waves): the bits of the same problems in
workgroups of 256 threads, which take neither of the two instances, for state,
time and status, with a problem that stops among them."""
import numpy as np
import pytest
import torch

from dg_amd import FARFIELD, MULTIFLUID, RUSANOV, SINGLEFLUID, Batch, Config, Mesh, nfields, problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ph", [SINGLEFLUID, MULTIFLUID])
@pytest.mark.parametrize("block,n", [(128, 512), (128, 513), (64, 1024), (64, 1025)])
def test_both_instances(device, ph, block, n):
    orders = [1 + k % 3 for k in range(n)]
    ne = [8 + (7 * k) % 23 for k in range(n)]  # one workgroup each
    meshes = {(p, m): Mesh(1, p, m, 1, -1.0, 1.0, bc=(FARFIELD, FARFIELD), nfields=nfields(1, ph))
              for p, m in set(zip(orders, ne))}
    states = [problems.smooth_random_state(meshes[p, m], ph, seed=k % 50) for k, (p, m) in enumerate(zip(orders, ne))]
    bad = n - 2
    states[bad] = states[bad].copy()
    states[bad].reshape(ne[bad], nfields(1, ph), -1)[:, 2] *= -1.0
    batch = Batch(Config(1, 1, ph, RUSANOV), ne, orders)
    out = []
    for b in (block, 256):
        batch.set_block_sizes([b])
        assert batch.block_sizes[1:] == [n, 0]
        U = torch.from_numpy(batch.pack(states)).to(device)
        T = torch.zeros(n, dtype=torch.float64, device=device)
        st = torch.zeros(n, dtype=torch.int32, device=device)
        batch.rk4(U, 0.3, 5, T, st)
        torch.cuda.synchronize()
        out.append((U.cpu().numpy(), T.cpu().numpy(), st.cpu().numpy()))
    (Ua, Ta, sa), (Ub, Tb, sb) = out
    assert np.array_equal(sa, sb) and np.array_equal(Ta, Tb) and np.array_equal(Ua, Ub, equal_nan=True)
    assert sa[bad] == 1 and sa.sum() == 1 and (np.delete(Ta, bad) > 0).all()
