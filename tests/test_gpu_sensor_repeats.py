"""Sensor flags over neighbour tables in which an element is listed more than
once, in any places: two elements across a periodic mesh that is two wide are
neighbours twice, and a caller's table may put the two sides anywhere.

Each element settles by walking the tree of those that point at it; the flags
must be the sequential loop's (every one equal).  Tables: random multigraphs of
small clusters, so that most elements have a repeated neighbour, with random
averages whose jumps lie around the thresholds.
"""
import ctypes

import numpy as np
import pytest
import torch

import dg_amd
import oracle
from dg_amd import MULTIFLUID, ROE, Config
from tests.helpers import small_mesh

pytestmark = pytest.mark.gpu


def _table(rng, n, nn, cluster):
    """nn neighbours an element, each pair listed on both sides; -2 where a side is left over."""
    nb = np.full((n, nn), -2, np.int32)
    for e0 in range(0, n, cluster):
        ends = [(e, k) for e in range(e0, min(n, e0 + cluster)) for k in range(nn)]
        rng.shuffle(ends)
        for (a, i), (b, j) in zip(ends[::2], ends[1::2]):
            if a != b:
                nb[a, i], nb[b, j] = b, a
    return nb


@pytest.mark.parametrize("nn", [2, 3, 4, 6])
def test_flags_with_repeated_neighbours(device, nn):
    lib = dg_amd.lib()
    i, d, b, vp = ctypes.c_int, ctypes.c_double, ctypes.c_bool, ctypes.c_void_p
    lib.dgx_calc_sensors_noalloc.argtypes = [i, i, b, d, b, d, b, d, vp, vp, vp]
    lib.dgx_calc_sensors_noalloc.restype = i
    assert lib.dgx_set_config(ctypes.byref(Config(2, 2, MULTIFLUID, ROE))) == 0
    prob = oracle.Problem(small_mesh(2, 2, MULTIFLUID).tables(), MULTIFLUID, ROE)
    on = np.ones(3, np.int32)
    repeats = 0
    for seed in range(12):
        rng = np.random.default_rng(100 * nn + seed)
        n = 6000 + seed
        nb = _table(rng, n, nn, (3, 5, 7, 9)[seed % 4])
        repeats += sum(len(set(r)) < len(r) for r in nb[nb.min(axis=1) >= 0].tolist())
        rho, p, alpha = (np.exp(rng.normal(0, 0.3, n)) for _ in range(3))
        vx, vy = rng.normal(0, 0.5, n), rng.normal(0, 0.5, n)
        ua = np.stack([rho, rho * vx, rho * vy, p * alpha + 0.5 * rho * (vx * vx + vy * vy), alpha], axis=1).reshape(-1).copy()
        th = np.array([(0.25, 0.2, 0.1), (0.35, 0.1, 0.3), (2.0, 0.05, 2.0), (0.4, 2.0, 2.0)][seed // 3])
        init = (rng.random(n) < 0.1 * (seed % 2)).astype(np.int32)
        c = type(prob.cfg).from_buffer_copy(prob.cfg)
        c.N_E, c.N_N = n, nn
        ref = init.copy()
        vptr = lambda a: a.ctypes.data_as(vp)
        oracle.lib().or_calc_sensors(ctypes.byref(c), vptr(on), vptr(th), vptr(np.ascontiguousarray(nb)), vptr(ua), vptr(ref))
        nbd, uad, sd = (torch.from_numpy(a).to(device) for a in (nb, ua, init))
        assert lib.dgx_calc_sensors_noalloc(n, nn, True, th[0], True, th[1], True, th[2], nbd.data_ptr(), uad.data_ptr(),
                                            sd.data_ptr()) == 0
        got = sd.cpu().numpy()
        assert 0.05 * n < (ref != 0).sum()
        assert np.array_equal(got, ref), (nn, seed, int((got != ref).sum()))
    assert nn == 2 or repeats > 1000
