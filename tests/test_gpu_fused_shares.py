"""Wave shares of the fused particle step: every brick's wave takes a
contiguous share of 64-particle chunks and compacts it in place.  Bricks hold
the particle counts where that can go wrong (none, one, around one chunk,
around one chunk per wave, a remainder past it), three species (odd ones deal
their shares in reverse), and one brick whose particles all leave (more of
them than its 64-record mailbox holds).  The last shape has an odd number of
lattice rows (the gather that follows takes them in pairs).  One lap against the oracle with the
bars of the other one-lap tests: particles bit-exact, fields within 1e-6."""

import numpy as np
import pytest

from gpu_common import build_gpu, build_oracle, canonical_lap, gpu_fields, gpu_particles, oracle_particles
from helpers import rel_err

pytestmark = pytest.mark.gpu

Q = [-0.02, 0.02, 0.01]
M = [1.0, 1.0, 3.0]
COUNTS = [0, 1, 63, 64, 65, 511, 512, 513, 577]


def share_inputs(nt, n, brick, seed):
    rng = np.random.default_rng(seed)
    nb = [a // b for a, b in zip(n, brick)]
    tiles, at = {}, 0
    for idx in np.ndindex(*nt):
        F = np.zeros((9,) + tuple(n))
        F[0:6] = 0.05 * rng.standard_normal((6,) + tuple(n))
        parts = [[] for _ in Q]
        for lb in np.ndindex(*nb):
            lo = np.array(idx) * n + np.array(lb) * brick
            for s in range(len(Q)):
                k = COUNTS[(at + 2 * s) % len(COUNTS)]
                pos = lo + rng.random((k, 3)) * brick
                u = (rng.random((k, 3)) * 2 - 1) * 1.5
                if at == 4 and s == 0:  # all leave across the upper x face
                    pos[:, 0] = lo[0] + brick[0] - 0.01
                    u[:, 0] = 2.0
                parts[s].append(np.concatenate([pos, u], 1))
            at += 1
        tiles[idx] = (F, [np.concatenate(p) for p in parts])
    return tiles


@pytest.mark.parametrize("n,brick", [((8, 8, 16), (8, 8, 8)), ((4, 4, 8), (4, 4, 4)), ((6, 7, 10), (6, 7, 5)),
                                     ((5, 7, 10), (5, 7, 5))])
@pytest.mark.parametrize("pusher", ["boris", "higuera_cary", "faraday"])
def test_one_lap_parity_share_edges(orc, n, brick, pusher):
    nt = (3, 3, 1)
    inputs = share_inputs(nt, n, brick, seed=91)
    conf, grid, sim = build_gpu(nt, n, Q, M, inputs, execution="batched", pusher=pusher, brick_shape=brick)
    assert tuple(grid.world.brick) == brick
    w = build_oracle(orc, nt, n, Q, M, inputs, pusher=pusher)
    sim.for_one_lap(canonical_lap(sim))
    w.lap(0)
    for s in range(len(Q)):
        tg, sg, ig = gpu_particles(grid, s)
        to, so, io = oracle_particles(w, s)
        assert np.array_equal(ig, io), s
        assert np.array_equal(tg, to), s
        assert np.array_equal(sg, so), s
    g, o = gpu_fields(grid), w.global_fields()
    assert rel_err(g[0:3], o[0:3]) < 1e-6
    assert rel_err(g[6:9], o[6:9]) < 1e-6


def test_timed_step_takes_the_same_work_under_its_categories():
    # the appends and the gather of the currents share a launch unless kernels
    # are timed; a cold plasma of a particle per cell has few leavers, so the
    # gather takes the longer
    import torch
    from runko_amd import _lib as L
    from runko_amd.init import turbulence_world
    from runko_amd.stepper import BatchedLap

    worlds = [turbulence_world(N=128, tile=32, ppc=1, theta=1e-4, sigma=1e-4, seed=3)[0] for _ in range(2)]
    laps = [BatchedLap(w) for w in worlds]
    ms, cnt = np.zeros((2, 9)), np.zeros(9, dtype=np.int64)
    for rep in range(2):
        for timed, (w, lap) in enumerate(zip(worlds, laps)):
            L.check(L.lib().rk_profile_enable(w.h, timed))
            lap()
            lap.settle()
            if timed:
                L.check(L.lib().rk_profile_read(w.h, ms[rep].ctypes.data, cnt.ctypes.data))
                L.check(L.lib().rk_profile_enable(w.h, 0))
        assert torch.equal(worlds[0].F, worlds[1].F)
        assert worlds[0].total_particles() == worlds[1].total_particles()
    deposit, append = (dict(zip(L.PROF_CATEGORIES, ms.min(0)))[k] for k in ("deposit", "append"))
    assert deposit > append > 0, (deposit, append)
