"""The batched updates that leave the ghost shell current (half B push, E push
with the current, current exchange) against the update followed
by the separate ghost exchanges, whole haloed lattices bit for bit.  Shapes:
more rows than one workgroup covers, exactly 2 * HALO cells along an axis
(every node has an image), one cell more, and fewer (the separate launches)."""

import numpy as np
import pytest
import torch

from gpu_common import build_gpu, random_inputs
from runko_amd.tools import comm_mode

pytestmark = pytest.mark.gpu

Q = [-0.02, 0.02]
M = [1.0, 1.0]
SHAPES = [((2, 2, 2), (8, 9, 37)), ((1, 1, 1), (6, 6, 6)), ((1, 1, 1), (7, 6, 13)), ((1, 2, 1), (6, 11, 70)),
          ((1, 1, 1), (4, 5, 8)), ((1, 1, 1), (3, 9, 9))]


def pair(nt, n, seed):
    """Two worlds with the same fields, ghost shells included (noise: nothing is current)."""
    ws = []
    for _ in range(2):
        _, grid, _ = build_gpu(nt, n, Q, M, random_inputs(nt, n, 2, seed=seed, ppc=1), execution="batched")
        g = torch.Generator().manual_seed(seed)
        grid.world.F.copy_(torch.randn(grid.world.F.shape, generator=g).to(grid.world.F))
        ws.append(grid)
    return ws


def same(a, b):
    return all(torch.equal(getattr(a, f), getattr(b, f)) for f in ("E", "B", "J"))


@pytest.mark.parametrize("nt,n", SHAPES)
def test_updates_leave_ghosts_current(nt, n):
    a, b = (g.world for g in pair(nt, n, 31))
    for w in (a, b):
        w.comm_local(int(comm_mode.emf_E))
    a.call("rk_push_half_b", -1)
    a.comm_local(int(comm_mode.emf_B))
    b.push_half_b_comm()
    assert same(a, b)
    a.call("rk_push_e_add_current", -1)
    a.comm_local(int(comm_mode.emf_E))
    b.push_e_add_current_comm()
    assert same(a, b)
    a.comm_local(int(comm_mode.emf_J_exchange))
    a.comm_local(int(comm_mode.emf_J))
    b.exchange_current()
    assert same(a, b)


@pytest.mark.parametrize("nt,n", SHAPES)
def test_fold_matches_the_images(nt, n):
    # interior node += its periodic images, x offsets slowest, the own node
    # first, then the image below, then the one above: in float32 on the host
    a = pair(nt, n, 32)[0].world
    J = a.J.cpu().numpy().copy()
    N = np.array(J.shape[1:]) - 6
    a.comm_local(int(comm_mode.emf_J_exchange))
    got = a.J.cpu().numpy()

    def images(c, m):
        return [c] + ([c - m] if c >= m else []) + ([c + m] if c < 6 else [])

    want = J.copy()
    for i in range(3, N[0] + 3):
        for j in range(3, N[1] + 3):
            edge = len(images(i, N[0])) * len(images(j, N[1])) > 1
            for k in range(3, N[2] + 3) if edge else [c for c in range(3, N[2] + 3) if c < 6 or c >= N[2]]:
                s = J[:, i, j, k].copy()
                for x in images(i, N[0]):
                    for y in images(j, N[1]):
                        for z in images(k, N[2]):
                            if (x, y, z) != (i, j, k):
                                s = s + J[:, x, y, z]
                want[:, i, j, k] = s
    assert np.array_equal(got, want)
