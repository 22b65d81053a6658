"""Per-tile readback in id order by one launch against the general path (bin
order copy, library sort, permutation): counts around a workgroup of 256, bins
that are empty, tiles of several bricks, ids above 2^63 and repeated ids.  A
tile whose bins hold more than 8192 slots takes the general path."""

import numpy as np
import pytest
import torch

from gpu_common import build_gpu, random_inputs

pytestmark = pytest.mark.gpu

Q = [-0.02, 0.02]
M = [1.0, 1.0]


@pytest.mark.parametrize("count", [0, 1, 255, 256, 257, 600, 4096])
@pytest.mark.parametrize("n", [(8, 8, 8), (12, 8, 4), (3, 3, 3)])
def test_readback_matches_general_path(n, count):
    nt = (1, 2, 1)
    inputs = random_inputs(nt, n, 2, seed=5, ppc=1)
    rng = np.random.default_rng(count)
    for idx, (F, parts) in inputs.items():
        lo = np.array(idx) * n
        # all in the lower half of the tile: with several bricks some stay empty
        parts[1] = np.concatenate([lo + rng.random((count, 3)) * n * [1, 1, 0.5], rng.standard_normal((count, 3))], 1)
    _, grid, _ = build_gpu(nt, n, Q, M, inputs)
    w = grid.world
    for p in w.pools:  # ids in any order, some equal, some with the top bit set
        g = torch.Generator().manual_seed(count)
        p.id.copy_(torch.randint(-50, 50, p.id.shape, generator=g) * (1 << 56))
    for t, tile in enumerate(grid.tiles()):
        for s in range(2):
            p, v, i = (a.cpu().numpy() for a in tile._particles(s))
            fast = [w.tile_particles_by_id(t, s, k) for k in range(3)]
            if len(i) == 0 and fast[0] is None:  # no bins yet: the general path
                continue
            assert np.array_equal(fast[0], p) and np.array_equal(fast[1], v)
            assert np.array_equal(fast[2], i.view(np.uint64))
            assert np.array_equal(np.stack(tile.get_positions(s)), p) and np.array_equal(tile.get_ids(s), fast[2])


def test_large_tile_takes_the_general_path():
    n = (16, 16, 16)
    _, grid, _ = build_gpu((1, 1, 1), n, Q, M, random_inputs((1, 1, 1), n, 2, seed=6, ppc=3))
    assert grid.world.tile_particles_by_id(0, 0, 0) is None
    assert np.array_equal(np.stack(grid.tiles()[0].get_positions(0)), grid.tiles()[0]._particles(0)[0].cpu().numpy())
