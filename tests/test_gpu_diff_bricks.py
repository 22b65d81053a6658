"""The differentiable box's particle phase by bricks, at the sizes where its
layout changes: sides shorter than a brick, ragged sides, bricks of 4 and of 8
cells, every length of a particle block, boxes whose bricks take their particles
through a list or are split over workgroups, moves longer than a cell, and
particles outside the box.  FP64 against the PyTorch PIC and its autograd (bars of
test_gpu_diff.py: 1e-12 forward, 1e-9 adjoint; FP32 boxes in these layouts:
test_gpu_ensemble.py).  Where a layout once made boxes of some shape slow, their
time is held against a like box that it suits."""

import numpy as np
import pytest
import torch

import torch_pic as tp
from runko_amd.diff import DiffBox, DiffEnsemble
from test_torch_pic import M, Q

pytestmark = pytest.mark.gpu

DEV = "cuda"


def rel(a, b):
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


def random_state(n, counts, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    E, B = (0.05 * torch.randn((3,) + n, generator=g, device=DEV, dtype=torch.float64) for _ in range(2))
    hi = torch.tensor(n, device=DEV, dtype=torch.float64).view(3, 1)
    x = torch.rand((3, sum(counts)), generator=g, device=DEV, dtype=torch.float64) * hi
    u = 1.5 * torch.randn((3, sum(counts)), generator=g, device=DEV, dtype=torch.float64)
    return E, B, x, u


@pytest.mark.parametrize("n, counts, cfl", [
    ((2, 3, 5), (40, 23), 0.45),            # sides shorter than a brick: windows wrap onto themselves
    ((2, 5, 700), (300, 200), 0.45),        # nodes in three windows; rows shared by three workgroups
    ((4, 4, 3), (9000, 8001), 0.45),        # one brick, split over 16 workgroups
    ((8, 7, 5), (20000, 20001), 1.4),       # 8 bricks split over 4, moves beyond the neighbouring cell
    ((5, 9, 17), (700, 901), 0.45),         # ragged bricks of at most 4 cells, 7 blocks of 256 particles
    ((6, 5, 9), (257, 1), 1.4),             # moves beyond the neighbouring cell
    ((41, 18, 20), (70001, 70000), 0.45),   # blocks of 1024 particles
    ((57, 66, 71), (530000, 530001), 0.45),  # bricks of at most 8 cells, blocks of 4096 particles
    ((64, 64, 64), (2200000, 2100000), 0.45),  # blocks of 8192 particles
    ((264, 256, 256), (60000, 60000), 0.45),  # listed: sorted by groups of 2^3 bricks
    ((3, 2048, 4096), (60000, 1), 0.45),      # listed: groups of 4^3, bricks of 3 x 8 x 8 cells
])
def test_brick_layouts(n, counts, cfl):
    check_step(n, counts, cfl, random_state(n, counts, seed=sum(n)))


def check_step(n, counts, cfl, s):
    box = DiffBox(n, Q, M, counts, cfl=cfl, dtype=torch.float64)
    q = tp.per_particle(Q, counts, torch.float64, DEV)
    qm = tp.per_particle([np.sign(a) / b for a, b in zip(Q, M)], counts, torch.float64, DEV)
    leaves = tuple(t.clone().requires_grad_(True) for t in s)
    ref = tp.step(*leaves, q, qm, cfl)
    for name, a, b in zip("EBxu", box.step(s), ref):
        assert rel(a, b.detach()) < 1e-12, name
    g = torch.Generator(device=DEV)
    g.manual_seed(3)
    cot = tuple(torch.randn(t.shape, generator=g, device=DEV, dtype=torch.float64) for t in s)
    grad = torch.autograd.grad(ref, leaves, grad_outputs=cot)
    for name, a, b in zip("EBxu", box.step_adjoint(s, cot), grad):
        assert rel(a, b) < 1e-9, name
    assert box.error_count() == 0


def test_listed_particles_in_cell_order():
    # whole waves of one brick's particles, most bricks empty
    n, counts = (264, 256, 256), (40000, 40000)
    E, B, x, u = random_state(n, counts, seed=12)
    x = x * (torch.tensor([[30.0], [20.0], [10.0]], device=DEV) / torch.tensor(n, device=DEV).view(3, 1))
    x = x[:, torch.argsort((x[0].floor() * 20 + x[1].floor()) * 10 + x[2].floor())].contiguous()
    check_step(n, counts, 0.45, (E, B, x, u))


def milliseconds(box, n_particles, n, shape, adjoint=True, passes=4):
    g = torch.Generator(device=DEV)
    g.manual_seed(2)
    hi = torch.tensor(n, device=DEV, dtype=torch.float32).view(3, 1)
    s = (0.05 * torch.randn(shape, generator=g, device=DEV), 0.05 * torch.randn(shape, generator=g, device=DEV),
         (torch.rand((3, n_particles), generator=g, device=DEV) * hi * 0.999999).contiguous(),
         torch.randn((3, n_particles), generator=g, device=DEV))
    out, times = box.empty_state(), []
    for _ in range(passes):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        box.step(s, out)
        if adjoint:
            box.step_adjoint(s, s, out)
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b))
    assert box.error_count() == 0
    return min(times)


def test_long_rows_cost_what_short_rows_cost():
    # a box of 2 x 2 x 4096 cells against the same lying along x: the nodes'
    # three windows in a chain, by four workgroups, took 3.5 times as long
    t = [milliseconds(DiffBox(n, Q, M, (20000, 20000)), 40000, n, (3,) + n, adjoint=False, passes=30)
         for n in ((2, 2, 4096), (4096, 2, 2))]
    assert t[0] < 2 * t[1], t


def test_few_full_bricks_fill_the_chip():
    # 8^3 cells with 1e6 particles against 64^3 with as many: one workgroup a brick
    # took 15 times as long
    t = [milliseconds(DiffBox(n, Q, M, (500000, 500000)), 1000000, n, (3,) + n, passes=8) for n in ((8, 8, 8), (64, 64, 64))]
    assert t[0] < 3 * t[1], t


def test_many_bricks_cost_what_their_parts_cost():
    # a box of 262144 bricks against 16 boxes of 16384 with the same cells and
    # particles in all: walking the runs of groups of 4^3 bricks took 2.6 times
    # as long (61 against 24 ms), the list takes 1.1 times
    whole, part, k = (2, 4096, 4096), (2, 1024, 1024), 1 << 24
    one = milliseconds(DiffBox(whole, Q, M, (k, k)), 2 * k, whole, (3,) + whole)
    parts = DiffEnsemble([dict(n=part, charges=Q, masses=M, counts=(k // 16, k // 16))] * 16)
    many = milliseconds(parts, 2 * k, part, (3, parts.field_view(parts.empty_state()[0], 0)[0].numel() * 16))
    assert one < 2 * many, (one, many)


def test_filter_rounds_no_more_than_the_27_taps():
    # from zero fields E' is minus the current, filtered or not: three FP32
    # passes against 64 bits, and against the reference's 27 taps a pass in FP32
    n, counts = (40, 36, 44), (60000, 60000)
    E, _, x, u = (t.to(torch.float32) for t in random_state(n, counts, seed=13))
    zero = torch.zeros_like(E)
    J, got = (-DiffBox(n, Q, M, counts, filter_passes=p).step((zero, zero, x, u))[0] for p in (0, 3))
    exact, taps = J.double(), J
    for _ in range(3):
        exact, taps = tp.binomial2(exact), tp.binomial2(taps)
    assert rel(got.double(), exact) <= rel(taps.double(), exact)


def test_segments_several_boxes_away():
    # up to 5.5 cells a step along a side of 2: the current's cells lie up to
    # three sides from the box
    n, counts = (2, 3, 5), (40, 23)
    E, B, x, u = random_state(n, counts, seed=11)
    u[0], u[1:] = 5.0 + u[0].abs(), 0.1 * u[1:]
    check_step(n, counts, 5.5, (E, B, x, u))


def test_particles_outside_the_box_pass_through():
    n, counts = (9, 8, 7), (300, 300)
    E, B, x, u = random_state(n, counts, seed=4)
    inside = DiffBox(n, Q, M, counts, dtype=torch.float64).step((E, B, x, u))
    x2, u2 = (torch.cat([v[:, :300], v[:, :1], v[:, 300:], v[:, -1:]], 1).contiguous() for v in (x, u))
    x2[0, 300], x2[2, 601] = 14.0, float("nan")
    box = DiffBox(n, Q, M, (301, 301), dtype=torch.float64)
    out = box.step((E, B, x2, u2))
    assert box.error_count() == 2
    keep = [i for i in range(602) if i not in (300, 601)]
    assert torch.equal(out[2][:, keep], inside[2]) and torch.equal(out[3][:, keep], inside[3])
    assert rel(out[0], inside[0]) < 1e-12
    assert torch.equal(out[2][:, 300], x2[:, 300]) and torch.equal(out[3][:, 601], u2[:, 601])
    lam = tuple(torch.randn_like(t) for t in (E, B, x2, u2))
    back = box.step_adjoint((E, B, x2, u2), lam)
    for k in (300, 601):
        assert torch.equal(back[2][:, k], lam[2][:, k]) and torch.equal(back[3][:, k], lam[3][:, k])
