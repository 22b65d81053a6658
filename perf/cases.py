"""What the framework's speed is measured on.

Twelve cases of what users run through the public entry points: laps of the
particle-in-cell world in its three forms (per tile through Simulation,
batched, replayed from HIP graphs), the reflecting-wall shock with the schemes
of its reference configuration, the differentiable box forward, backward and
as a rollout, the ensemble, and the diagnostics that are written every few
laps.  Sizes are those of the repository's benchmark, tests and workloads
where they fit the card three times over, else smaller or ragged ones.

A world keeps the particles of a bin in no defined order, so the laps return
their fields (which the particles' moves and currents make); the per-tile lap
returns its particles too, tile by tile in id order.

`exact` restates the step in float64 with plain torch.
"""

import math

import numpy as np
import torch

import runko_amd as runko
from runko_amd import _lib as L
from runko_amd import diff, workloads
from runko_amd.snapshots import MpiioFieldsWriter, MpiioSpectraWriter
from runko_amd.stepper import BatchedLap, GraphLap, ShockLap
from runko_amd.tiles import stencil_from_config
from runko_amd.world import HALO, World

CFL = 0.45
C_OMP = 10.0  # cells per skin depth
DEV = "cuda"

# the extended-stencil coefficients of the reference's 3D shock configuration
# (projects/pic-shock/3d_shock.ini:48-70)
SHOCK_STENCIL = {
    "stencil_x_delta": -0.13512912586798165, "stencil_x_gamma": 0.016100341594971104,
    "stencil_x_beta_p1": 0.022350417588794424, "stencil_x_beta_p2": 0.022350417588794424,
    "stencil_x_zeta_p1": 0.012206124727660462, "stencil_x_zeta_p2": 0.012206124727660462,
    "stencil_y_delta": 0.010144292861133962, "stencil_y_gamma": 0.012206124727660462,
    "stencil_y_beta_p1": 0.022350417588794424, "stencil_y_beta_p2": -0.11902878427301054,
    "stencil_y_zeta_p1": 0.012206124727660462, "stencil_y_zeta_p2": 0.016100341594971104,
    "stencil_z_delta": 0.010144292861133962, "stencil_z_gamma": 0.012206124727660462,
    "stencil_z_beta_p1": -0.11902878427301054, "stencil_z_beta_p2": 0.022350417588794424,
    "stencil_z_zeta_p1": 0.016100341594971104, "stencil_z_zeta_p2": 0.012206124727660462,
}


def listed():
    return [
        # a driver that runs the drop-in per-tile form and reads every particle
        # back after a lap, on the grid of the smoke test
        dict(name="sim_plain_16", kind="sim", n0=8, n1=8, n2=8, t0=2, t1=2, t2=2, ppc=4, theta=0.3, sigma=1.0),
        # the 64^3 pair plasma of the benchmark, replayed from graphs: launches count
        dict(name="pair_graph_64", kind="world", form="graph", n0=16, n1=16, n2=16, t0=4, t1=4, t2=4, ppc=8,
             theta=0.3, sigma=1.0, pusher="boris", filt="binomial2"),
        # decaying turbulence in 32^3 tiles, the largest world that fits three times
        dict(name="turbulence_graph_256", kind="world", form="graph", n0=32, n1=32, n2=32, t0=8, t1=8, t2=8, ppc=16,
             theta=0.3, sigma=10.0, pusher="boris", filt="binomial2"),
        # tiles that no cube of eight divides, the other pusher and the unrolled filter, eager
        dict(name="ragged_batched", kind="world", form="batched", n0=12, n1=10, n2=14, t0=5, t1=4, t2=3, ppc=6,
             theta=1.0, sigma=3.0, pusher="higuera_cary", filt="binomial2_unrolled"),
        # the reflecting-wall shock with the schemes of its configuration
        dict(name="shock_graph_512", kind="shock", n0=32, n1=32, n2=32, t0=16, t1=2, t2=2, ppc=8, theta=1e-4,
             sigma=0.1, gamma=10.0),
        # one forward step of the differentiation workload after a long rollout:
        # the particles keep their places in the arrays and have mixed over the box
        dict(name="diff_step_96", kind="diff", what="step", n0=96, n1=96, n2=96, ppc=16, theta=0.3, double=False,
             mixed=True),
        # the adjoint of that step
        dict(name="diff_adjoint_96", kind="diff", what="adjoint", n0=96, n1=96, n2=96, ppc=16, theta=0.3,
             double=False, mixed=True),
        # the first steps of a rollout, whose particles still lie cell by cell
        dict(name="diff_step_cells_64", kind="diff", what="step", n0=64, n1=64, n2=64, ppc=8, theta=0.3,
             double=False, mixed=False),
        # double precision on a ragged box, forward and adjoint
        dict(name="diff_double_ragged", kind="diff", what="both", n0=45, n1=38, n2=51, ppc=4, theta=1.0, double=True,
             mixed=True),
        # the gradient of a short rollout of a small box, as an optimiser calls it: launches count
        dict(name="rollout_16", kind="rollout", sides="16", ppcs="2", theta=0.3, steps=8, every=4),
        # boxes of an ensemble stepped and differentiated together
        dict(name="ensemble_rollout", kind="rollout", sides="32,48,64,32,48", ppcs="8,4,4,16,8", theta=1.0, steps=3,
             every=2),
        # what a driver writes every few laps: fields, spectra and energies
        dict(name="diagnostics_64", kind="diagnostics", n0=16, n1=16, n2=16, t0=4, t1=4, t2=4, ppc=8, theta=0.3,
             stride=2, nbins=128),
    ]


# sides of tiles that no brick of eight cells divides
RAGGED = (6, 7, 9, 10, 12, 14, 15, 18, 20, 21, 25)


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sim", "world", "world", "world", "shock", "diff", "diff", "diff", "rollout", "diagnostics"])
    theta = round(math.exp(rng.uniform(math.log(0.05), math.log(3.0))), 4)
    sigma = round(math.exp(rng.uniform(math.log(0.1), math.log(10.0))), 4)
    if kind == "sim":
        n, t = [rng.choice(RAGGED) for _ in range(3)], [rng.randint(2, 3) for _ in range(3)]
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], t0=t[0], t1=t[1], t2=t[2], ppc=rng.randint(1, 8),
                    theta=theta, sigma=sigma)
    if kind == "world":
        # tiles of 8^3 to 32^3 cells, cubes of eight or ragged, 2^3 to 6^3 of them
        n = [rng.choice([8, 16, 24, 32])] * 3 if rng.random() < 0.6 else [rng.choice(RAGGED) for _ in range(3)]
        t = [rng.randint(2, 6) for _ in range(3)]
        return dict(kind=kind, form=rng.choice(["graph", "graph", "batched"]), n0=n[0], n1=n[1], n2=n[2], t0=t[0],
                    t1=t[1], t2=t[2], ppc=_log(rng, 2, 16), theta=theta, sigma=sigma,
                    pusher=rng.choice(["boris", "boris", "higuera_cary", "faraday"]),
                    filt=rng.choice(["binomial2", "binomial2", "binomial2_unrolled"]))
    if kind == "shock":
        return dict(kind=kind, n0=32, n1=32, n2=32, t0=rng.randint(3, 16), t1=rng.randint(1, 2),
                    t2=rng.randint(1, 2), ppc=rng.randint(2, 8), theta=1e-4, sigma=round(rng.uniform(0.05, 1.0), 3),
                    gamma=round(rng.uniform(3.0, 12.0), 2))
    if kind == "diff":
        double = rng.random() < 0.25
        hi = 56 if double else 88
        n = [_log(rng, 8, hi) for _ in range(3)]
        return dict(kind=kind, what=rng.choice(["step", "adjoint", "both"]), n0=n[0], n1=n[1], n2=n[2],
                    ppc=_log(rng, 1, 16), theta=theta, double=double, mixed=rng.random() < 0.6)
    if kind == "rollout":
        m = rng.randint(1, 6)
        return dict(kind=kind, sides=",".join(str(_log(rng, 10, 48)) for _ in range(m)),
                    ppcs=",".join(str(rng.choice([2, 4, 8])) for _ in range(m)), theta=theta, steps=rng.randint(2, 4),
                    every=rng.randint(1, 3))
    n, t = 2 * rng.randint(4, 12), [rng.randint(2, 4) for _ in range(3)]
    return dict(kind="diagnostics", n0=n, n1=n, n2=n, t0=t[0], t1=t[1], t2=t[2], ppc=rng.randint(1, 12), theta=theta,
                stride=rng.choice([1, 2]), nbins=rng.choice([64, 100, 200]))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _momenta(n, theta, gen):
    """Isotropic relativistic Maxwellian momenta [3, n] float64, the magnitude
    by the tabulated inverse of the distribution's cumulative."""
    umax = math.sqrt((1.0 + 30.0 * theta) ** 2 - 1.0)
    u = torch.linspace(0, umax, 16384, dtype=torch.float64, device=DEV)
    f = u * u * torch.exp((1.0 - torch.sqrt(1 + u * u)) / theta)
    c = torch.cumsum(f, 0)
    c = c / c[-1]
    r = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)
    i = torch.searchsorted(c, r).clamp_(1, u.numel() - 1)
    m = u[i - 1] + (r - c[i - 1]) / (c[i] - c[i - 1]).clamp_min(1e-30) * (u[i] - u[i - 1])
    z = 2 * torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) - 1
    p = 2 * math.pi * torch.rand(n, generator=gen, device=DEV, dtype=torch.float64)
    s = m * torch.sqrt(1 - z * z)
    return torch.stack([s * torch.cos(p), s * torch.sin(p), m * z])


def _in_cells(cells, gen):
    """float32 positions uniform in the given cells ([3, k] float64)."""
    pos = (cells + torch.rand(cells.shape, generator=gen, device=DEV, dtype=torch.float64)).to(torch.float32)
    top = (cells + 1).to(torch.float32)
    return torch.where(pos >= top, torch.nextafter(top, torch.zeros_like(top)), pos)


def _cells(lo, n, ppc):
    g = torch.meshgrid(*(torch.arange(l, l + v, device=DEV, dtype=torch.float64) for l, v in zip(lo, n)), indexing="ij")
    return torch.stack([v.reshape(-1) for v in g]).repeat_interleave(ppc, 1)


def _plasma(c, gamma=1.0):
    """(charges, guide field) of the turbulence and shock drivers."""
    ppc, theta = c["ppc"], c["theta"]
    q = (CFL / C_OMP) ** 2 * gamma / (2 * ppc)
    if gamma > 1.0:
        return [-q, q], CFL * math.sqrt(gamma * 2 * ppc * q * c["sigma"])
    return [-q, q], math.sqrt((1 + 1.5 * theta) * 2 * ppc * q * CFL ** 2 * c.get("sigma", 1.0))


def _shape(c):
    n, t = [c["n0"], c["n1"], c["n2"]], [c["t0"], c["t1"], c["t2"]]
    return n, t, [a * b for a, b in zip(n, t)]


def _waves(N, amp, gen):
    """Bx, By of a few waves of a vector potential along z, rms amp."""
    k = torch.randint(1, 5, (6, 2), generator=gen, device=DEV).to(torch.float64) * 2 * math.pi
    ph = 2 * math.pi * torch.rand(6, generator=gen, device=DEV, dtype=torch.float64)
    X = torch.arange(N[0] + 1, device=DEV, dtype=torch.float64).view(-1, 1) / N[0]
    Y = torch.arange(N[1] + 1, device=DEV, dtype=torch.float64).view(1, -1) / N[1]
    A = sum(torch.cos(k[m, 0] * X + k[m, 1] * Y + ph[m]) for m in range(6))
    bx, by = A[:-1, 1:] - A[:-1, :-1], A[:-1, :-1] - A[1:, :-1]
    s = amp / torch.sqrt((bx ** 2 + by ** 2).mean())
    return (s * bx).to(torch.float32), (s * by).to(torch.float32)


def _fields(c, gen):
    """float32 E, B [3, *N] of a periodic world."""
    N = _shape(c)[2]
    B0 = _plasma(c)[1]
    E = torch.zeros([3] + N, device=DEV)
    B = torch.zeros([3] + N, device=DEV)
    bx, by = _waves(N, 0.5 * B0, gen)
    B[0], B[1], B[2] = bx[:, :, None], by[:, :, None], float(B0)
    ex, ey = _waves(N, 0.1 * B0, gen)
    E[0], E[1] = ex[:, :, None], ey[:, :, None]
    return E, B


def _tiles(c, seed):
    """Tile by tile: (index, positions, momenta of each species), float32."""
    n, t, _ = _shape(c)
    for k in range(t[0] * t[1] * t[2]):
        g = _gen(seed * 1_000_003 + 17 * k + 5)
        i = (k // (t[1] * t[2]), k // t[2] % t[1], k % t[2])
        pos = _in_cells(_cells([a * b for a, b in zip(i, n)], n, c["ppc"]), g)
        perm = torch.randperm(pos.shape[1], generator=g, device=DEV)
        pos = pos[:, perm].contiguous()
        yield i, pos, [_momenta(pos.shape[1], c["theta"], g).to(torch.float32) for _ in range(2)]


WALL = 15.0


def _shock_fields(c):
    N = _shape(c)[2]
    B0, beta = _plasma(c, c["gamma"])[1], math.sqrt(1 - 1 / c["gamma"] ** 2)
    E, B = torch.zeros([3] + N, device=DEV), torch.zeros([3] + N, device=DEV)
    E[1], B[2] = float(-beta * B0), float(B0)
    return E, B


def _shock_tiles(c, seed):
    """The cold flow along -x in front of the wall."""
    gam = c["gamma"]
    beta = math.sqrt(1 - 1 / gam ** 2)
    for i, pos, us in _tiles(c, seed):
        keep = pos[0] >= WALL
        out = []
        for u in us:
            u = u.double()
            u[0] = -gam * (beta * torch.sqrt(1 + (u * u).sum(0)) - u[0])
            out.append(u[:, keep].to(torch.float32).contiguous())
        yield i, pos[:, keep].contiguous(), out


def _world(c, tiles, E, B, charges, filt, pusher, stencil=None):
    n, t, N = _shape(c)
    w = World(n, t, (0, 0, 0), t, periodic=True, cfl=CFL, charges=charges, masses=[1.0, 1.0], current_filter=filt)
    if pusher != "boris" or stencil is not None:
        w.set_schemes(pusher, stencil)
    inner = (slice(None),) + tuple(slice(HALO, HALO + v) for v in N)
    w.F[0][inner], w.F[1][inner] = E, B
    per_tile = n[0] * n[1] * n[2] * c["ppc"]
    per_brick = w.brick[0] * w.brick[1] * w.brick[2] * c["ppc"]
    w.ensure_migration(max(1 << 16, per_tile, int(0.12 * 2 * per_tile * w.ntiles)))
    w.presize_all({s: np.full(w.nbricks, per_brick, dtype=np.int64) for s in range(2)})
    for k, (_, pos, us) in enumerate(tiles):
        ids = (k << 40) + torch.arange(pos.shape[1], device=DEV)
        for s in range(2):
            w.inject(k, s, pos, us[s], ids)
    w.comm_local(int(runko.tools.comm_mode.emf_E))
    w.comm_local(int(runko.tools.comm_mode.emf_B))
    w.ensure_mailbox()
    return w


def _box_state(c, seed, dtype):
    """E, B, x, u of a differentiable box, as float32 values in dtype."""
    n = [c["n0"], c["n1"], c["n2"]]
    g = _gen(seed)
    charges, B0 = _plasma(c)
    np_ = n[0] * n[1] * n[2] * c["ppc"]
    bx, by = _waves(n, 0.5 * B0, g)
    B = torch.zeros([3] + n, device=DEV)
    B[0], B[1], B[2] = bx[:, :, None], by[:, :, None], float(B0)
    E = (0.1 * B0 * torch.randn([3] + n, generator=g, device=DEV)).to(torch.float32)
    xs = []
    for _ in range(2):
        if c.get("mixed"):
            hi = torch.tensor(n, device=DEV, dtype=torch.float32).view(3, 1)
            x = torch.rand((3, np_), generator=g, device=DEV) * hi
            x = torch.where(x >= hi, torch.zeros_like(x), x)
        else:
            x = xs[0] if xs else _in_cells(_cells([0, 0, 0], n, c["ppc"]), g)
        xs.append(x)
    x = torch.cat(xs, 1)
    u = torch.cat([_momenta(np_, c["theta"], g) for _ in range(2)], 1).to(torch.float32)
    return charges, np_, [v.to(dtype).contiguous() for v in (E, B, x, u)]


def _box_adjoint(state, seed):
    g = _gen(seed + 77)
    return [torch.randn(v.shape, generator=g, device=DEV, dtype=torch.float32).to(v.dtype) for v in state]


def _boxes(c):
    return [dict(n0=int(s), n1=int(s), n2=int(s), ppc=int(p), theta=c["theta"], mixed=False)
            for s, p in zip(c["sides"].split(","), c["ppcs"].split(","))]


# ---------------------------------------------------------------- the cases
def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "sim":
        E, B = _fields(c, _gen(seed))
        E, B = E.cpu().double().numpy(), B.cpu().double().numpy()
        n, t, _ = _shape(c)
        inputs = {}
        for i, pos, us in _tiles(c, seed):
            sl = (slice(None),) + tuple(slice(a * b, (a + 1) * b) for a, b in zip(i, n))
            inputs[i] = (np.concatenate([E[sl], B[sl], np.zeros([3] + n)]),
                         [torch.cat([pos, u]).t().double().cpu().numpy() for u in us])
        conf, grid, sim = workloads.build_simulation(tuple(t), tuple(n), _plasma(c)[0], [1.0, 1.0], inputs,
                                                     execution="plain")
        return dict(case=c, grid=grid, sim=sim, lap=workloads.turbulence_lap(sim, sort_every=0))
    if kind == "world":
        E, B = _fields(c, _gen(seed))
        w = _world(c, _tiles(c, seed), E, B, _plasma(c)[0], c["filt"], c["pusher"])
        return dict(case=c, w=w, lap=GraphLap(w) if c["form"] == "graph" else BatchedLap(w))
    if kind == "shock":
        E, B = _shock_fields(c)
        N = _shape(c)[2]
        w = _world(c, _shock_tiles(c, seed), E, B, _plasma(c, c["gamma"])[0], "binomial2_unrolled", "faraday",
                   stencil_from_config(SHOCK_STENCIL))
        ey, bz = float(E[1, 0, 0, 0]), float(B[2, 0, 0, 0])
        zero = (0.0, 0.0, 0.0)
        walls = [L.ReflectorWall(WALL, 0.0, 1.0)]
        bcs = [L.EdgeBC(0, 0, WALL, zero, zero, zero, 0b110, 0, 0b111),
               L.EdgeBC(0, 1, float(N[0] - 5), (0.0, ey, 0.0), (0.0, 0.0, bz), zero, 0b111, 0b111, 0b111)]
        lap = ShockLap(w, walls, bcs)
        lap()  # a graph of the lap is captured after one eager lap
        lap.settle()
        return dict(case=c, w=w, lap=GraphLap(w, lap=lap))
    if kind == "diff":
        dtype = torch.float64 if c["double"] else torch.float32
        charges, np_, state = _box_state(c, seed, dtype)
        box = diff.DiffBox((c["n0"], c["n1"], c["n2"]), charges, [1.0, 1.0], [np_, np_], cfl=CFL, dtype=dtype)
        s = dict(case=c, box=box, state=tuple(state))
        if c["what"] != "adjoint":
            s["out"] = box.empty_state()
        if c["what"] != "step":
            s["adj"] = tuple(_box_adjoint(state, seed))
            s["back"] = box.empty_state()
        return s
    if kind == "rollout":
        boxes, parts = [], []
        for k, b in enumerate(_boxes(c)):
            charges, np_, state = _box_state(b, seed + 1009 * k, torch.float32)
            boxes.append(dict(n=(b["n0"],) * 3, charges=charges, masses=[1.0, 1.0], counts=[np_, np_]))
            parts.append([state[0].reshape(3, -1), state[1].reshape(3, -1), state[2], state[3]])
        if len(boxes) == 1:
            b = boxes[0]
            box = diff.DiffBox(b["n"], b["charges"], b["masses"], b["counts"], cfl=CFL)
            state = [v.reshape((3,) + b["n"]) if i < 2 else v for i, v in enumerate(parts[0])]
        else:
            box = diff.DiffEnsemble(boxes, cfl=CFL)
            state = [torch.cat([p[i] for p in parts], 1).contiguous() for i in range(4)]
        return dict(case=c, box=box, state=[v.requires_grad_() for v in state])
    if kind == "diagnostics":
        E, B = _fields(dict(c, sigma=1.0), _gen(seed))
        g = _gen(seed + 3)
        E = 0.3 * torch.randn(E.shape, generator=g, device=DEV)
        J = 0.1 * torch.randn(E.shape, generator=g, device=DEV)
        e, b, j = (v.cpu().double().numpy() for v in (E, B, J))
        n, t, _ = _shape(c)
        inputs = {}
        for i, pos, us in _tiles(c, seed):
            sl = (slice(None),) + tuple(slice(p * q, (p + 1) * q) for p, q in zip(i, n))
            inputs[i] = (np.concatenate([e[sl], b[sl], j[sl]]),
                         [torch.cat([pos, u]).t().double().cpu().numpy() for u in us])
        conf, grid, sim = workloads.build_simulation(tuple(t), tuple(n), _plasma(c)[0], [1.0, 1.0], inputs)
        dims = (t[0], n[0], t[1], n[1], t[2], n[2])
        return dict(case=c, grid=grid, fields=MpiioFieldsWriter("", *dims, stride=c["stride"]),
                    spectra=MpiioSpectraWriter("", *dims, stride=c["stride"], nbins=c["nbins"], umin=1e-3, umax=1e2))
    raise ValueError(kind)


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "sim":
        state["sim"].for_one_lap(state["lap"])
        out = dict(pos=[], vel=[])
        for s in range(2):
            tiles = state["grid"].tiles()
            out["pos"].append(np.concatenate([np.stack(t.get_positions(s)) for t in tiles], 1))
            out["vel"].append(np.concatenate([np.stack(t.get_velocities(s)) for t in tiles], 1))
        w = state["grid"].world
        return dict(out, E=w.E, B=w.B)
    if kind in ("world", "shock"):
        state["lap"]()
        state["lap"].settle()
        return dict(E=state["w"].E, B=state["w"].B)
    if kind == "diff":
        box, out = state["box"], {}
        if "out" in state:
            out["step"] = box.step(state["state"], state["out"])
        if "adj" in state:
            out["adjoint"] = box.step_adjoint(state["state"], state["adj"], state["back"])
        return out
    if kind == "rollout":
        E, B, x, u = state["state"]
        for v in state["state"]:
            v.grad = None
        end = diff.rollout(state["box"], E, B, x, u, c["steps"], c["every"])
        (0.5 * (end[1].double() ** 2).sum()).backward()
        return dict(end=[v.detach() for v in end], grad=[v.grad for v in state["state"]])
    return dict(fields=state["fields"].pack(state["grid"]), spectra=state["spectra"].pack(state["grid"]),
                energies=state["grid"].world.energies())


def work(case):
    """Positions and momenta read and written once, and per cell the fields:
    E and B read and written, the current made, filtered and taken."""
    c, kind = case, case["kind"]
    if kind == "rollout":
        b = _boxes(c)
        cells = sum(v["n0"] ** 3 for v in b)
        parts = sum(2 * v["ppc"] * v["n0"] ** 3 for v in b)
        # each step forward, again from its checkpoint, and its adjoint
        passes = 3 * c["steps"]
        return dict(bytes=passes * (48.0 * parts + 96.0 * cells), flops=c["steps"] * (2 * 500.0 + 1500.0) * parts)
    if kind == "diff":
        cells = c["n0"] * c["n1"] * c["n2"]
        parts = 2 * c["ppc"] * cells
        item = 2 if c["double"] else 1
        f, a = c["what"] != "adjoint", c["what"] != "step"
        return dict(bytes=item * (f * (48.0 * parts + 48.0 * cells) + a * (72.0 * parts + 72.0 * cells)),
                    flops=(f * 500.0 + a * 1500.0) * parts)
    N = _shape(c)[2]
    cells = N[0] * N[1] * N[2]
    parts = 2 * c["ppc"] * cells
    if kind == "diagnostics":
        out = cells // c["stride"] ** 3
        return dict(bytes=36.0 * cells + 24.0 * parts + 44.0 * out, flops=40.0 * parts + 30.0 * cells)
    return dict(bytes=48.0 * parts + 228.0 * cells, flops=500.0 * parts + 150.0 * cells)


# ---------------------------------------------------------------- float64
def _sh(F, axis, off):
    return torch.roll(F, -off, axis)


def _curl_e(E):
    d = lambda F, a: _sh(F, a, 1) - F  # noqa: E731
    return torch.stack([d(E[1], 2) - d(E[2], 1), d(E[2], 0) - d(E[0], 2), d(E[0], 1) - d(E[1], 0)])


def _curl_b(B):
    d = lambda F, a: _sh(F, a, -1) - F  # noqa: E731
    return torch.stack([d(B[1], 2) - d(B[2], 1), d(B[2], 0) - d(B[0], 2), d(B[0], 1) - d(B[1], 0)])


def _curl_e_stencil(E):
    def D(F, a):
        # differences over 1, 3 and 5 cells along a (row 0, 1, 2), on the axis
        # (ax 0) or at +-o cells along the first or second axis across it
        v = {k[len("stencil_x_"):]: float(np.float32(m)) for k, m in SHOCK_STENCIL.items() if k[8] == "xyz"[a]}
        rows = [("delta", 1, 0, 0), ("gamma", 2, 0, 0), ("beta_p1", 0, 1, 1), ("beta_p2", 0, 2, 1),
                ("zeta_p1", 0, 1, 2), ("zeta_p2", 0, 2, 2)]
        out, one = 0, 1.0
        for name, r, ax, o in rows:
            m = v.get(name, 0.0)
            d = _sh(F, a, r + 1) - _sh(F, a, -r)
            if ax:
                p = (a + ax) % 3
                d = _sh(d, p, o) + _sh(d, p, -o)
            out = out + m * d
            one -= m * (2 * r + 1) * (2 if ax else 1)
        return out + one * (_sh(F, a, 1) - F)

    return torch.stack([D(E[1], 2) - D(E[2], 1), D(E[2], 0) - D(E[0], 2), D(E[0], 1) - D(E[1], 0)])


def _filter(J):
    for a in (1, 2, 3):
        J = 0.25 * _sh(J, a, -1) + 0.5 * J + 0.25 * _sh(J, a, 1)
    return J


def _nodes(E, B):
    """[cells, 6] values of E and B at the cell nodes."""
    m = [(E[a] + _sh(E[a], a, -1)) / 2 for a in range(3)]
    for a in range(3):
        p, q = [d for d in range(3) if d != a]
        h = B[a] + _sh(B[a], p, -1)
        m.append((h + _sh(h, q, -1)) / 4)
    return torch.stack(m).reshape(6, -1).t()


def _at(nodes, N, x):
    """E and B [3, k] at positions x by trilinear weights."""
    i = torch.floor(x.detach())
    d, i = x - i, i.long()
    out = 0
    for k in range(8):
        o = (k >> 2, k >> 1 & 1, k & 1)
        q = 0
        wt = 1
        for a in range(3):
            q = q * N[a] + (i[a] + o[a]) % N[a]
            wt = wt * (d[a] if o[a] else 1 - d[a])
        out = out + nodes[q] * wt[:, None]
    return out[:, :3].t(), out[:, 3:].t()


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _push(x, u, E, B, sign, pusher="boris"):
    """Moved positions (not wrapped) and momenta; sign: +-1 over the mass, [k]."""
    h = 0.5 * sign
    if pusher == "boris":
        a = u * CFL + E * h
        b = B * (h / torch.sqrt(CFL ** 2 + (a * a).sum(0)))
        f = 2 / (1 + (b * b).sum(0))
        v = (a + _cross(a, b)) * f
        v = a + _cross(v, b) + E * h
    elif pusher == "higuera_cary":
        a, t = u + E * h / CFL, B * h / CFL
        g2, t2, ta = 1 + (a * a).sum(0), (t * t).sum(0), (t * a).sum(0)
        g = torch.sqrt(0.5 * (g2 - t2 + torch.sqrt((g2 - t2) ** 2 + 4 * (t2 + (CFL * ta) ** 2))))
        b = t / g
        v = (a + _cross(a, b)) * (2 / (1 + (b * b).sum(0)))
        v = (a + _cross(v, b) + E * h / CFL) * CFL
    else:
        # (1 - K) w' = (1 + K) w for the four-velocity w = (gamma, u) and the
        # field tensor K over the gamma after half the electric push
        w0, w = torch.sqrt(CFL ** 2 + ((u * CFL) ** 2).sum(0)), u * CFL
        k = h / torch.sqrt(CFL ** 2 + ((w + E * h) ** 2).sum(0))
        e, b = E * k, B * k
        r = w + e * w0 + _cross(w, b) + e * (w0 + (e * w).sum(0))
        inv = lambda y: (y + _cross(y, b) + b * (b * y).sum(0)) / (1 + (b * b).sum(0))  # noqa: E731
        r, m = inv(r), inv(e)
        v = r + m * ((e * r).sum(0) / (1 - (e * m).sum(0)))
    return x + v * (CFL / torch.sqrt(CFL ** 2 + (v * v).sum(0))), v / CFL


def _deposit(J, N, x1, x2, q):
    """J [cells, 3] += the two zigzag segments of moves x1 -> x2 of charges q."""
    f1, f2 = torch.floor(x1.detach()), torch.floor(x2.detach())
    xr = torch.minimum(torch.minimum(f1, f2) + 1, torch.maximum(torch.maximum(f1, f2), 0.5 * (x1 + x2)))
    for f, a, b in ((f1, x1, xr), (f2, xr, x2)):
        F, W, i = (b - a) * q, 0.5 * (a + b) - f, f.long()
        for c in range(3):
            d, e = [v for v in range(3) if v != c]
            for k in range(4):
                o = [0, 0, 0]
                o[d], o[e] = k >> 1, k & 1
                wt = (W[d] if o[d] else 1 - W[d]) * (W[e] if o[e] else 1 - W[e])
                idx = 0
                for m in range(3):
                    idx = idx * N[m] + (i[m] + o[m]) % N[m]
                J = J.index_add(0, idx * 3 + c, F[c] * wt)
    return J


def _back(x, u):
    return x - u * (CFL / torch.sqrt(1 + (u * u).sum(0)))


def _wrap(x, N):
    n = torch.tensor(N, dtype=x.dtype, device=x.device).view(3, 1)
    return torch.where(x < 0, x + n, torch.where(x >= n, x - n, x))


def _haloed(F):
    for a in (1, 2, 3):
        n = F.shape[a]
        F = torch.cat([F.narrow(a, n - HALO, HALO), F, F.narrow(a, 0, HALO)], a)
    return F


def _exact_world(c, tiles, E, B, charges, pusher="boris", shock=False, laps=1, keep=False):
    """The fields after some laps, and with keep the moved particles."""
    N = _shape(c)[2]
    E, B = E.double(), B.double()
    E0, B0 = E.clone(), B.clone()
    curl = _curl_e_stencil if shock else _curl_e
    flip = torch.tensor([[-1.0], [1.0], [1.0]], dtype=torch.float64, device=DEV)

    def edge(F, what):
        if shock:
            left, right = slice(0, int(WALL) + 1), slice(N[0] - 5, None)
            if what == "E":
                F[1:, left] = 0
            if what == "J":
                F[:, left] = 0
            F[:, right] = 0 if what == "J" else (E0 if what == "E" else B0)[:, right]
        return F

    parts = ((s, pos.double(), us[s].double()) for _, pos, us in tiles for s in range(2))
    for lap in range(laps):
        B = edge(B + CFL / 2 * curl(E), "B")
        nodes = _nodes(E, B)
        J = torch.zeros(N[0] * N[1] * N[2] * 3, dtype=torch.float64, device=DEV)
        moved = []
        for s, x, u in parts:
            q = torch.full_like(x[0], charges[s])
            sign = torch.full_like(x[0], math.copysign(1.0, charges[s]))
            x, u = _push(x, u, *_at(nodes, N, x), sign, pusher)
            if shock:
                # behind the wall after the push: the move is cut there and goes on
                # mirrored; its whole current is the two pieces in front of the wall
                hit = x[0] < WALL
                x0, xh, uh, qh = _back(x, u)[:, hit], x[:, hit], u[:, hit], q[hit]
                col = x0 + (x0[0] - WALL) / (x0[0] - xh[0]) * (xh - x0)
                rest = torch.clamp((xh[0] - col[0]) / (xh[0] - x0[0]), max=1.0)
                xn, un = col + rest * (xh - x0) * flip, uh * flip
                J = _deposit(J, N, x0, col, qh)
                J = _deposit(J, N, _back(xn, un), col, -qh)
                x[:, hit], u[:, hit] = xn, un
            x = _wrap(x, N)
            J = _deposit(J, N, _back(x, u), x, q)
            if keep or lap + 1 < laps:
                moved.append((s, x, u))
        parts = moved
        J = edge(J.view(N + [3]).permute(3, 0, 1, 2).clone(), "J")
        for _ in range(3):
            J = _filter(J)
        J = edge(J, "J")
        B = edge(B + CFL / 2 * curl(E), "B")
        E = edge(edge(E + CFL * _curl_b(B), "E") - J, "E")
    return E, B, parts


def _exact_step(E, B, x, u, q):
    """One step of a differentiable box, as a whole autograd graph."""
    N = list(E.shape[1:])
    B1 = B + CFL / 2 * _curl_e(E)
    xn, un = _push(x, u, *_at(_nodes(E, B1), N, x), torch.sign(q))
    xn = _wrap(xn, N)
    J = _deposit(torch.zeros(E.numel(), dtype=torch.float64, device=DEV), N, _back(xn, un), xn, q)
    J = J.view(N + [3]).permute(3, 0, 1, 2)
    for _ in range(3):
        J = _filter(J)
    B2 = B1 + CFL / 2 * _curl_e(E)
    return E + CFL * _curl_b(B2) - J, B2, xn, un


def _charge_of(charges, np_):
    return torch.cat([torch.full((np_,), v, dtype=torch.float64, device=DEV) for v in charges])


def _exact_diff(c, seed):
    charges, np_, state = _box_state(c, seed, torch.float64)
    E, B, x, u = state
    N = list(E.shape[1:])
    q = _charge_of(charges, np_)
    fwd, adj = c["what"] != "adjoint", c["what"] != "step"
    lam = _box_adjoint([v.to(torch.float64 if c["double"] else torch.float32) for v in state], seed) if adj else None
    half = CFL / 2
    if adj:
        lE, lB, lx, lu = (v.double() for v in lam)
        lJ = -lE
        for _ in range(3):
            lJ = _filter(lJ)
        lJ = lJ.permute(1, 2, 3, 0).reshape(-1)
    B1 = (B + half * _curl_e(E)).requires_grad_(adj)
    Ei = E.clone().requires_grad_(adj)
    J = torch.zeros(E.numel(), dtype=torch.float64, device=DEV)
    xo, uo = torch.empty_like(x), torch.empty_like(u)
    gx, gu = torch.empty_like(x), torch.empty_like(u)
    chunk = 2_000_000
    for a in range(0, x.shape[1], chunk):
        sl = slice(a, a + chunk)
        xc, uc = x[:, sl].clone().requires_grad_(adj), u[:, sl].clone().requires_grad_(adj)
        xn, un = _push(xc, uc, *_at(_nodes(Ei, B1), N, xc), torch.sign(q[sl]))
        xn = _wrap(xn, N)
        Jc = _deposit(torch.zeros_like(J), N, _back(xn, un), xn, q[sl])
        if adj:
            ((lx[:, sl] * xn).sum() + (lu[:, sl] * un).sum() + (lJ * Jc).sum()).backward()
            gx[:, sl], gu[:, sl] = xc.grad, uc.grad
        xo[:, sl], uo[:, sl] = xn.detach(), un.detach()
        J += Jc.detach()
    out = {}
    if fwd:
        Jf = J.view(N + [3]).permute(3, 0, 1, 2)
        for _ in range(3):
            Jf = _filter(Jf)
        B2 = B1.detach() + half * _curl_e(E)
        out["step"] = (E + CFL * _curl_b(B2) - Jf, B2, xo, uo)
    if adj:
        e, b = E.clone().requires_grad_(), B.clone().requires_grad_()
        b1 = b + half * _curl_e(e)
        b2 = b1 + half * _curl_e(e)
        ((lE * (e + CFL * _curl_b(b2))).sum() + (lB * b2).sum() + (B1.grad * b1).sum() + (Ei.grad * e).sum()).backward()
        out["adjoint"] = (e.grad, b.grad, gx, gu)
    return out


def _exact_rollout(c, seed):
    ends, grads = [], []
    boxes = _boxes(c)
    for k, b in enumerate(boxes):
        charges, np_, state = _box_state(b, seed + 1009 * k, torch.float64)
        q = _charge_of(charges, np_)
        state = [v.requires_grad_() for v in state]
        s = state
        for _ in range(c["steps"]):
            s = _exact_step(*s, q)
        (0.5 * (s[1] ** 2).sum()).backward()
        one = len(boxes) == 1
        ends.append([v.detach() if one else v.detach().reshape(3, -1) for v in s])
        grads.append([v.grad if one else v.grad.reshape(3, -1) for v in state])
        del s, state
    return dict(end=[torch.cat([e[i] for e in ends], 1) if len(ends) > 1 else ends[0][i] for i in range(4)],
                grad=[torch.cat([g[i] for g in grads], 1) if len(grads) > 1 else grads[0][i] for i in range(4)])


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sim":
        n, t, _ = _shape(c)
        E, B, kept = _exact_world(c, _tiles(c, seed), *_fields(c, _gen(seed)), _plasma(c)[0], keep=True)
        out = dict(pos=[], vel=[])
        for s in range(2):
            # by the tile that holds the particle after the lap, then by id
            x, u = (torch.cat([p[k] for p in kept if p[0] == s], 1) for k in (1, 2))
            tile = 0
            for a in range(3):
                tile = tile * t[a] + torch.floor(x[a] / n[a]).long()
            o = torch.sort(tile, stable=True).indices
            out["pos"].append(x[:, o])
            out["vel"].append(u[:, o])
        return dict(out, E=_haloed(E), B=_haloed(B))
    if kind == "world":
        E, B, _ = _exact_world(c, _tiles(c, seed), *_fields(c, _gen(seed)), _plasma(c)[0], c["pusher"])
        return dict(E=_haloed(E), B=_haloed(B))
    if kind == "shock":
        # run() is the lap after the one that prepare() takes
        E, B, _ = _exact_world(c, _shock_tiles(c, seed), *_shock_fields(c), _plasma(c, c["gamma"])[0], "faraday",
                               shock=True, laps=2)
        return dict(E=_haloed(E), B=_haloed(B))
    if kind == "diff":
        return _exact_diff(c, seed)
    if kind == "rollout":
        return _exact_rollout(c, seed)
    N = _shape(c)[2]
    s = c["stride"]
    g = _gen(seed)
    B = _fields(dict(c, sigma=1.0), g)[1].double()
    g = _gen(seed + 3)
    E = (0.3 * torch.randn(B.shape, generator=g, device=DEV)).double()
    J = (0.1 * torch.randn(B.shape, generator=g, device=DEV)).double()
    M = [v // s for v in N]
    dens = torch.zeros((2,) + tuple(M), dtype=torch.float64, device=DEV)
    energy = [0.5 * float((E ** 2).sum()), 0.5 * float((B ** 2).sum()), 0.0, 0.0]
    for i, pos, us in _tiles(c, seed):
        q = torch.floor(pos.double() / s).long()
        q = (q[0] * M[1] + q[1]) * M[2] + q[2]
        for k in range(2):
            dens[k].view(-1).index_add_(0, q, torch.ones_like(q, dtype=torch.float64))
            energy[2 + k] += float((torch.sqrt(1 + (us[k].double() ** 2).sum(0)) - 1).sum())
    J = J.view(3, M[0], s, M[1], s, M[2], s).sum((2, 4, 6))
    fields = torch.cat([E[:, ::s, ::s, ::s], B[:, ::s, ::s, ::s], J, dens])
    # the spectra are counts of values near bin edges: only the same code gives the same
    return dict(fields=fields.permute(0, 3, 2, 1).contiguous(), spectra=None, energies=np.array(energy))
