"""The extended-stencil half B push with coefficients off the axial line in the
first row only, as the shock configuration has them (132 of the 324 reads per
cell), against the oracle, which sums every term: bit-exact, also where an
infinity or a NaN in E, or an overflowing sum of two values, turns the dropped
terms (0 times it) into NaN.  Tiles of
37 x planes end in a partial segment, 10 y rows in a partial block."""

import numpy as np
import pytest

import runko_amd as runko
from gpu_common import build_gpu, build_oracle, gpu_fields, random_inputs

pytestmark = pytest.mark.gpu

AXIAL = dict(stencil_delta=-0.06, stencil_gamma=0.004, stencil_beta_p1=0.011, stencil_beta_p2=-0.007,
             stencil_zeta_p1=0.003, stencil_zeta_p2=0.002, stencil_x_delta=-0.05)


@pytest.mark.parametrize("bad", [None, np.inf, np.nan, 3e38])
@pytest.mark.parametrize("execution", ["plain", "batched"])
def test_axial_stencil_half_b(orc, execution, bad):
    nt, n = (2, 1, 1), (37, 10, 7)
    inputs = random_inputs(nt, n, 0, seed=89)
    if bad is not None:
        inputs[(0, 0, 0)][0][1][20, [4, 6], 3] = bad
    conf, grid, sim = build_gpu(nt, n, [], [], inputs, execution=execution, stencil=AXIAL)
    w = build_oracle(orc, nt, n, [], [], inputs, stencil=AXIAL)
    cm = runko.tools.comm_mode

    def lap(x):
        x.grid_push_half_b()
        x.comm_local(cm.emf_B)

    sim.for_one_lap(lap)
    w.push_half_b()
    w.comm_local("emf_B")
    got, want = gpu_fields(grid), w.global_fields()
    assert np.isnan(want[3:6]).any() == (bad is not None)
    assert np.array_equal(got, want, equal_nan=True)
