"""GPU tests of the advection tiles next to the poles with the metric update and
a fast zonal flow: departure points leave the staged windows (PolarStage) in
phi, also those of the antipodal u_theta rows, whose samples then come from the
global sampler.  Only u_phi is scaled, since the update's cubic has its one root
whatever u_phi is, as long as 1 + G v stays positive (v the mean u_theta)."""
import math

import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import TOL_FIELD, oracle_advect_geo, rel_l2, seeded_state
from test_gpu_polar_tiles import advected

pytestmark = pytest.mark.gpu

ROWS = 8  # rows next to either pole that flow fast


def fast_state(nt, dt):
    """A seeded flow whose ROWS rows at a pole are scaled until the nodes of
    u_theta's row next to it move one and a half times the side columns of a
    window: what a flow of speed 1.25 moves in u_phi's row there and three more,
    rounded up to four, at most 64."""
    up, ut, rho = seeded_state(nt, L=min(8, nt // 4), seed=500 + nt, dens=1)
    h = math.pi / nt
    side = min(64.0, 1.25 * (dt / h) / math.sin(0.5 * h) + 3 + 4)
    for pole, rows in ((0, slice(0, ROWS)), (-1, slice(nt - ROWS, nt))):
        up[rows] *= np.float32(1.5 * side / (np.abs(up[pole]).max() * (dt / h) / math.sin(h)))
    assert np.abs(ut).max() * dt / math.tan(0.5 * h) < 0.9  # 1 + G v > 0
    return up, ut, rho


# The tolerance is the step's own.  A departure of x <= 100 cells carries FP32
# errors of 6e-8 x from its rounding and 2e-7 x from its velocities, and the flow
# (m <= 8) changes by at most 8 pi / nt of itself per cell: 2e-6 at 512, 4e-6 at
# 16 (x <= 14).
@pytest.mark.parametrize("nt", [16, 50, 75, 128, 256, 512])
def test_departures_outside_the_windows_against_oracle(nt):
    dt = 0.5 / nt
    state = fast_state(nt, dt)
    got = advected(nt, dt, state, True)
    ref, masks, _ = oracle_advect_geo(nt, dt, *state, True)
    for g, r, m in zip(got, ref, masks):
        assert rel_l2(g, r, m) <= TOL_FIELD


@pytest.mark.parametrize("nt", [16, 75, 128])
def test_tile_shapes_give_the_same_fields(nt):
    """Tile shapes change how much of a row the windows hold, and no value."""
    dt = 0.5 / nt
    state = fast_state(nt, dt)
    ref = advected(nt, dt, state, True)
    for tune in [(1, 64, 0), (2, 128, 0), (3, 16, 0), (4, 64, 0), (5, 17, 0), (16, 128, 0), (33, 64, 0)]:
        for a, b in zip(advected(nt, dt, state, True, tune), ref):
            np.testing.assert_array_equal(a, b)
