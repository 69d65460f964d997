"""GPU tests of the advection tiles next to the poles: flows whose departure
points leave the staged windows in phi and theta, small, odd and ragged sizes,
tiles of every height, with and without the metric update, against the FP64
oracle; and the same fields from every tile shape."""
import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import TOL_FIELD, oracle_advect_geo, rel_l2, seeded_state

pytestmark = pytest.mark.gpu


def advected(nt, dt, state, geometric, tune=None):
    try:
        if tune:
            K.tune_set(nt, *tune)
        with K.Sim(nt, dt, geometric=geometric) as s:
            s.set_fields(*state)
            s.step_phases(K.PHASE_ADVECT)
            return s.get_fields()
    finally:
        K.tune_set(nt, 0, 0, 0)


# the speed scales the seeded flow (|u| ~ 1): at 1 the row next to a pole moves
# about nt / 10 columns, at 6 six times that and rows move up to about one row
# and a half
@pytest.mark.parametrize("nt", [4, 6, 9, 16, 32, 50, 75, 128, 256])
@pytest.mark.parametrize("speed", [1.0, 6.0])
@pytest.mark.parametrize("geometric", [True, False])
def test_polar_rows_against_oracle(nt, speed, geometric):
    dt = 0.5 / nt
    up, ut, rho = seeded_state(nt, L=max(1, min(8, nt // 4)), seed=300 + nt, dens=1)
    # the metric update's cubic needs G u < 1 for its one root
    up, ut = (np.float32(speed) * up, np.float32(speed) * ut) if not geometric else (up, ut)
    got = advected(nt, dt, (up, ut, rho), geometric)
    ref, masks, _ = oracle_advect_geo(nt, dt, up, ut, rho, geometric)
    for g, r, m in zip(got, ref, masks):
        # FP32 weights: a departure of x cells carries 6e-8 x; the rows with
        # x ~ 100 are a few of many, so the whole field keeps the step's bound
        assert rel_l2(g, r, m) <= TOL_FIELD


@pytest.mark.parametrize("nt", [9, 32, 75, 128])
@pytest.mark.parametrize("geometric", [True, False])
def test_tile_shapes_give_the_same_fields(nt, geometric):
    dt = 0.5 / nt
    state = seeded_state(nt, L=max(1, min(8, nt // 4)), seed=400 + nt, dens=1)
    ref = advected(nt, dt, state, geometric)
    for tune in [(1, 64, 0), (2, 128, 0), (3, 16, 0), (4, 64, 0), (5, 17, 0), (8, 100, 0), (16, 128, 0), (33, 64, 0)]:
        for a, b in zip(advected(nt, dt, state, geometric, tune), ref):
            np.testing.assert_array_equal(a, b)
