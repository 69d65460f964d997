"""GPU test of the pressure solve where a lane holds up to 32 rows: the plain
solve takes its row tables through registers, the residual-reporting one from
LDS, and both leave the same solution, whose residual formed in FP64 meets the
solver's gate."""
import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [1080, 1500, 2000, 2048])  # 17, 24 and 32 rows a lane, the last one full
def test_plain_solve_equals_reporting_solve(nt):
    state = seeded_state(nt, L=16, seed=11, dens=1)
    with K.Sim(nt, 0.5 / nt) as s:
        s.set_fields(*state)
        s.step_phases(K.PHASE_ADVECT | K.PHASE_DIVFFT)
        spec = s.spectrum()
        res = s.poisson_residual()
        reported = s.spectrum()
        s.set_fields(*state)
        s.step_phases(K.PHASE_ADVECT | K.PHASE_DIVFFT)
        np.testing.assert_array_equal(s.spectrum(), spec)
        s.step_phases(K.PHASE_TRI)
        np.testing.assert_array_equal(s.spectrum(), reported)
    assert np.all(np.isfinite(res)) and res.max() <= 1e-6
