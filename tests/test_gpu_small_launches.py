"""GPU test of the advection's two workgroup sizes: a launch of few cells takes
eight waves a workgroup and its tiles apart from those of a large batch, and
a sphere steps to the same bits in either."""
import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [4, 9, 15, 32, 45, 75, 128, 192, 216])
@pytest.mark.parametrize("geometric", [True, False])
def test_alone_equals_batched(nt, geometric):
    steps, dt = 4, 0.5 / nt
    state = seeded_state(nt, L=max(1, min(8, nt // 4)), seed=nt, dens=1)
    with K.Sim(nt, dt, geometric=geometric) as s:
        s.set_fields(*state)
        s.step(steps)
        alone = s.get_fields()
        assert s.status() == 0
    members = [(nt, state)] + [(256, seeded_state(256, L=8, seed=1, dens=1))]  # 131072 cells more
    total = sum(K.lib().kam_sim_bytes(n, 2 * n) + 4096 for n, _ in members)
    with K.Engine(hbm_budget_bytes=total + (64 << 20)) as e:
        ids = [e.admit(n, 0.5 / n, *f, steps=steps, geometric=geometric) for n, f in members]
        e.step(steps)
        batched = e.fetch(ids[0], nt)
    for a, b in zip(alone, batched):
        np.testing.assert_array_equal(a, b)
