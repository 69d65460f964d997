"""GPU test of the forward transform's row points in tall tiles of
power-of-two sizes (row coefficients taken per wavefront, u_theta of the row
above from the slot before): heights that fill a thread's slots, that end
inside them and that take several batches.  One sphere alone runs tiles of a
row or two, so each batch holds enough spheres to keep the height set, and its
members' fields equal the sphere alone bitwise."""
import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [K.PREC_FP32, K.PREC_FP64_PRESSURE])
@pytest.mark.parametrize("nt,rows", [(32, 9), (64, 3), (64, 16), (64, 17), (128, 5), (128, 9), (256, 2), (256, 3),
                                     (256, 4), (256, 5), (256, 9), (512, 2), (512, 3), (512, 5), (1024, 2), (1024, 3)])
def test_tall_tiles_equal_one_sphere(nt, rows, precision):
    count = 512 * rows // nt + 2  # tiles are halved until a CU has two
    states = [seeded_state(nt, L=8, seed=nt + k, dens=1) for k in range(2)]
    alone = []
    for st in states:
        with K.Sim(nt, 0.5 / nt, precision=precision) as s:
            s.set_fields(*st)
            s.step(1)
            alone.append(s.get_fields())
    try:
        K.tune_set(nt, 0, 0, rows)
        with K.Engine(max_slots=count, hbm_budget_bytes=count * (K.lib().kam_sim_bytes(nt, 2 * nt) + 4096) + (1 << 24)) as e:
            ids = [e.admit(nt, 0.5 / nt, *states[k % 2], steps=1, precision=precision) for k in range(count)]
            e.step(1)
            for k in sorted({0, 1, count // 2, count - 1}):
                for a, b in zip(e.fetch(ids[k], nt), alone[k % 2]):
                    np.testing.assert_array_equal(a, b)
    finally:
        K.tune_set(nt, 0, 0, 0)
