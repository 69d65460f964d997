"""GPU test of the particle step at the edges of its tiles (runs of particles,
one a thread) and of its sampler's fast case: the phi seam, the rows next to
the poles, where the checked sampler takes over, and positions a fold away."""
import math

import numpy as np
import pytest

import kaminogpu_amd as K
from oracle import oracle as O
from test_particles import TOL_POS, rel_pos

pytestmark = pytest.mark.gpu


def positions(nt, n, seed):
    """n positions: a third uniform, the others on the seams of the fast case."""
    rng = np.random.default_rng(seed)
    h = math.pi / nt
    pos = np.stack([rng.uniform(0, 2 * math.pi, n), rng.uniform(0, math.pi, n)], 1)
    pos[1::6, 0] = rng.uniform(-h, h, len(pos[1::6])) % (2 * math.pi)
    pos[2::6, 1] = rng.uniform(0, 4 * h, len(pos[2::6]))
    pos[3::6, 1] = math.pi - rng.uniform(0, 4 * h, len(pos[3::6]))
    pos[4::6, 1] = rng.uniform(-0.5, 4, len(pos[4::6])).clip(-0.9 * h, math.pi + 0.9 * h)
    return pos.astype(np.float32)


@pytest.mark.parametrize("nt", [4, 5, 6, 27, 75, 128, 135, 144, 256])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 5000])
def test_particle_step_vs_oracle(nt, n):
    dt = 0.5 / nt
    up, ut, rho = [np.ascontiguousarray(a, np.float32) for a in O.init_fields(nt, 2 * nt, max(1, min(8, nt // 4)), nt, 1)]
    pos = positions(nt, n, nt + n)
    with K.Sim(nt, dt) as s:
        s.set_fields(up, ut, rho)
        s.set_particles(pos)
        s.step(1)
        got = s.get_particles()
        assert s.status() == 0
    ref, amb = O.advect_particles(nt, 2 * nt, dt, up, ut, pos)
    if not amb.all():
        assert rel_pos(got, ref, amb) < TOL_POS


@pytest.mark.parametrize("nt", [80, 125, 128, 135])
@pytest.mark.parametrize("n", [1536 * 256, 600001, 8192 * 256 + 65])
def test_staged_particles_equal_gathered(nt, n):
    """Many particles are sampled from LDS; the same particles set a few at a
    time are sampled from memory and land on the same positions to the bit."""
    dt = 0.5 / nt
    state = [np.ascontiguousarray(a, np.float32) for a in O.init_fields(nt, 2 * nt, 8, nt, 1)]
    pos = positions(nt, n, nt)
    pos[:4] = [[np.nan, 1.0], [1.0, np.inf], [1e30, 1.0], [-1e9, 0.5]]
    with K.Sim(nt, dt) as s:
        s.set_fields(*state)
        s.set_particles(pos)
        s.step_phases(K.PHASE_ADVECT)
        got = s.get_particles()
    part = 300000
    for k in range(0, n, part):
        with K.Sim(nt, dt) as s:
            s.set_fields(*state)
            s.set_particles(pos[k:k + part])
            s.step_phases(K.PHASE_ADVECT)
            np.testing.assert_array_equal(got[k:k + part], s.get_particles())
