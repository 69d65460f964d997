"""GPU tests of the row FFT at the sizes where its plan changes: every kind of
pass, powers of two (kernels of their own), rows wider than a wavefront, and
batches that mix them.  The forward and inverse transforms are compared with
FP64 transforms of the same inputs."""
import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import seeded_state

pytestmark = pytest.mark.gpu

# FP32: a transform of M values rounds each value about log2(M) <= 11 times and
# the divergence six times, 6e-8 each, relative to the row: 1.0e-6; twice that
TOL = 2e-6


def random_state(nt, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((r, 2 * nt)).astype(np.float32) for r in (nt, nt - 1, nt)]


def divergence(nt, up, ut):
    h, tc = np.pi / nt, (np.arange(nt)[:, None] + 0.5) * np.pi / nt
    flux = np.zeros((nt + 1, 2 * nt))
    flux[1:-1] = ut * np.sin(np.arange(1, nt) * h)[:, None]
    return (flux[1:] - flux[:-1] + np.roll(up, -1, axis=1) - up) / (h * np.sin(tc))


@pytest.mark.parametrize("nt", [4, 5, 6, 8, 9, 10, 16, 24, 30, 32, 45, 50, 64, 75, 81, 96, 128, 160, 243, 256, 375, 405,
                                512, 625, 720, 1000, 1024, 1250, 2000, 2048])
@pytest.mark.parametrize("precision", [K.PREC_FP32, K.PREC_FP64_PRESSURE])
def test_transforms_against_fp64(nt, precision):
    if precision == K.PREC_FP64_PRESSURE and nt > 1024:
        pytest.skip("the FP64 pressure holds n_theta <= 1024")
    up, ut, rho = random_state(nt, nt)
    h, sn = np.pi / nt, np.sin((np.arange(nt)[:, None] + 0.5) * np.pi / nt)
    with K.Sim(nt, 0.5 / nt, precision=precision) as s:
        s.set_fields(up, ut, rho)
        s.step_phases(K.PHASE_DIVFFT)
        spec = s.spectrum()
        s.step_phases(K.PHASE_TRI)
        solved = s.spectrum().astype(np.complex128)
        p = s.pressure().astype(np.float64)
        s.step_phases(K.PHASE_IFFT)
        gu, gt, _ = s.get_fields()
        assert s.status() == 0
    up, ut = up.astype(np.float64), ut.astype(np.float64)
    ref = np.fft.rfft(divergence(nt, up, ut), axis=1).T / (2 * nt)
    ref[0] = ref[0].real + 1j * ref[nt].real  # slot 0 holds modes 0 and n_theta
    ref = ref[:nt]
    assert np.all(np.linalg.norm(spec - ref, axis=0) <= TOL * np.linalg.norm(ref, axis=0))
    if precision == K.PREC_FP32:
        # the pressure is the inverse transform of the solved spectrum, mode 0 dropped
        full = np.zeros((nt, nt + 1), np.complex128)
        full[:, :nt] = solved.T
        full[:, nt] = solved[0].imag
        full[:, 0] = 0
        ref_p = np.fft.irfft(full, n=2 * nt, axis=1) * 2 * nt
        norm = np.linalg.norm(ref_p, axis=1)
        assert np.all(np.linalg.norm(p - ref_p, axis=1) <= TOL * norm + 1e-30)
        tol_p = TOL
    else:
        ref_p, norm, tol_p = p, np.linalg.norm(p, axis=1), 1.2e-7  # p was rounded once for the readback
    # the gradient: a rounding of u and twice the pressure's error over the step
    du = np.linalg.norm(gu - (up - (ref_p - np.roll(ref_p, 1, axis=1)) / (h * sn)), axis=1)
    assert np.all(du <= 3e-7 * np.linalg.norm(gu, axis=1) + 2 * tol_p * norm / (h * sn[:, 0]))
    dt = np.linalg.norm(gt - (ut - (ref_p[1:] - ref_p[:-1]) / h), axis=1)
    assert np.all(dt <= 3e-7 * np.linalg.norm(gt, axis=1) + tol_p * (norm[1:] + norm[:-1]) / h)


def test_mixed_sizes_equal_alone():
    sizes = [(1000, K.PREC_FP32), (64, K.PREC_FP32), (375, K.PREC_FP64_PRESSURE), (720, K.PREC_FP32),
             (256, K.PREC_FP64_PRESSURE), (1024, K.PREC_FP32), (9, K.PREC_FP32)]
    states = [seeded_state(nt, L=max(1, min(8, nt // 4)), seed=nt, dens=1) for nt, _ in sizes]
    with K.Engine(groups=2) as eng:
        ids = [eng.admit(nt, 0.5 / nt, *st, steps=2, precision=pr) for (nt, pr), st in zip(sizes, states)]
        eng.step(2)
        got = [eng.fetch(i, nt) for i, (nt, _) in zip(ids, sizes)]
    for (nt, pr), st, g in zip(sizes, states, got):
        with K.Sim(nt, 0.5 / nt, precision=pr) as s:
            s.set_fields(*st)
            s.step(2)
            for a, b in zip(g, s.get_fields()):
                np.testing.assert_array_equal(a, b)
