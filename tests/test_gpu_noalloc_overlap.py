"""GPU test of kam_sim_step_noalloc on fields that share memory (one buffer
given twice, or fields that begin inside one another): every field is read
before any is written, and u_phi, u_theta and rho are written back in that
order, so a shared value ends as the last field that holds it has it.  Sizes
whose fields are whole runs of 16 bytes and sizes whose fields are not."""
import ctypes as C

import numpy as np
import pytest

import kaminogpu_amd as K
from test_zz_no_alloc import Hip, solo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [9, 32, 256])
@pytest.mark.parametrize("offs", ["rho is u_phi", "u_theta in u_phi", "u_phi in rho"])
def test_fields_that_share_memory(nt, offs):
    N, Nt = 2 * nt * nt, 2 * nt * (nt - 1)
    at = {"rho is u_phi": (0, N, 0), "u_theta in u_phi": (0, N // 2 + 1, 2 * N), "u_phi in rho": (7, 2 * N, 0)}[offs]
    spans = [slice(o, o + n) for o, n in zip(at, (N, Nt, N))]
    shapes = [(nt, 2 * nt), (nt - 1, 2 * nt), (nt, 2 * nt)]
    host = (0.1 * np.random.default_rng(nt).standard_normal(3 * N)).astype(np.float32)
    hip = Hip()
    buf = hip.upload(host)
    try:
        d = K.SimDesc(nt, 2 * nt, 1.0, 0.05 / nt, 1, K.PREC_FP32, 0)
        ptrs = [C.c_void_p(buf.value + 4 * o) for o in at]
        K.check(K.lib().kam_sim_step_noalloc(C.byref(d), *ptrs, 2, None))
        hip.ok(hip.h.hipStreamSynchronize(None), "hipStreamSynchronize")
        state = [host[s].reshape(shape) for s, shape in zip(spans, shapes)]
        want = host.copy()
        for s, r in zip(spans, solo(nt, 0.05 / nt, state, 2, K.PREC_FP32)):
            want[s] = r.ravel()
        np.testing.assert_array_equal(hip.download(buf, host.shape), want)
    finally:
        hip.free(buf)
