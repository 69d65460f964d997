"""GPU test of kam_sim_step_noalloc's copies of the caller's fields: buffers at
addresses that are not 16-byte aligned, fields whose size is no multiple of
four values, pinned host buffers, and nothing written outside a field; results
equal kam_sim_step's bitwise."""
import ctypes as C

import numpy as np
import pytest

import kaminogpu_amd as K
from parity_util import seeded_state
from test_zz_no_alloc import Hip, solo

pytestmark = pytest.mark.gpu

GUARD = np.float32(-7.25)


def padded(a, off):
    """a with `off` guard values before it and five behind it."""
    g = np.full(off + a.size + 5, GUARD, np.float32)
    g[off:off + a.size] = a.ravel()
    return g


@pytest.mark.parametrize("nt,offs", [(32, (0, 0, 0)), (32, (1, 2, 3)), (45, (0, 0, 0)), (45, (4, 1, 0)), (9, (2, 0, 1))])
def test_unaligned_and_odd_sized_fields(nt, offs):
    hip = Hip()
    state = seeded_state(nt, L=max(1, min(16, nt // 4)), seed=60 + nt, dens=1)
    host = [padded(a, o) for a, o in zip(state, offs)]
    bufs = [hip.upload(h) for h in host]
    try:
        d = K.SimDesc(nt, 2 * nt, 1.0, 0.5 / nt, 1, K.PREC_FP32, 0)
        ptrs = [C.c_void_p(b.value + 4 * o) for b, o in zip(bufs, offs)]
        K.check(K.lib().kam_sim_step_noalloc(C.byref(d), *ptrs, 2, None))
        hip.ok(hip.h.hipStreamSynchronize(None), "hipStreamSynchronize")
        ref = solo(nt, 0.5 / nt, state, 2, K.PREC_FP32)
        for b, h, o, r in zip(bufs, host, offs, ref):
            np.testing.assert_array_equal(hip.download(b, h.shape), padded(r, o))
    finally:
        for b in bufs:
            hip.free(b)


def test_pinned_host_fields():
    nt = 32
    hip = Hip()
    state = seeded_state(nt, L=8, seed=61, dens=1)
    bufs = []
    try:
        for a in state:
            p = C.c_void_p()
            hip.ok(hip.h.hipHostMalloc(C.byref(p), C.c_size_t(a.nbytes), 0), "hipHostMalloc")
            C.memmove(p, a.ctypes.data, a.nbytes)
            bufs.append(p)
        d = K.SimDesc(nt, 2 * nt, 1.0, 0.5 / nt, 1, K.PREC_FP32, 0)
        K.check(K.lib().kam_sim_step_noalloc(C.byref(d), *bufs, 3, None))
        hip.ok(hip.h.hipStreamSynchronize(None), "hipStreamSynchronize")
        for p, a, r in zip(bufs, state, solo(nt, 0.5 / nt, state, 3, K.PREC_FP32)):
            got = np.ctypeslib.as_array((C.c_float * a.size).from_address(p.value)).reshape(a.shape).copy()
            np.testing.assert_array_equal(got, r)
    finally:
        for p in bufs:
            hip.h.hipHostFree(p)
