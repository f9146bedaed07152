"""Copies between host memory and the GPU (transfer.hpp): the host-pointer
entry points against the device ones on the same values, at sizes below and
at the threshold, of a few chunks, of about the pinned ring and beyond it (its
slots are used again) and with a last chunk that is not full; pinned host
arrays; and several threads at once, of which one has the ring.  A copy
changes nothing, so the results are equal bit for bit."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(384, 384), (512, 1024), (512, 1152), (1458, 1536), (2048, 2048), (2048, 3072)]


def _hip():
    """the HIP runtime that the library runs on"""
    from fsibe_2d_amd._lib import lib

    lib()
    return C.CDLL("libamdhip64.so.7")


def _device(sp, a):
    from fsibe_2d_amd._lib import check, lib

    h, n = _hip(), C.c_size_t(a.nbytes)
    p = [C.c_void_p() for _ in range(3)]
    for q in p:
        assert h.hipMalloc(C.byref(q), n) == 0
    assert h.hipMemcpy(p[0], C.c_void_p(a.ctypes.data), n, 1) == 0
    check(lib().fsibe_dev_coftxy(sp.h, p[0], p[1], None))
    check(lib().fsibe_dev_spectral_op(sp.h, 0, p[1], p[2], None))
    out = [np.empty_like(a), np.empty_like(a)]
    for o, q in zip(out, p[1:]):
        assert h.hipMemcpy(C.c_void_p(o.ctypes.data), q, n, 2) == 0
    for q in p:
        assert h.hipFree(q) == 0
    return out


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("pinned", [False, True])
def test_host_calls_equal_device_calls(nx, ny, pinned):
    from fsibe_2d_amd.spectral import Spectral

    sp = Spectral(nx, ny, 4.0, 4.0, 1e-3)
    a = np.random.default_rng(nx + ny).standard_normal((ny, nx))
    q = C.c_void_p()
    if pinned:
        assert _hip().hipHostMalloc(C.byref(q), C.c_size_t(a.nbytes), 0) == 0
        b = np.ctypeslib.as_array(C.cast(q, C.POINTER(C.c_double)), shape=a.shape)
        b[:] = a
        a = b
    fk, dx = _device(sp, a)
    for _ in range(2):
        hk = sp.coftxy(a)
        assert np.array_equal(hk, fk) and np.array_equal(sp.cofdx(hk), dx)
    sp.close()
    if pinned:
        assert _hip().hipHostFree(q) == 0


def test_threads_copy_at_the_same_time():
    from fsibe_2d_amd.spectral import Spectral

    nx, ny, n = 768, 768, 4
    sps = [Spectral(nx, ny, 4.0, 4.0, 1e-3) for _ in range(n)]
    a = [np.random.default_rng(i).standard_normal((ny, nx)) for i in range(n)]
    want = [_device(sps[i], a[i])[0] for i in range(n)]
    ok = [0] * n

    def work(i):
        for _ in range(10):
            ok[i] += int(np.array_equal(sps[i].coftxy(a[i]), want[i]))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [10] * n
    for s in sps:
        s.close()
