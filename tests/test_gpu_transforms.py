"""coftxy and cofitxy on every shape of their kernels (kernels_spectral.hpp): one
workgroup for a small grid, rows sharing a workgroup with and without a
remainder, columns by two and by four, odd numbers of columns and lengths
that keep the staged kernels; against numpy's transform in the packed layout,
and in place on the GPU.  Tolerance 1e-13 of the largest value: both sides
round each of the log2(nx ny) <= 22 levels to 1.1e-16."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(64, 64), (128, 32), (64, 32), (64, 36), (96, 96), (128, 54), (192, 128), (256, 192), (384, 256), (512, 384),
         (54, 384), (768, 512), (1024, 768), (1536, 64), (64, 1536), (2048, 96), (96, 2048), (72, 72), (108, 162)]


def _packed(a):
    from fsibe_2d_amd.inputs import half_to_packed

    ny, nx = a.shape
    z = np.fft.rfft2(a)[:, : nx // 2] / (nx * ny)
    z[ny // 2] = 0.0
    return half_to_packed(z)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_transforms_against_numpy(nx, ny):
    from fsibe_2d_amd.spectral import Spectral

    a = np.random.default_rng(nx * 7 + ny).standard_normal((ny, nx))
    sp = Spectral(nx, ny, 4.0, 4.0, 1e-3)
    want = _packed(a)
    got = sp.coftxy(a)
    assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()
    # without the Nyquist modes, which the packed layout does not hold
    z = np.fft.rfft2(a)
    z[:, nx // 2] = 0.0
    z[ny // 2] = 0.0
    b = np.fft.irfft2(z, s=(ny, nx))
    assert np.abs(sp.cofitxy(got) - b).max() <= 1e-13 * np.abs(a).max() * np.log2(nx * ny)
    sp.close()


@pytest.mark.parametrize("nx,ny", [(64, 64), (128, 32), (96, 96), (512, 384)])
def test_transforms_in_place(nx, ny):
    from fsibe_2d_amd._lib import check, lib
    from fsibe_2d_amd.spectral import Spectral

    a = np.random.default_rng(nx + ny).standard_normal((ny, nx))
    sp = Spectral(nx, ny, 4.0, 4.0, 1e-3)
    fk = sp.coftxy(a)
    f = sp.cofitxy(fk)
    h = C.CDLL("libamdhip64.so.7")
    p, n, out = C.c_void_p(), C.c_size_t(a.nbytes), np.empty_like(a)
    assert h.hipMalloc(C.byref(p), n) == 0 and h.hipMemcpy(p, C.c_void_p(a.ctypes.data), n, 1) == 0
    for op, want in ((lib().fsibe_dev_coftxy, fk), (lib().fsibe_dev_cofitxy, f)):
        check(op(sp.h, p, p, None))
        assert h.hipDeviceSynchronize() == 0 and h.hipMemcpy(C.c_void_p(out.ctypes.data), p, n, 2) == 0
        assert np.array_equal(out, want)
    assert h.hipFree(p) == 0
    sp.close()
