"""Fields damped to the end of the number range: the fused stages form their
quotients from reciprocals (div_by, kernels_fused.hpp), the batched stages and
the separate row kernel divide, and both round alike down to denormal numbers,
so the fields agree bit for bit.  Amplitudes: the quotients' dividends around
2^-1020, 2^-1040 (denormal) and, for comparison, 2^-900."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _flow(nx, ny, scale):
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.inputs import half_to_packed, normals

    r = 12
    g = np.array(normals(7, 2 * r * r)).reshape(2, r, r)
    z = np.zeros((ny, nx // 2), dtype=np.complex128)
    z[1:r + 1, 1:r + 1] = (g[0] + 1j * g[1]) * scale
    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=1e-4, iBeam=0, iSaveBeam=0, iSponge=0, iMotion=0,
               iMeanVelocity=4, U_mean_true=0.0)
    return p, half_to_packed(z)


# four slots, two slots and one buffer of the column stage; rows of 32, 64, 128
# and 512 values
@pytest.mark.parametrize("nx,ny", [(64, 64), (128, 512), (256, 256), (1024, 96), (64, 1024), (96, 1536), (128, 2048)])
@pytest.mark.parametrize("e", [-900, -1020, -1040])
def test_quotients_of_damped_fields_round_as_divisions(nx, ny, e):
    from fsibe_2d_amd.solver import Batch, FluidSim

    p, vk = _flow(nx, ny, 2.0 ** e)
    b = Batch([p], [vk])
    b.run(4)
    s = FluidSim(p)
    s.set_vortk(vk)
    s.run(4)
    for f in ("vortk", "u1", "u2", "vor_mean"):
        got, want = s.field(f), b.members[0].field(f)
        assert np.abs(want).max() > 0.0, f
        assert np.array_equal(got, want), (f, np.abs(got - want).max())
    s.close()
    b.close()
