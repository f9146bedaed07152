"""Which of two routes a step takes where the choice depends on more than the
lengths: the fused column stage for 4096-point columns (fsibe_hip.hip,
with_col_step).  The route shows in the launches that the profile counts for
K5, which only the separate stages have; either route gives the same bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COLS_VORTK_N1, NCLASS = 6, 13


def _flow(nx, ny):
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.inputs import half_to_packed, normals
    from fsibe_2d_amd.solver import FluidSim

    z = np.zeros((ny, nx // 2), dtype=np.complex128)
    g = normals(5, 2 * 6 * 7).reshape(2, 6, 7)
    z[1:7, :7] = 1e-3 * (g[0] + 1j * g[1])
    z[1:7, 0] = 0.0
    s = FluidSim(Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=1e-4, iBeam=0, iSaveBeam=0, iSponge=0, iMotion=0,
                        iMeanVelocity=4))
    s.set_vortk(half_to_packed(z))
    return s


def _k5(s, steps):
    """launches of K5 in calls of one step each (a timed run forms nothing ahead)"""
    from fsibe_2d_amd._lib import check, lib

    L = lib()
    check(L.fsibe_profile_enable(s.h, -1))
    for _ in range(steps):
        s.run(1)
    ms, cnt = (C.c_double * NCLASS)(), (C.c_longlong * NCLASS)()
    L.fsibe_profile_read(s.h, ms, cnt, NCLASS)
    check(L.fsibe_profile_enable(s.h, 0))
    return int(cnt[COLS_VORTK_N1])


# lengths on either side of each line of the rule, and whether a step without a
# following one takes the separate stages; in a call of several steps 64, 192,
# 216 and 288 x 4096 take the fused one
@pytest.mark.parametrize("nx,ny,separate", [
    (48, 4096, True), (64, 4096, True), (128, 4096, True), (192, 4096, True), (216, 4096, True), (256, 4096, True),
    (288, 4096, True), (384, 4096, False), (64, 2048, False), (128, 1024, False)])
def test_column_stage_of_long_columns(nx, ny, separate):
    a, b = _flow(nx, ny), _flow(nx, ny)
    assert _k5(a, 4) == (4 if separate else 0)
    b.run(4)
    for f in ("vortk", "nlk", "u1", "u2", "vor_mean"):
        assert np.array_equal(a.field(f), b.field(f)), f
    a.close()
    b.close()


@pytest.mark.parametrize("nx,ny", [(1024, 1536), (1024, 2048), (256, 768)])
@pytest.mark.parametrize("loads", [0, 1])
def test_row_stage_with_and_without_the_next_term(nx, ny, loads):
    """rows of 128, and of 512 beyond 1024 of them without the pressure, take
    the row stage where the next step's term is formed and K6 alone otherwise:
    the same operations, so the fields, row sums and CFL maximum agree bit for bit"""
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.solver import FluidSim

    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=1e-4, iSaveBeam=loads, iSponge=0)
    a, b = FluidSim(p), FluidSim(p)
    oa = a.run(3)
    for _ in range(3):
        ob = b.run(1)
    for f in ("vortk", "nlk", "u1", "u2", "vor_mean"):
        assert np.array_equal(a.field(f), b.field(f)), f
    for k in ("dt1", "u_max", "Force", "energies"):
        assert oa[k] == ob[k], k
    a.close()
    b.close()


@pytest.mark.parametrize("nx,ny", [(1024, 1152), (1024, 1296), (1024, 1024)])
def test_rows_of_512_against_the_oracle(nx, ny, oracle_mod):
    """K6 alone (1152 rows: a last round of an eighth) and the row stage (1296:
    more than a quarter; 1024: one round), with the pressure, within the suite's
    1e-10 of the oracle's fields"""
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.solver import FluidSim
    from tests.conftest import rel_l2
    from tests.test_gpu_variants import PKEYS

    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=1e-4)
    o = oracle_mod.Oracle(oracle_mod.make_params(**{k: getattr(p, k) for k in PKEYS}))
    o.run(2)
    s = FluidSim(p)
    s.run(2)
    for k in ("vortk", "u1", "u2", "vor_mean"):
        assert rel_l2(s.field(k), o.field(k)) <= 1e-10, k
    s.close()
