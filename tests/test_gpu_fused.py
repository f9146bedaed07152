"""The fused column and row stages of the time loop (kernels_fused.hpp): a run
of several steps in one call forms each next step's dw/dy column and
convective term inside the stages of the step before, a run of one step per
call forms them with kernels of their own.  Both do the same operations on
every value, so the fields and the loads agree bit for bit: no tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# every shape of the two stages, and lengths that have one of them or none
GRIDS = [(64, 64), (128, 96), (96, 128), (192, 192), (256, 64), (64, 256), (384, 384), (512, 192), (1024, 768),
         (256, 1024), (384, 1536), (72, 96), (128, 2048), (1024, 1024)]


def _run(p, steps, split):
    from fsibe_2d_amd.inputs import half_to_packed, normals
    from fsibe_2d_amd.solver import FluidSim

    z = np.zeros((p.ny, p.nx // 2), dtype=np.complex128)
    g = normals(5, 2 * 6 * 7).reshape(2, 6, 7)
    z[1:7, :7] = 1e-3 * (g[0] + 1j * g[1])
    z[1:7, 0] = 0.0  # kx = 0 needs its conjugate row
    s = FluidSim(p)
    s.set_vortk(half_to_packed(z))
    if split:
        for _ in range(steps):
            out = s.run(1)
    else:
        out = s.run(steps)
    got = [s.field(f) for f in ("vortk", "nlk", "u1", "u2", "vor_mean")]
    b = s.beam()
    s.close()
    return got, out, b


@pytest.mark.parametrize("nx,ny", GRIDS)
@pytest.mark.parametrize("kind", ["beam", "loads off", "no body"])
def test_one_call_of_several_steps_equals_several_calls_of_one(nx, ny, kind):
    from fsibe_2d_amd import Params

    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=2e-4)
    if kind == "loads off":
        p = p.replace(iSaveBeam=0, iSponge=0)
    if kind == "no body":
        p = p.replace(iBeam=0, iSaveBeam=0, iSponge=0, iMotion=0, iMeanVelocity=4)
    a, oa, ba = _run(p, 4, False)
    b, ob, bb = _run(p, 4, True)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    for k in ("dt1", "u_max", "Force", "Force_press", "energies", "bsi"):
        assert oa[k] == ob[k], k
    assert np.array_equal(ba["pressure"], bb["pressure"]) and np.array_equal(ba["tau"], bb["tau"])


@pytest.mark.parametrize("nx,ny", [(64, 64), (128, 96), (64, 128), (108, 192), (256, 256), (128, 384), (192, 512),
                                   (256, 768), (128, 1024), (64, 1536)])
def test_pressure_stage_equals_the_batched_one(nx, ny):
    """the single path's pressure stage (two slots per column) against the
    batch's (columns staged in LDS): the same operations, so the loads agree
    bit for bit; 108 x 192 has an odd number of columns and shares the code"""
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.solver import Batch, FluidSim

    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=2e-4)
    b = Batch([p], [None])
    b.run(3)
    s = FluidSim(p)
    out, want = s.run(3), b.members[0].step_out()
    for k in ("Force_press", "bsi"):
        assert out[k] == want[k], k
    for k in ("pressure", "tau"):
        assert np.array_equal(s.beam()[k], b.members[0].beam()[k]), k
    assert np.abs(s.beam()["pressure"]).max() > 0.0
    s.close()
    b.close()


@pytest.mark.parametrize("nx,ny", [(64, 64), (96, 128), (192, 96), (72, 256), (128, 1024), (384, 64), (512, 128)])
@pytest.mark.parametrize("idealis", [0, 1])
def test_dealiased_columns_against_the_oracle(nx, ny, idealis, oracle_mod):
    """the stages leave out what dealiasing makes zero: from an initial
    vorticity with every mode set (so the first step's inputs are not
    dealiased), with and without dealiasing, in one call and step by step,
    within the suite's 1e-10 of the oracle's fields"""
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.inputs import half_to_packed, normals
    from fsibe_2d_amd.solver import FluidSim
    from tests.conftest import rel_l2
    from tests.test_gpu_variants import PKEYS

    p = Params(nx=nx, ny=ny, ns=33, nu=2e-3, dt_fixed=1e-4, idealis=idealis)
    H = nx // 2
    g = np.array(normals(11, 2 * ny * H)).reshape(2, ny, H)
    z = 1e-6 * (g[0] + 1j * g[1])
    z[ny // 2] = 0.0
    z[0, 0] = 0.0
    for j in range(1, ny // 2):  # kx = 0: the spectrum of a real field
        z[-j, 0] = np.conj(z[j, 0])
    vk = half_to_packed(z)
    o = oracle_mod.Oracle(oracle_mod.make_params(**{k: getattr(p, k) for k in PKEYS}))
    o.set_vortk(vk)
    o.run(4)
    for split in (False, True):
        s = FluidSim(p)
        s.set_vortk(vk)
        for n in (1, 1, 1, 1) if split else (4,):
            s.run(n)
        # (nlk is not comparable: the reference multiplies the older level by
        # its viscous factor in place, NavierStokes.f90:485)
        for k in ("vortk", "u1", "u2", "vor_mean"):
            assert rel_l2(s.field(k), o.field(k)) <= 1e-10, (k, split)
        s.close()
