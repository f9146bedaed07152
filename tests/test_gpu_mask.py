"""The mask kernel where its passes over the primitive list have edges: more
primitives than threads of a workgroup (two groups of the list), many rounds
of 64 primitives on one tile, tiles that few or none meet, a sharp trailing
edge in the last round, walls below, and the batched form (256 threads per
workgroup).  Against the oracle at 1e-12 of the field's norm: both evaluate
the same expressions with an erf good to a few units in the last place."""
import numpy as np
import pytest

from tests.conftest import rel_l2
from tests.test_gpu_variants import _pair

pytestmark = pytest.mark.gpu

CASES = {
    "two groups": dict(nx=64, ny=64, ns=300),
    "two groups, sharp end": dict(nx=64, ny=64, ns=300, iSharpTrailing=1),
    "one group and one": dict(nx=64, ny=64, ns=257),
    "walls": dict(nx=96, ny=64, ns=200, iWalls=1, h_channel=0.4),
    "tilted, few per tile": dict(nx=256, ny=192, ns=40, iSharpTrailing=1, AngleBeam=30.0),
    "sharp mask": dict(nx=64, ny=128, ns=300, N_smooth=0.0, AngleBeam=-20.0),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_mask_against_the_oracle(name, oracle_mod):
    o, g = _pair(oracle_mod, dt_fixed=1e-4, iSaveBeam=0, **CASES[name])
    o.run(1)
    g.run(1)
    for k in ("mask", "maskvx", "maskvy"):
        assert rel_l2(g.field(k), o.field(k)) <= 1e-12, k
    assert np.abs(g.field("mask")).max() > 0.0


def test_batched_mask_is_the_single_one():
    from fsibe_2d_amd import Params
    from fsibe_2d_amd.solver import Batch, FluidSim

    ps = [Params(nx=64, ny=64, ns=n, dt_fixed=1e-4, iSaveBeam=0, iSharpTrailing=e) for n, e in ((300, 0), (130, 1))]
    b = Batch(ps, [None, None])
    b.run(2)
    for p, m in zip(ps, b.members):
        s = FluidSim(p)
        s.run(2)
        for k in ("mask", "maskvx", "maskvy"):
            assert np.array_equal(m.field(k), s.field(k)), k
        s.close()
    b.close()
