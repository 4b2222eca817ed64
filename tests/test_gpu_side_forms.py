"""Derivatives near the sides of bounded blocks (GPU): which side conditions take part in them, and how exact the
one-sided forms are."""
import numpy as np
import pytest

import cfdx
from test_gpu_bounded import perturbed

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "u", "v", "w", "p", "mu")
PRECISIONS = pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])


@pytest.fixture(scope="module")
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    return cfdx.Ctx(0)


def desc(dims, periodic, bc, precision):
    d = cfdx.BlockDesc(*dims, periodic, precision)
    for q in range(6):
        d.bc[q] = bc[q]
    return d


@PRECISIONS
@pytest.mark.parametrize("periodic, bc", [(6, (cfdx.BC_EXTRAP, cfdx.BC_OUTFLOW, 0, 0, 0, 0)),
                                          (2, (cfdx.BC_EXTRAP, cfdx.BC_OUTFLOW, 0, 0, cfdx.BC_WALL, cfdx.BC_WALL))],
                         ids=["bounded-i", "bounded-ik"])
def test_conditions_of_a_periodic_direction_are_ignored(ctx, periodic, bc, precision):
    """A wake cut named on the j- side of a block that is periodic in j (a descriptor whose mask was changed) has no
    effect: the bits of the block without it, in the right-hand side and after steps."""
    out = []
    for left_over in (0, cfdx.BC_WALL_CUT):
        d = desc((12, 10, 9), periodic, bc, precision)
        d.bc[2], d.cut_i0, d.cut_i1 = left_over, 4, 7
        xyz, geo = cfdx.box_geometry(d, (1.3, 1.1, 0.9), 0.02, (0.3, 1.2, 2.1))
        prm = cfdx.default_params(mach=0.4, reyl=300.0)
        b = cfdx.Block.of(d, ctx=ctx)
        b.set_geometry_soa(geo)
        b.configure(0.4, 0.0, prm)
        b.set_flow(perturbed(xyz[cfdx.owned_index(d)], 0.4, 2.0))
        L = b.rhs(prm)
        b.step(2, 0.4, 0.5 * b.cfl_dt(0.5), prm)
        out.append((L, b.get_flow()))
        b.close()
    (L0, f0), (L1, f1) = out
    assert np.array_equal(L0, L1)
    for f in FIELDS:
        assert np.array_equal(f0[f], f1[f]), f
