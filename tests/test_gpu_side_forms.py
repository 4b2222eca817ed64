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


@PRECISIONS
@pytest.mark.parametrize("periodic", [4, 0, 6], ids=["bounded-ij", "bounded-ijk", "bounded-i"])
def test_a_uniform_state_has_no_derivative_at_the_sides(ctx, periodic, precision):
    """A uniform state on a uniform grid: every difference of two points is exactly 0, so every one-sided form and
    the central one give exactly 0, and with them the viscous fluxes, their divergence and the whole right-hand
    side. (Weighted sums of the values leave rounding of the state's own size, 1e-17 of it.) The primitives are numbers
    of 32 bits: a mixed block rounds those of its side nodes to them."""
    d = desc((12, 10, 9), periodic, (cfdx.BC_EXTRAP,) * 6, precision)
    for q in range(3):
        if (periodic >> q) & 1:
            d.bc[2 * q] = d.bc[2 * q + 1] = 0
    dims, _ = cfdx.padded(d)
    geo = np.zeros((22, int(np.prod(dims))))
    geo[0] = 0.07                             # det
    for c, m in zip((1, 5, 9), (2.3, 3.1, 1.7)):
        geo[c] = m                            # zeta_x, eta_y, xi_z
        geo[c + 9] = m                        # the same on the faces of that direction
    geo[19:] = 0.07
    prm = cfdx.default_params(mach=0.4, reyl=300.0)
    f = cfdx.freestream(d.ni * d.nj * d.nk, 0.4, 3.0)
    for c, x in zip(("rho", "u", "v", "w", "p"), (1.125, 0.6875, 0.3125, -0.1875, 3.25)):
        f[c] = x
    b = cfdx.Block.of(d, ctx=ctx)
    b.set_geometry_soa(geo)
    b.configure(0.4, 0.0, prm)
    b.set_flow(f)
    L = b.rhs(prm)
    b.close()
    assert (L == 0).all(), np.abs(L).max()
