"""The number of kernels that a block's step launches, as cfdx_block_timing gives it (GPU): a viscous stage takes its viscous
tiles and face sweeps in one launch and its update in another; timed, with the overlap off or with other tile shapes they are
five. Side conditions add one launch for i and j together and one for any other direction."""
import math

import pytest

import cfdx
from test_gpu_bounded import CASES, perturbed

pytestmark = pytest.mark.gpu
MACH = 0.4


@pytest.fixture(scope="module")
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    return cfdx.Ctx(0)


def make(ctx, name, prm):
    if name == "periodic":
        b = cfdx.Block(12, 10, 8, ctx=ctx)
        b.init_case(grid="sinusoid", length=(2 * math.pi,) * 3, amp=0.02, phases=(0.3, 1.1, 2.0), init="tgv", mach=MACH)
        return b
    d, xyz, geo, mach, aoa, _ = CASES[name]()
    b = cfdx.Block.of(cfdx.BlockDesc.from_buffer_copy(d), ctx=ctx)
    b.set_geometry_soa(geo)
    b.configure(MACH, 0.0, prm)
    b.set_flow(perturbed(xyz[cfdx.owned_index(d)], MACH, aoa))
    return b


@pytest.mark.parametrize("name, sides", [("periodic", 0), ("cgrid", 1), ("box-all-bounded", 2)])
@pytest.mark.parametrize("viscous", [True, False], ids=["viscous", "inviscid"])
def test_launches_of_a_step(ctx, name, sides, viscous):
    prm = cfdx.default_params(mach=MACH, reyl=800.0) if viscous else cfdx.euler_params()
    apart = 5 if viscous else 4
    b = make(ctx, name, prm)

    def count(steps):
        b.step(steps, MACH, 1e-5, prm)
        return b.timing()["launches"]

    assert count(1) == 3 * (2 + sides)
    assert count(2) == 6 * (2 + sides)
    b.set_timing(True)
    assert count(1) == 3 * (apart + sides)
    b.set_timing(False)
    ctx.set_overlap(False)
    try:
        assert count(1) == 3 * (apart + sides)
    finally:
        ctx.set_overlap(True)
    b.set_tiles((1, 1, 2, 1, 4))
    assert count(1) == 3 * (apart + sides)
    b.close()
