"""The launch that takes a stage's viscous node tiles and face sweeps together (GPU): bitwise the results
of the kernels run one after the other, over the shapes where its tile bookkeeping can go wrong: the
smallest blocks, partial tiles in every direction, fewer tiles than XCDs, kinds with very different
tile counts, bounded blocks with their shells, inviscid blocks, lists of both."""
import math

import numpy as np
import pytest

import cfdx
from test_gpu_bounded import CASES, perturbed

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "u", "v", "w", "p", "mu")


@pytest.fixture(scope="module")
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    c = cfdx.Ctx(0)
    yield c
    c.set_overlap(True)


def periodic(ctx, shape, precision, prm):
    b = cfdx.Block(*shape, precision=precision, ctx=ctx)
    b.init_case(grid="sinusoid", length=(2 * math.pi,) * 3, amp=0.05 * 2 * math.pi / max(shape), phases=(0.3, 1.1, 2.0),
                init="tgv", mach=0.3)
    b.configure(0.3, 0.02 * 2 * math.pi / max(shape), prm)
    return b


def bounded(ctx, name, precision):
    d, xyz, geo, mach, aoa, pk = CASES[name]()
    prm = cfdx.default_params(**pk)
    b = cfdx.Block(d.ni, d.nj, d.nk, precision=precision, ctx=ctx, desc=cfdx.BlockDesc.from_buffer_copy(d))
    b.set_geometry_soa(geo)
    b.configure(mach, 0.0, prm)
    b.set_flow(perturbed(xyz[cfdx.owned_index(d)], mach, aoa))
    b.configure(mach, 0.5 * b.cfl_dt(0.5), prm)
    return b


def both(ctx, make, steps):
    """The flows of make()'s blocks after `steps` batch steps, together and apart."""
    out = []
    for on in (True, False):
        ctx.set_overlap(on)
        blocks = make()
        q = cfdx.Batch(blocks[0].precision, ctx)
        for b in blocks:
            q.add(b)
        q.step(steps, False)
        out.append([b.get_flow() for b in blocks])
        q.close()
        for b in blocks:
            b.close()
    ctx.set_overlap(True)
    return out


def same(pair):
    for a, r in zip(*pair):
        for f in FIELDS:
            assert np.array_equal(a[f], r[f]), f
            assert np.isfinite(a[f]).all(), f


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("viscous", [True, False], ids=["viscous", "inviscid"])
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 3, 90), (130, 3, 5), (3, 75, 4), (64, 16, 16), (65, 17, 19), (128, 4, 33)],
                         ids=lambda s: "x".join(map(str, s)))
def test_one_launch_gives_the_bits_of_the_kernels_apart(ctx, shape, viscous, precision):
    prm = cfdx.default_params(mach=0.3, reyl=900.0) if viscous else cfdx.euler_params()
    same(both(ctx, lambda: [periodic(ctx, shape, precision, prm)], 2))


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
def test_one_launch_over_a_mixed_list(ctx, precision):
    """Bounded and periodic, viscous and inviscid blocks of uneven sizes in one list."""
    visc, inv = cfdx.default_params(mach=0.3, reyl=900.0), cfdx.euler_params()

    def make():
        return ([periodic(ctx, s, precision, p) for s, p in (((5, 4, 3), visc), ((40, 21, 9), inv), ((66, 10, 7), visc))]
                + [bounded(ctx, n, precision) for n in CASES])
    same(both(ctx, make, 2))


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
def test_streaming_accesses_give_the_same_bits(ctx, precision):
    """A block past the last-level cache with rows of whole 64-byte pieces steps with non-temporal
    accesses; in a list with a block whose rows are not, with plain ones: a hint, so the same bits."""
    prm = cfdx.default_params(mach=0.3, reyl=900.0)
    shape = (112, 112, 112)
    alone = periodic(ctx, shape, precision, prm)
    alone.step(2, 0.3, 0.02 * 2 * math.pi / 112, prm)
    want = alone.get_flow()
    alone.close()
    b, odd = periodic(ctx, shape, precision, prm), periodic(ctx, (7, 5, 9), precision, prm)
    q = cfdx.Batch(precision, ctx)
    q.add(b)
    q.add(odd)
    q.step(2, False)
    got = b.get_flow()
    q.close()
    for x in (b, odd):
        x.close()
    for f in FIELDS:
        assert np.array_equal(got[f], want[f]), f


@pytest.mark.parametrize("tiles", [(0, 0, 0, 0, 4), (1, 1, 2, 1, 4)], ids=["default", "forked"])
@pytest.mark.parametrize("graph", [True, False], ids=["graph", "eager"])
def test_groups_of_a_batch_give_the_bits_of_each_block_alone(ctx, graph, tiles):
    """More blocks than one cache-sized group holds (134 MB each of three, and small ones, bounded and
    inviscid among them), also after a block has left: every block as if stepped alone."""
    visc, inv = cfdx.default_params(mach=0.3, reyl=900.0), cfdx.euler_params()

    def make():
        return ([periodic(ctx, s, cfdx.FP64, p) for s, p in (((12, 10, 8), visc), ((64, 64, 64), visc), ((64, 64, 64), inv),
                                                             ((33, 20, 9), inv), ((64, 64, 64), visc))]
                + [bounded(ctx, "cgrid", cfdx.FP64)])
    want = []
    for b, n in zip(make(), (3, 3, 3, 2, 3, 3)):
        q = cfdx.Batch(cfdx.FP64, ctx)
        q.add(b)
        q.step(n, False)
        want.append(b.get_flow())
        q.close()
        b.close()
    blocks = make()
    q = cfdx.Batch(cfdx.FP64, ctx)
    q.set_tiles(tiles)
    for b in blocks:
        q.add(b)
    q.step(2, graph)
    q.remove(blocks[3])
    q.step(1, graph)
    for b, w in zip(blocks, want):
        got = b.get_flow()
        for f in FIELDS:
            assert np.array_equal(got[f], w[f]), f
    q.close()
    for b in blocks:
        b.close()


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("side", ["periodic", "bounded"])
def test_line_tiles_give_the_bits_of_rectangular_ones(ctx, side, precision):
    """The i sweep's default tiles take 256 faces (fewer on lines of under 17) of the lines one after the other:
    line lengths about the points where the faces of a tile change, its lines end, or it holds many."""
    prm = cfdx.default_params(mach=0.3, reyl=900.0)

    def make(ni):
        shape = (ni, 5 if ni > 100 else 11, 7)
        if side == "periodic":
            return periodic(ctx, shape, precision, prm)
        d = cfdx.BlockDesc(*shape[:1], shape[1] + 4, shape[2], 6, precision)
        d.bc[0], d.bc[1] = cfdx.BC_EXTRAP, cfdx.BC_OUTFLOW
        xyz, geo = cfdx.box_geometry(d, (0.1 * ni, 1.1, 0.9), 0.005, (0.3, 1.2, 2.1))
        b = cfdx.Block.of(d, ctx=ctx)
        b.set_geometry_soa(geo)
        b.configure(0.3, 0.0, prm)
        b.set_flow(perturbed(xyz[cfdx.owned_index(d)], 0.3, 2.0))
        b.configure(0.3, 0.5 * b.cfl_dt(0.5), prm)
        return b

    low = 3 if side == "periodic" else 7
    for ni in (low, low + 1, 12, 15, 16, 17, 18, 51, 63, 64, 65, 127, 128, 255, 256, 257, 511):
        out = []
        for variant in (0, 1, 2):
            b = make(ni)
            b.set_tiles((variant, 0, 0, 0, 4))
            b.step(2, 0.3, b.dt, prm)
            out.append(b.get_flow())
            b.close()
        for f in FIELDS:
            assert np.isfinite(out[0][f]).all(), (ni, f)
            assert np.array_equal(out[0][f], out[1][f]) and np.array_equal(out[0][f], out[2][f]), (ni, f)
