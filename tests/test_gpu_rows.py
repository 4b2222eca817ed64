"""Blocks past the last-level cache keep each row's owned nodes on whole 64-byte pieces (GPU): a pitch of more
than the stored nodes, and a lead before a bounded direction's ghosts. Results may not depend on it: a block that
repeats a small one (rows end to end) along a periodic k gives the small one's bits in every repeat, and the two
ways its geometry comes in, from the host and built on the device, give the same right-hand side."""
import math

import numpy as np
import pytest

import cfdx
from test_gpu_bounded import perturbed

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "u", "v", "w", "p", "mu")
NK = 8


@pytest.fixture(scope="module")
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    return cfdx.Ctx(0)


def box(ni, nj, bc, periodic, precision):
    d = cfdx.BlockDesc(ni, nj, NK, periodic, precision)
    for q in range(6):
        d.bc[q] = bc[q]
    return (d, *cfdx.box_geometry(d, (1.3, 1.1, 0.4), 0.005, (0.3, 1.2, 2.1)))


def cgrid(ni, nj, precision):
    d, g = cfdx.cgrid_desc(ni, nj, NK, precision, naca=(0.02, 0.4, 0.12), n_wake=ni // 4, aoa_deg=2.0)
    return (d, *cfdx.cgrid_geometry(d, g))


# rows of 61, 61 + 6 and 70 + 6 stored nodes: no multiple of 8 or 16, and within a twelfth of the next
BLOCKS = {
    "periodic": lambda p: box(61, 43, (0,) * 6, 7, p),
    "bounded-i": lambda p: box(69, 20, (4, 3, 0, 0, 0, 0), 6, p),
    "bounded-ij": lambda p: box(69, 20, (3, 2, 1, 1, 0, 0), 4, p),
    "cgrid": lambda p: cgrid(70, 24, p),
}


def run(ctx, d, geo, flow, prm, dt, steps):
    b = cfdx.Block.of(d, ctx=ctx)
    b.set_geometry_soa(geo)
    b.configure(0.4, 0.0, prm)
    b.set_flow(flow)
    dt = dt or 0.5 * b.cfl_dt(0.5)
    b.set_monitor(True)
    b.step(steps, 0.4, dt, prm)
    out = b.get_flow(), b.residual(), b.rhs(prm)
    b.close()
    return dt, out


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name", list(BLOCKS))
def test_rows_of_a_large_block_give_the_bits_of_a_small_one(ctx, name, precision):
    d, xyz, geo = BLOCKS[name](precision)
    prm = cfdx.default_params(mach=0.4, reyl=900.0)
    flow = perturbed(xyz[cfdx.owned_index(d)], 0.4, 2.0)
    dims, _ = cfdx.padded(d)
    plane = dims[0] * dims[1]
    # past the 384 MiB of what a stage touches where blocks get whole rows
    times = (384 << 20) // ((304 if precision == cfdx.MIXED else 512) * plane * NK) + 1
    big = cfdx.BlockDesc.from_buffer_copy(d)
    big.nk = NK * times
    per_node = [cfdx.Block.bytes_for(x.ni, x.nj, x.nk, precision, desc=x) / (plane * x.nk) for x in (d, big)]
    assert per_node[1] > 1.02 * per_node[0]   # its rows are longer than their nodes
    dt, (f, r, L) = run(ctx, d, geo, flow, prm, None, 2)
    _, (F, R, LL) = run(ctx, big, np.tile(geo.reshape(22, 1, -1), (1, times, 1)).reshape(-1), np.tile(flow, times), prm, dt, 2)
    assert R == r
    for c in FIELDS:
        assert np.array_equal(F[c].reshape(times, -1), np.broadcast_to(f[c], (times, f.size))), c
    assert np.array_equal(LL.reshape(5, times, -1), np.broadcast_to(L[:, None, :], (5, times, f.size)))


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("batch", [False, True], ids=["block", "batch"])
def test_streaming_accesses_give_the_bits_of_plain_ones(ctx, batch, precision):
    """Rows that are whole 64-byte pieces as they are: the small block is stepped with plain accesses, the one that
    repeats it along k past the last-level cache with non-temporal ones, by itself and in a batch with others."""
    d, xyz, geo = box(64, 43, (0,) * 6, 7, precision)
    prm = cfdx.default_params(mach=0.4, reyl=900.0)
    flow = perturbed(xyz[cfdx.owned_index(d)], 0.4, 2.0)
    times = (384 << 20) // ((304 if precision == cfdx.MIXED else 512) * 64 * 43 * NK) + 1
    big = cfdx.BlockDesc.from_buffer_copy(d)
    big.nk = NK * times
    out, dt = [], None
    for x, n in ((d, 1), (big, times)):
        b = cfdx.Block.of(x, ctx=ctx)
        b.set_geometry_soa(np.tile(geo.reshape(22, 1, -1), (1, n, 1)).reshape(-1))
        b.configure(0.4, 0.0, prm)
        b.set_flow(np.tile(flow, n))
        dt = dt or 0.5 * b.cfl_dt(0.5)
        b.configure(0.4, dt, prm)
        if batch:
            others = [cfdx.Block(s, 12, 10, precision=precision, ctx=ctx) for s in (16, 21)]
            q = cfdx.Batch(precision, ctx)
            for o in others:
                o.init_case(grid="box", length=(2 * math.pi,) * 3, init="tgv", mach=0.4)
                o.configure(0.4, 1e-3, prm)
                q.add(o)
            q.add(b)
            q.step(2, False)
        else:
            b.step(2, 0.4, dt, prm)
        out.append(b.get_flow())
        if batch:
            q.close()
            for o in others:
                o.close()
        b.close()
    for c in FIELDS:
        assert np.array_equal(out[1][c].reshape(times, -1), np.broadcast_to(out[0][c], (times, flow.size))), c


def test_geometry_built_on_the_device_in_long_rows(ctx):
    """The sinusoidal map and its Taylor-Green state, from the host's arrays and from the device's set-up: the
    same formulas through two libraries' sines, a few ulp apart in the metrics (1e-15), and the right-hand side
    differences of fluxes about a hundred times its own size."""
    kw = dict(length=(2 * math.pi,) * 3, amp=0.02, phases=(0.3, 1.1, 2.0))
    shape, prm = (61, 120, 112), cfdx.default_params(mach=0.3, reyl=900.0)
    case = cfdx.periodic_case(*shape, grid="sinusoid", metrics="analytic", init="tgv", mach=0.3, **kw)
    out = []
    for fill in (lambda b: b.set_case(case), lambda b: b.init_case(grid="sinusoid", init="tgv", mach=0.3, **kw)):
        b = cfdx.Block(*shape, precision=cfdx.FP64, ctx=ctx)
        fill(b)
        b.configure(0.3, 1e-3, prm)
        out.append((b.get_flow(), b.rhs(prm)))
        b.close()
    for c in ("rho", "u", "v", "w", "p"):
        assert np.abs(out[0][0][c] - out[1][0][c]).max() <= 1e-13 * np.abs(out[0][0][c]).max() + 1e-14, c
    assert np.abs(out[0][1] - out[1][1]).max() <= 1e-11 * np.abs(out[0][1]).max()
