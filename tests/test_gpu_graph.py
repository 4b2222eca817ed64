"""Batches that step from a captured graph (GPU): tile shapes or a grid cap that fork a stage onto the second
stream, the only lists that cfdx_batch_step captures. A graph is dropped, and the step captured again, when
the overlap switch, the context's stream, the tiles, the grid or the blocks change; every replay gives the bits of
the blocks stepped alone, with eager work and synchronisations between the replays."""
import numpy as np
import pytest

import cfdx
from cfdx import serve
from test_gpu_serve import small_stream
from test_gpu_tiles import ragged

pytestmark = pytest.mark.gpu
FIELDS = ("rho", "u", "v", "w", "p", "mu")
FORKED = (1, 1, 2, 1, 4)
SHAPES = [(24, 16, 8), (19, 13, 11)]
PRM = dict(mach=0.2, reyl=900.0)


@pytest.fixture()
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    c = cfdx.Ctx(0)
    yield c
    c.close()


def block(ctx, shape, precision=cfdx.MIXED):
    b = ragged(ctx, precision, *shape)
    prm = cfdx.default_params(**PRM)
    b.configure(0.2, 0.0, prm)
    b.configure(0.2, 0.5 * b.cfl_dt(0.5), prm)
    return b


def alone(ctx, shape, steps, precision=cfdx.MIXED):
    """The block's flow after each number of steps in `steps`, stepped eagerly by itself."""
    b, out, done = block(ctx, shape, precision), {}, 0
    for n in steps:
        b.step(n - done, 0.2, b.dt, cfdx.default_params(**PRM))
        out[done := n] = b.get_flow()
    b.close()
    return out


def same(got, want, what):
    for f in FIELDS:
        assert np.array_equal(got[f], want[f]), (what, f)


@pytest.mark.parametrize("precision", [cfdx.FP64, cfdx.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("cap", [0, 5], ids=["tiles", "grid-cap"])
def test_replays_and_recaptures(ctx, cap, precision):
    want = [alone(ctx, s, range(2, 15, 2), precision) for s in SHAPES]
    blocks = [block(ctx, s, precision) for s in SHAPES]
    q = cfdx.Batch(precision, ctx)
    if cap:
        q.set_grid(cap)
    else:
        q.set_tiles(FORKED)
    for b in blocks:
        q.add(b)
    eager = block(ctx, (12, 10, 8), precision)

    def check(n, what):
        eager.step(1, 0.2, eager.dt, cfdx.default_params(**PRM))
        ctx.sync()
        for b, w in zip(blocks, want):
            same(b.get_flow(), w[n], what)

    q.step(2, True)
    check(2, "captured")
    q.step(2, True)
    check(4, "replayed")
    ctx.set_overlap(False)
    q.step(2, True)
    check(6, "overlap off")
    ctx.set_overlap(True)
    q.step(2, True)
    check(8, "overlap on again")
    other = cfdx.Ctx(0)
    assert cfdx._lib.cfdx_ctx_set_stream(ctx.h, cfdx._lib.cfdx_ctx_stream(other.h)) == 0
    q.step(2, True)
    check(10, "another stream")
    assert cfdx._lib.cfdx_ctx_set_stream(ctx.h, None) == 0
    q.step(1, True)
    q.step(1, True)
    check(12, "a stream of its own again")
    q.set_tiles((2, 1, 1, 2, 4))
    q.step(2, True)
    check(14, "other tiles")
    q.close()
    for b in blocks + [eager]:
        b.close()
    other.close()


def test_a_destroyed_block_takes_the_graph_with_it(ctx):
    want = alone(ctx, SHAPES[0], (4, 6))
    a, b = (block(ctx, s) for s in SHAPES)
    q = cfdx.Batch(cfdx.MIXED, ctx)
    q.set_tiles(FORKED)
    q.add(a)
    q.add(b)
    q.step(2, True)
    ctx.sync()
    b.close()                       # not removed first
    assert len(q) == 1
    c = block(ctx, SHAPES[1])       # may take b's memory from the pool
    before = c.get_flow()
    q.step(2, True)
    same(a.get_flow(), want[4], "after the block left")
    q.step(2, True)
    same(a.get_flow(), want[6], "replayed")
    same(c.get_flow(), before, "a block that is in no batch")
    q.close()
    a.close()
    c.close()


@pytest.mark.parametrize("clock", ["steps", "wall"])
def test_served_requests_of_a_batch_that_captures(ctx, clock):
    """A server whose batch has a capped grid captures its step again at every admission and retirement, on the wall
    clock beside the set-up thread's own library calls: every result is that of the request alone."""
    reqs = small_stream()
    for r in reqs:
        r.nsteps *= 3
        if clock == "wall":
            r.arrival *= 1e-3
    srv = serve.Server(precision=cfdx.MIXED, ctx=ctx, reserve_bytes=0, chunk=4, graph=True, grid_cap=9)
    res = srv.run(reqs, clock=clock)
    srv.close()
    assert sorted(res) == [r.rid for r in reqs] and srv.peak_active >= 2
    for r in reqs:
        want = serve.run_alone(r, cfdx.MIXED, ctx)
        assert res[r.rid].dt == want.dt
        for f in FIELDS[:5]:
            assert np.array_equal(res[r.rid].flow[f], want.flow[f]), (r.rid, f)
