"""Device-to-host copies (GPU): the sizes at which a copy changes its route (straight below 8 MB, chunks
of 4 MB through a ring of 8 pinned buffers from there) and around the chunk and ring ends give every
byte, also from two contexts on two threads at once, and after the pinned buffers were given back."""
import threading

import numpy as np
import pytest

import cfdx

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def ctx():
    if cfdx.device_count() < 1:
        pytest.skip("no HIP device")
    return cfdx.Ctx(0)


def pattern(n, seed):
    return np.random.default_rng(seed).integers(0, 256, n, dtype=np.uint8)


@pytest.mark.parametrize("n", [1, 8 * MB - 1, 8 * MB, 8 * MB + 1, 12 * MB, 32 * MB, 32 * MB + 1, 69 * MB + 5])
def test_every_byte_arrives(ctx, n):
    a = pattern(n, n)
    d = ctx.to_device(a)
    got = d.numpy()
    d.free()
    assert np.array_equal(got, a)


def test_two_threads_and_a_trim(ctx):
    wrong = []

    def copies(seed):
        c = cfdx.Ctx(0)
        for k in range(3):
            a = pattern(37 * MB + seed, 10 * seed + k)
            d = c.to_device(a)
            if not np.array_equal(d.numpy(), a):
                wrong.append((seed, k))
            d.free()
        c.close()

    threads = [threading.Thread(target=copies, args=(s,)) for s in (1, 2, 3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    ctx.pool_trim()
    copies(4)
    assert not wrong
