"""Downloads through the staging buffers (csrc/hostcopy.hip): sizes around the
short list's limit and the chunk (2^17 values), every format, and several
threads at once, against what was uploaded."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("P", [1, 1000, 2 ** 17 - 17, 2 ** 17 - 16, 2 ** 17 + 1, 2 ** 20 + 3])
def test_roundtrip_1d(P, precision):
    import picgolf
    N, dt = 32, 1 / 256
    rng = np.random.default_rng(P)
    x, v, E = rng.random(P), rng.standard_normal(P), rng.standard_normal(N)
    with picgolf.Context(picgolf.Config(N=N, P=P, W=100.0, dt=dt, precision=precision)) as c:
        c.upload(x, v, E)
        gx, gv, gE = c.download()
        assert np.array_equal(c.download_field(), E)
    assert np.array_equal(gE, E)
    if precision == "fp64":
        assert np.array_equal(gx, x) and np.array_equal(gv, v)
    else:
        # the 2^-32 grid of the box, and a hi + lo float pair of v (2^-48 of it)
        assert np.array_equal(gx, np.rint(x * 2.0 ** 32) % 2.0 ** 32 / 2.0 ** 32)
        assert np.max(np.abs(gv - v)) <= 2.0 ** -47 * np.max(np.abs(v))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("P", [7, 40000, 300001])
def test_caller_order_2d(P, precision):
    import picgolf
    rng = np.random.default_rng(P)
    s = [1.0 - rng.integers(0, 2 ** 32, P) / 2.0 ** 32 for _ in range(2)]
    s += [rng.standard_normal(P).astype(np.float32).astype(np.float64) for _ in range(3)]
    with picgolf.Context2D(picgolf.Config2D(NX=64, NY=32, P=P, dt=1 / 512, w=1.0 / P, B0=1.0,
                                            precision=precision)) as c:
        c.upload(*s)
        got = c.download()
        again = c.download()
        assert all(np.array_equal(a, b) for a, b in zip(got[:5], s))
        assert all(np.array_equal(a, b) for a, b in zip(got, again))
        c.run(3)                                     # the run goes on from the same state
        one = c.download()
    with picgolf.Context2D(c.cfg) as d:
        d.upload(*s)
        d.run(3)
        assert all(np.array_equal(a, b) for a, b in zip(one, d.download()))


def test_threads():
    import picgolf
    P, bad = 400000, []

    def one(k):
        rng = np.random.default_rng(k)
        x, v = rng.random(P), rng.standard_normal(P)
        with picgolf.Context(picgolf.Config(N=64, P=P, W=100.0, dt=1 / 256)) as c:
            c.upload(x, v)
            for _ in range(3):
                gx, gv, _ = c.download()
                if not (np.array_equal(gx, x) and np.array_equal(gv, v)):
                    bad.append(k)

    ts = [threading.Thread(target=one, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
