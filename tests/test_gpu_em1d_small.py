"""The 1D electromagnetic fixed point around the edges of its short chain of
kernels (64 particles to a block, 4096 particles, 256 cells and 4 sweeps at
most; the general chain beyond), bit for bit against the CPU restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("N,P,sort,max_sweeps", [
    (8, 1, 1, 3), (8, 65, 0, 3), (16, 64, 1, 1), (32, 63, 1, 4), (64, 1000, 1, 2), (128, 2048, 0, 3),
    (256, 4096, 1, 3), (256, 4097, 1, 3), (512, 300, 1, 3), (64, 500, 1, 5), (8, 5000, 0, 3), (16, 5000, 1, 3)])
def test_run_bitwise(orc, N, P, sort, max_sweeps):
    import picgolf
    rng = np.random.default_rng(N + P)
    eps = 0.1
    dt, w = eps ** 2 / N / 2, 400 / P * N
    x, v = rng.random(P), rng.standard_normal((3, P))
    x[::7] = x[0]                                    # ties of the sort
    x[1::11] = np.round(x[1::11] * N) / N            # cell edges and centres
    if P > 8:
        x[2], x[3], x[4] = 0.25 / N, 1 - 0.25 / N, 0.0   # centres whose wrapped cell is N cells away
    with picgolf.ContextEM1D(picgolf.ConfigEM1D(N=N, P=P, eps=eps, dt=dt, w=w, sort=bool(sort),
                                                max_sweeps=max_sweeps)) as c:
        for _ in range(2):                           # a second upload starts afresh
            c.upload(x, v)
            f1, s1 = c.run(3)
            _, s2 = c.run(2, want_fields=False)
            f3, s3 = c.run(2)
            xg, vg, Eg, Bg = c.download()
    xo, vo, Eo, Bo, _, fo, so = orc.em_run(N, eps, dt, w, x, v, 7, sort=sort, max_sweeps=max_sweeps)
    assert np.array_equal(np.concatenate([s1, s2, s3]), so)
    assert same(f1, fo[:, :3]) and same(f3, fo[:, 5:])
    assert same(xg, xo) and same(vg, vo) and same(Eg, Eo) and same(Bg, Bo)


@pytest.mark.parametrize("N", [8, 16, 64])
def test_operators_where_centres_wrap(orc, N):
    """Centres in and out of the box: the centre's cell wraps, the centre does not."""
    import picgolf
    rng = np.random.default_rng(N)
    k = rng.integers(-3 * N, 4 * N, 400)
    y = np.concatenate([7 * rng.random(1500) - 3, k / N, (k + 0.5) / N, np.nextafter((k + 0.5) / N, 9),
                        1 + rng.random(100) / N, -rng.random(100) / N, 1e12 * rng.random(20)])
    u = rng.standard_normal((3, y.size))
    e3, b2 = rng.standard_normal((3, N)), rng.standard_normal((2, N))
    with picgolf.ContextEM1D(picgolf.ConfigEM1D(N=N, P=64, eps=0.1, dt=1e-3, w=0.5)) as c:
        assert same(c.deposit(y, 0.5), orc.em_deposit(N, y, 0.5))
        assert same(c.deposit(y, 0.5, u=u[0]), orc.em_deposit(N, y, 0.5, u=u[0]))
        v = c.push(y, e3, b2, u)
    ref = np.stack([orc.em_push(y[p], *e3, *b2, 1e-3, u[:, p]) for p in range(y.size)], axis=1)
    assert same(v, ref)
