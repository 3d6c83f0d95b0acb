"""The Gaussian kernels at centres where the edge intervals meet (cell edges
and cell centres) and at centres too far out for them, bit for bit against the
CPU restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,R", [(8, 7), (64, 6), (64, 7), (4096, 7)])
def test_edge_centres_bitwise(orc, N, R):
    import picgolf
    rng = np.random.default_rng(N + R)
    k = rng.integers(-N, 2 * N, 300)
    x = np.concatenate([k / N, (k + 0.5) / N, np.nextafter((k + 0.5) / N, 9), np.nextafter((k + 0.5) / N, -9),
                        (k + rng.choice([1e-9, -1e-9, 0.25, 0.15625], 300)) / N, 1e12 * rng.random(20),
                        2.0 ** 51 / N * (1 + 0.9 * rng.random(20)), -2.0 ** 51 / N * (1 + 0.9 * rng.random(20)), rng.random(77)])
    P, w, E = x.size, 400.0 / x.size * N, rng.standard_normal(N)
    V = rng.standard_normal(P)
    with picgolf.Context(picgolf.Config(N=N, P=P, W=400.0, dt=1 / (6 * N), shape=R)) as c:
        got = c.deposit(x, w=w, shape=R)
        v = np.zeros(P)
        c.push_midpoint(x, V, x, v, E, 1 / (6 * N), shape=R)
    assert np.array_equal(got.view(np.int64), orc.deposit(N, R, x, w=w).view(np.int64))
    ref = orc.push_midpoint(N, R, x, V, x, E, 1 / (6 * N))
    assert np.array_equal(v.view(np.int64), ref.view(np.int64))


@pytest.mark.parametrize("R", [6, 7])
def test_every_weight_of_many_centres_bitwise(orc, R):
    """The device's own arithmetic (its reciprocals above all): a field of one
    cell makes the gather a single weight, at random centres and at centres
    with an edge within a few roundings of a branch point of erf."""
    import picgolf
    N, M = 16, 150000
    rng = np.random.default_rng(R)
    z = np.repeat([0.84375, 1.0, 1.25, 2.0, 1 / 0.35, 3.0, 4.0, 5.0, 6.0, 2.0 ** -28], 1200)
    z = z * (1 + rng.integers(-6, 7, z.size) * 2.0 ** -52) * rng.choice([-1.0, 1.0], z.size)
    k = rng.integers(1, N + 1, z.size)
    near = (k - 0.5 - z) / N                         # edge k - 1/2 at z
    near = near + rng.integers(-2, 3, z.size) * np.spacing(near)
    c = np.concatenate([rng.random(M), near])
    zero, got = np.zeros_like(c), np.zeros_like(c)
    with picgolf.Context(picgolf.Config(N=N, P=64, W=400.0, dt=1.0, shape=R)) as ctx:
        for cell in range(N):
            E = np.zeros(N)
            E[cell] = 1.0
            ctx.push_midpoint(c, zero, c, got, E, 1.0, shape=R)
            ref = orc.push_midpoint(N, R, c, zero, c, E, 1.0)
            bad = np.flatnonzero(got.view(np.int64) != ref.view(np.int64))
            assert bad.size == 0, (cell, c[bad[:5]], got[bad[:5]], ref[bad[:5]])
