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
