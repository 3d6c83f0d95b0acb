"""The structured module's particle diagnostics (kinetic energy over 3P entries,
momenta over P) at the edges of their common chunk of 4096 particles, in the
caller's order, bit for bit against the CPU restatement; the largest has more
partials of the kinetic energy than a chunk of the final sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("P", [1, 255, 1365, 1366, 2731, 4096, 4097, 9000, 5600000])
def test_rows(orc, P):
    import picgolf
    from picgolf.core2d3v import Config2D3V, SpeciesConfig
    rng = np.random.default_rng(P)
    n = 3 if P < 10000 else 1
    xyv = np.vstack([rng.uniform(0, 1, P), rng.uniform(0, 1, P), 0.5 * rng.standard_normal((3, P))])
    sc = SpeciesConfig(P=P, shape="bspline2", charge=-1.0, mass=1.0, weight=1 / P)
    cfg = Config2D3V(NX=16, NY=16, dt=0.05, species=[sc], B0=(0.0, 0.0, 2.0), ntskip=1, ngskip=1)
    with picgolf.Context2D3V(cfg) as c:
        c.upload(0, xyv)
        rows = c.run(n)
    _, _, ref, _, _ = orc.run23(16, 16, 1.0, 1.0, 0.05, cfg.B0,
                                [dict(shape="bspline2", charge=-1.0, mass=1.0, weight=1 / P, xyv=xyv)], n)
    assert same(rows, ref)
