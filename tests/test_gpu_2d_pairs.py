"""The FP64 2D3V state holds (vx, vy) as pairs: upload, tile sorts, a run with
diagnostics in the caller's order and download at the edges of a diagnostics
chunk (4096 particles, 256 lanes), bit for bit against the CPU restatement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("P", [1, 255, 257, 4096, 4097, 12289])
def test_upload_diagnostics_download(orc, P):
    import picgolf
    NX, NY = 32, 64
    rng = np.random.default_rng(P)
    x, y = rng.random(P), rng.random(P)
    v = [rng.standard_normal(P) for _ in range(3)]
    cfg = picgolf.Config2D(NX=NX, NY=NY, P=P, w=0.5 / P, dt=1 / 128, B0=1.5, sort_every=2)
    with picgolf.Context2D(cfg) as c:
        for _ in range(2):
            c.upload(x, y, *v)
            for a, b in zip(c.download()[:5], (x, y, *v)):
                assert same(a, b)
        K = c.run(6)
        got = c.download()
    ref = orc.run2d(NX, NY, cfg.dt, cfg.B0, cfg.w, x, y, *v, 6, ns=2, textbook=0, nthreads=8)
    for g, r in zip(got, ref[:7]):
        assert same(g, r)
    assert same(K, ref[7])


@pytest.mark.parametrize("w", [1e-200, 1e-9, 3.7, 2.0 ** 40, 1e100])
def test_deposits_over_the_weight_range(orc, w):
    """The window's limbs, split in doubles, against the exact integers."""
    import picgolf
    NX, NY, P = 32, 32, 3000
    rng = np.random.default_rng(3)
    x, y = rng.random(P), rng.random(P)
    x[:64] = (np.arange(64) + 1) / 64                     # cell edges and centres
    y[:4] = [1.0, 0.25 / NY, 1 - 2.0 ** -53, 0.5]
    v = [0.01 * rng.standard_normal(P) for _ in range(3)]
    cfg = picgolf.Config2D(NX=NX, NY=NY, P=P, w=w, dt=1e-3 / max(w, 1.0), B0=1.5)
    with picgolf.Context2D(cfg) as c:
        c.upload(x, y, *v)
        c.run(2)
        got = c.download()
    ref = orc.run2d(NX, NY, cfg.dt, cfg.B0, cfg.w, x, y, *v, 2, ns=2, textbook=0, nthreads=8)
    for g, r in zip(got, ref[:7]):
        assert same(g, r)
