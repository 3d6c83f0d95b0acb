"""The magnetised 1D2V step around the edges of its one-launch form (32 particles
to a block, 512 cells and 16384 particles of all species at most; the general
chain beyond), bit for bit against the CPU restatement."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("species,N,P,bin", [
    (1, 8, 1, 1), (1, 16, 31, 3), (2, 64, 16, 2), (1, 128, 33, 5), (2, 256, 2049, 4), (2, 512, 4097, 6),
    (1, 512, 16384, 7), (2, 512, 8192, 12), (2, 64, 8193, 6), (1, 1024, 500, 6)])
def test_run_bitwise(orc, species, N, P, bin):
    import picgolf
    from picgolf import configs
    cfg = dataclasses.replace(configs.bernstein(species)[0], N=N, P=P, bin=bin)
    rng = np.random.default_rng(N + P)
    st = [[rng.random(P), rng.standard_normal(P) / 50, rng.standard_normal(P) / 50] for _ in range(species)]
    for x, _, _ in st:
        x[1::11] = np.round(x[1::11] * N) / N        # cell edges and centres
    runs = (5, 1, 26, 13)                            # ends at odd and even steps, on and off the graph's turns
    T = sum(runs)
    with picgolf.Context1D2V(cfg) as c:
        for s in range(species):
            c.upload(s, *st[s])
        c.run_raw(3)
        c.upload(0, *st[0])                          # restarts the run; the other species stays as it is
        now = [c.download(s) for s in range(species)]
        D = np.vstack([c.run_raw(n) for n in runs])
        Es = c.fields_raw()
        got = [c.download(s) for s in range(species)]
    if species == 2:
        ref = [[a.copy() for a in s] for s in st]
        xs, vxs, vys, _, _ = run(orc, cfg, ref, 3)
        assert same(now[1], [xs[1], vxs[1], vys[1]])
    assert same(now[0], st[0])
    xs, vxs, vys, Eo, Do = run(orc, cfg, [[np.array(a) for a in s] for s in now], T)
    assert same(D, Do[:D.shape[0]]) and D.shape[0] == T // bin
    assert same(Es, Eo)
    for s in range(species):
        assert same(got[s][0], xs[s]) and same(got[s][1], vxs[s]) and same(got[s][2], vys[s])


def run(orc, cfg, st, T):
    return orc.run_1d2v(cfg.N, 7, cfg.q, cfg.q_m, cfg.mass, cfg.w, cfg.n0, cfg.B0, cfg.dt, cfg.bin,
                        [s[0] for s in st], [s[1] for s in st], [s[2] for s in st], T, nthreads=16)


@pytest.mark.parametrize("path", ["graph", "persistent", "1d2v"])
def test_a_nan_particle_adds_no_charge(orc, path):
    import picgolf
    from picgolf import configs
    if path == "1d2v":
        cfg, st, _ = configs.bernstein(1)
        st = [np.array(a) for a in st[0]]
        st[2][3] = np.nan
        with picgolf.Context1D2V(cfg) as c:
            c.upload(0, *st)
            c.run_raw(5)
            E = c.fields_raw()
            x = c.download(0)[0]
        xs, _, _, Eo, _ = run(orc, cfg, [st], 5)
        xo = xs[0]
    else:
        cfg, x, v, _ = configs.quiet_two_stream()
        v = np.array(v)
        v[3] = np.nan
        with picgolf.Context(cfg) as c:
            c.set_run_path(path)
            c.upload(x, v)
            c.run(5)
            xg, _, E = c.download()
        xo, _, Eo, _, _ = orc.run(cfg.N, 7, 1, cfg.W, cfg.w, cfg.dt, x, v, 5, rtol=cfg.rtol,
                                  max_sweeps=cfg.max_sweeps, E=None, nthreads=8)
        x = xg
    assert np.isnan(x[3]) and np.isnan(xo[3])
    keep = np.arange(len(x)) != 3
    assert same(E, Eo) and same(np.asarray(x)[keep], np.asarray(xo)[keep])
