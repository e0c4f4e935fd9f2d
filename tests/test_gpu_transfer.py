"""Field transfers: every order and variable count over the edges of tiles, chunks and workers come back bit for bit, the
padding of the last element group holds element K - 1, and two contexts transfer at the same time."""
import threading

import numpy as np
import pytest

from hopefoam_amd import DGH_EQ_ADVECT, DGH_FLUX_UPWIND, DGH_PREC_FP64, Context, RhsDesc

pytestmark = pytest.mark.gpu


def _values(rng, shape):
    a = rng.standard_normal(shape)
    flat = a.reshape(-1)
    flat[:: max(1, flat.size // 7)] = [np.inf, -0.0, np.nan, 5e-324][flat.size % 4]   # moved as they are
    return a


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("nx,ny", [(1, 1), (4, 2), (3, 3), (17, 9)])   # K = 2, 16, 18, 306
def test_round_trip(N, nx, ny):
    rng = np.random.default_rng(N)
    with Context(0) as ctx:
        m = ctx.mesh_structured(N, nx, ny, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
        for nvar in (1, 2, 3, 4):
            f, g = m.field(nvar), m.field(nvar)
            a = _values(rng, (nvar, m.K, m.Np))
            f.upload(a)
            g.copy_from(f)
            np.testing.assert_array_equal(g.download().reshape(a.shape).view(np.uint64), a.view(np.uint64))


@pytest.mark.parametrize("K2", [(200, 163), (256, 256)])   # 7.3 MB: several chunks; 117 MB: every worker, its slots reused
def test_large_round_trip_and_threads(K2):
    def one(seed, out):
        rng = np.random.default_rng(seed)
        with Context(0) as ctx:
            m = ctx.mesh_structured(6 if K2[0] == 256 else 2, K2[0], K2[1], 0.0, 1.0, 0.0, 1.0)
            f = m.field(4)
            ok = True
            for _ in range(2):
                a = rng.standard_normal((4, m.K, m.Np))
                f.upload(a)
                ok = ok and np.array_equal(f.download(), a)
            out[seed] = ok
    out = {}
    threads = [threading.Thread(target=one, args=(s, out)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == {1: True, 2: True}


def test_padding_repeats_last_element():
    """A stage evolves the padding columns from what the upload left there; a wrong value there would show as a
    difference between an upload into a fresh field and one over other data."""
    with Context(0) as ctx:
        m = ctx.mesh_structured(3, 3, 3, 0.0, 1.0, 0.0, 1.0)
        d = RhsDesc(DGH_EQ_ADVECT, DGH_FLUX_UPWIND, DGH_PREC_FP64, 0, 1.0, 0.5, 0.0)
        a = np.random.default_rng(5).standard_normal((m.K, m.Np))
        f, g = m.field(1, a), m.field(1, np.full((m.K, m.Np), np.nan))
        g.upload(a)
        m.lserk4_run(d, f, 3, 1e-3)
        m.lserk4_run(d, g, 3, 1e-3)
        np.testing.assert_array_equal(f.download(), g.download())


def test_ensemble_round_trip():
    cases = [dict(N=N, nx=n, ny=n, ax=1.0, ay=0.5, nu=1e-3, dt=1e-4) for N, n in ((1, 3), (4, 5), (8, 9))]
    with Context(0) as ctx:
        ens = ctx.ensemble(cases, autotune=False)
        rng = np.random.default_rng(3)
        u = [rng.standard_normal((c["K"], c["Np"])) for c in ens.cases]
        for i, a in enumerate(u):
            ens.set(i, a)
        for i, a in enumerate(u):
            np.testing.assert_array_equal(ens.get(i), a)
        ens.close()
