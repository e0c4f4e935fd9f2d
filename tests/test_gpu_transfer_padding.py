"""What an upload writes on the device, read as it lies there: every element at its place and the padding of the last group
(of an ensemble case: up to three whole groups more) holding element K - 1, also over other data."""
import numpy as np
import pytest

from hopefoam_amd import Context

pytestmark = pytest.mark.gpu


def _expected(a, groups):
    """[var][K][Np] in groups of 16 elements, the last element repeated"""
    nvar, K, Np = a.shape
    e = np.minimum(np.arange(16 * groups), K - 1)
    return a[:, e].reshape(nvar, groups, 16, Np).transpose(1, 0, 3, 2)


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 3), (4, 2), (5, 3), (73, 29)])   # K = 2, 18, 16, 30, 4234
def test_field(N, nx, ny):
    with Context(0) as ctx:
        m = ctx.mesh_structured(N, nx, ny, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
        rng = np.random.default_rng(N)
        for nvar in (1, 3, 4):
            f = m.field(nvar)
            for _ in range(2):
                a = rng.standard_normal((nvar, m.K, m.Np))
                f.upload(a if nvar > 1 else a[0])
                np.testing.assert_array_equal(f.raw(), _expected(a, -(-m.K // 16)))


def test_ensemble():
    sizes = [(1, 3, 3), (3, 4, 4), (5, 5, 5), (8, 3, 9), (4, 8, 4)]   # K = 18, 32, 50, 54, 64 of 64
    cases = [dict(N=N, nx=nx, ny=ny, ax=1.0, ay=0.5, nu=1e-3, dt=1e-4) for N, nx, ny in sizes]
    with Context(0) as ctx:
        ens = ctx.ensemble(cases, autotune=False)
        rng = np.random.default_rng(3)
        for _ in range(2):
            for i, c in enumerate(ens.cases):
                a = rng.standard_normal((1, c["K"], c["Np"]))
                ens.set(i, a[0])
                np.testing.assert_array_equal(ens.raw(i), _expected(a, -(-c["K"] // 64) * 4)[:, 0])
        ens.close()
