"""Field transfers around the sizes at which they are cut differently: one chunk up to 512 KiB (down 384), several equal ones
beyond; upload, download and a kernel that reads the field come one after the other without a wait in between."""
import numpy as np
import pytest

from hopefoam_amd import Context

pytestmark = pytest.mark.gpu


# tiles of 16 elements: 3584 bytes at order 6, 5760 at order 8; 146 and 91 of them make a chunk up, 109 and 68 one down
@pytest.mark.parametrize("N,nx,ny,nvar", [(6, 18, 16, 4),    # 144 tiles: one chunk up, two down
                                          (6, 73, 4, 4),     # 148 tiles of which one in 37 is ragged: two chunks
                                          (6, 18, 12, 4),    # 108 tiles: one chunk
                                          (8, 182, 4, 1),    # 91 tiles: exactly one chunk up
                                          (8, 184, 4, 1),    # 92 tiles: two chunks
                                          (8, 137, 4, 1),    # 69 tiles: one up, two down, 35 and 34
                                          (8, 365, 4, 1),    # 183 tiles: three of 61
                                          (8, 16, 15, 3)])   # 90 tiles of three variables
def test_chunk_edges(N, nx, ny, nvar):
    with Context(0) as ctx:
        m = ctx.mesh_structured(N, nx, ny, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
        f, g = m.field(nvar), m.field(nvar)
        rng = np.random.default_rng(N * nx)
        for _ in range(3):
            a = rng.standard_normal((nvar, m.K, m.Np))
            f.upload(a if nvar > 1 else a[0])
            g.copy_from(f)
            f.upload(0.0 * a if nvar > 1 else 0.0 * a[0])
            np.testing.assert_array_equal(g.download().reshape(a.shape), a)
            assert not f.download().any()
