"""Positivity scaling on meshes of more than 512 element groups, where four groups share a block: blocks in which none, one,
two, three and all four groups hold cells that fail, the last group of two cells; and on meshes of fewer, where one group
has a block: the oracle's scaling, and the same bits either way."""
import numpy as np
import pytest

from hopefoam_amd import dgh
from meshgen import split_quads
from oracle_lib import OracleMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", range(1, 9))
def test_blocks_of_four_groups(N):
    nx, ny = 457, 9   # 8226 cells: 514 groups and two cells
    vxy, vid = split_quads(nx, ny, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
    bct = np.full(np.asarray(vid).shape, 2, np.int32)
    om = OracleMesh(N, vxy, vid, bct)
    K, Np = om.K, om.Np
    rng = np.random.default_rng(N)
    q = np.stack([1.0 + 0.1 * rng.uniform(-1, 1, (K, Np)), 0.3 * rng.uniform(-1, 1, (K, Np)),
                  0.3 * rng.uniform(-1, 1, (K, Np)), 2.6 + 0.2 * rng.uniform(-1, 1, (K, Np))])
    group = np.arange(K) // 16
    bad = (group % 4 < group // 4 % 5) & (rng.random(K) < 0.4)   # none to all four groups of a block, some of their cells
    for v, size in ((0, 1.5), (1, 3.0), (3, 3.0)):               # densities and pressures below zero, now and then both
        pick = bad & (rng.random(K) < 0.5)
        q[v, pick] += size * rng.uniform(-1, 1, (int(pick.sum()), Np))
    want, sc = om.positivity(q)
    assert 100 < sc.sum() < K // 2
    with dgh.Context(0) as ctx:
        f = ctx.mesh(N, vxy, vid, bct).field(4, q)
        f.mesh.limit(f, M=1e30, positivity=True, flags=False)
        got = f.download()
        assert np.array_equal(np.any(got != q, axis=(0, 2)), sc)
        assert np.abs(got - want).max() <= 1e-13 * np.abs(q).max()   # as for the small meshes
        # the scaling of a cell depends on its own values alone: the same cells on a mesh of 511 groups and one cell
        small = ctx.mesh_structured(N, 4089, 1, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
        for part in (slice(0, small.K), slice(K - small.K, K)):
            g = small.field(4, q[:, part])
            small.limit(g, M=1e30, positivity=True, flags=False)
            np.testing.assert_array_equal(g.download(), got[:, part])
