"""Every tile shape of the ensemble kernels at every order, whatever the autotuner would take: right-hand side, q and LSERK4
steps (eager, then replayed from a graph) against the oracle, with last groups of 2, 14, 16 and 8 elements and one to five
work items per XCD range.  The bars are those of the tests with the default shapes."""
import numpy as np
import pytest

from hopefoam_amd import dgh
from test_gpu_ensemble import BETA, TAU, initial, make_cases, oracle_mesh

pytestmark = pytest.mark.gpu

SHAPES = {1: (1, 2), 2: (1, 2, 4, 16), 3: (2, 4, 8, 16), 4: (2, 4, 8, 16), 5: (4, 8, 16), 6: (4, 8, 16), 7: (8, 16), 8: (8, 16)}


@pytest.mark.parametrize("N,P", [(N, P) for N, shapes in SHAPES.items() for P in shapes])
def test_shape(N, P):
    cases = make_cases([(N, nx, ny, 1.0, (0.9, -0.4), 0.004) for nx, ny in ((3, 3), (5, 3), (4, 6), (20, 13), (16, 31))])
    oms = [oracle_mesh(c) for c in cases]
    us = [initial(om, c, 60 + i) for i, (om, c) in enumerate(zip(oms, cases))]
    with dgh.Context(0) as ctx:
        ens = ctx.ensemble(cases, tau=TAU, beta=BETA, autotune=False)
        ens.set_split(N, P)
        assert ens.info()["split"][N] == P
        for i, u in enumerate(us):
            ens.set(i, u)
        ens.rhs()
        for i, c in enumerate(cases):
            want, q = oms[i].ldg_rhs(us[i], c["ax"], c["ay"], c["nu"], tau=TAU, beta=BETA, with_q=True)
            assert np.abs(ens.get(i, 1) - want).max() <= 1e-12 * np.abs(want).max()
            assert np.abs(ens.get(i, 2) - q).max() <= 1e-12 * np.abs(q).max()
        ens.run(2, graph=False)
        ens.run(1, graph=True)
        ens.run(1, graph=True)
        for i, c in enumerate(cases):
            want = oms[i].ldg_lserk4(us[i], 4, c["dt"], c["ax"], c["ay"], c["nu"], tau=TAU, beta=BETA)
            assert np.abs(ens.get(i) - want).max() <= 1e-11 * np.abs(want).max()
        ens.close()


def test_refused_shapes():
    with dgh.Context(0) as ctx:
        ens = ctx.ensemble(make_cases([(1, 3, 3, 1.0, (0.9, -0.4), 0.004), (8, 3, 3, 1.0, (0.9, -0.4), 0.004)]), autotune=False)
        before = ens.info()["split"].copy()
        for N, P in ((1, 16), (1, 4), (8, 1), (8, 3), (4, 16), (0, 1), (9, 8)):
            with pytest.raises(dgh.DghError):
                ens.set_split(N, P)
        np.testing.assert_array_equal(ens.info()["split"], before)
        ens.close()
