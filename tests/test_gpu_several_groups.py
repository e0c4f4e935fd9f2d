"""Stage kernels whose wavefronts walk several element groups: every order, precision and flux on a capped grid (two or
three groups a wavefront, the last one ragged) gives the bits of the grid with at most one group a wavefront, for the
right-hand side, the LSERK4 loop and the SSP-RK2 loop."""
import numpy as np
import pytest

from hopefoam_amd import (DGH_BC_ZERO_GRADIENT, DGH_EQ_ADVECT, DGH_EQ_EULER, DGH_FLUX_LF, DGH_FLUX_ROE, DGH_FLUX_UPWIND,
                          DGH_PREC_BF16X3, DGH_PREC_FP32, DGH_PREC_FP64, Context, RhsDesc)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("kind", ["lf", "roe", "upwind"])
def test_capped_grid_gives_the_same_bits(N, kind):
    nvar = 1 if kind == "upwind" else 4
    flux = {"lf": DGH_FLUX_LF, "roe": DGH_FLUX_ROE, "upwind": DGH_FLUX_UPWIND}[kind]
    with Context(0) as ctx:
        # 2178 elements: 136 groups and two elements, on 8 blocks of 4 or 8 wavefronts
        gm = ctx.mesh_structured(N, 33, 33, 0.0, 1.0, 0.0, 1.0, periodic=(False, False), bc_tag=DGH_BC_ZERO_GRADIENT)
        rng = np.random.default_rng(N)
        q = 0.05 * rng.standard_normal((nvar, gm.K, gm.Np)) + np.array([1.0, 0.4, -0.2, 2.5])[:nvar, None, None]
        q0, f = gm.field(nvar, q if nvar == 4 else q[0]), gm.field(nvar)
        for prec in (DGH_PREC_FP64, DGH_PREC_FP32, DGH_PREC_BF16X3):
            d = RhsDesc(DGH_EQ_ADVECT if nvar == 1 else DGH_EQ_EULER, flux, prec, 0, 0.7, -0.4, 1.4)
            got = []
            for cap in (0, 8):
                ctx.set_launch_cap(cap)
                gm.rhs(d, q0, f)
                out = [f.download()]
                for run in (gm.lserk4_run, gm.ssprk2_run):
                    f.copy_from(q0)
                    run(d, f, 2, 1e-5)
                    out.append(f.download())
                got.append(out)
            for one, several in zip(*got):
                assert np.isfinite(one).all()
                np.testing.assert_array_equal(one, several)
