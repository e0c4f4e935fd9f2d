"""The time loops keep no residual they do not read and form q^n - q^(1) inside the second SSP-RK2 stage; the stage calls,
which return the residual, are the general path: the same bits, at every order and precision, on ragged last groups."""
import numpy as np
import pytest

from hopefoam_amd import (DGH_EQ_ADVECT, DGH_EQ_EULER, DGH_FLUX_LF, DGH_FLUX_ROE, DGH_FLUX_UPWIND, DGH_PREC_BF16X3,
                          DGH_PREC_FP32, DGH_PREC_FP64, Context, RhsDesc)
from meshgen import split_quads

pytestmark = pytest.mark.gpu


def _state(rng, nvar, K, Np):
    q = 0.05 * rng.standard_normal((nvar, K, Np)) + np.array([1.0, 0.4, -0.2, 2.5])[:nvar, None, None]
    return q if nvar == 4 else q[0]


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("prec", [DGH_PREC_FP64, DGH_PREC_FP32, DGH_PREC_BF16X3])
@pytest.mark.parametrize("kind,nx,ny", [("lf", 5, 5), ("roe", 3, 7), ("upwind", 9, 1)])   # K = 50, 42, 18
def test_loops_equal_stages(N, prec, kind, nx, ny):
    vxy, vid = split_quads(nx, ny, 0.0, 1.0, 0.0, 1.0, periodic=(False, False))
    bct = np.full(np.asarray(vid).shape, 2, np.int32)
    K, Np, dt = 2 * nx * ny, (N + 1) * (N + 2) // 2, 1e-4
    nvar = 1 if kind == "upwind" else 4
    flux = {"lf": DGH_FLUX_LF, "roe": DGH_FLUX_ROE, "upwind": DGH_FLUX_UPWIND}[kind]
    d = RhsDesc(DGH_EQ_ADVECT if nvar == 1 else DGH_EQ_EULER, flux, prec, 0, 0.7, -0.4, 1.4)
    rng = np.random.default_rng(17 * N + K)
    q0 = _state(rng, nvar, K, Np)
    with Context(0) as ctx:
        gm = ctx.mesh(N, vxy, vid, bct)
        run, cur, nxt, res, rhs = (gm.field(nvar) for _ in range(5))
        run.upload(q0)
        cur.upload(q0)
        res.upload(np.zeros_like(q0))
        gm.lserk4_run(d, run, 2, dt)
        for s in 2 * list(range(5)):
            gm.lserk4_stage(d, cur, nxt, res, s, dt)
            cur, nxt = nxt, cur
        np.testing.assert_array_equal(run.download(), cur.download())
        gm.ssprk2_run(d, run, 2, dt)
        for _ in range(2):
            gm.ssprk2_stage(d, cur, nxt, res, 0, dt)
            before, first = cur.download(), nxt.download()
            gm.ssprk2_stage(d, nxt, cur, res, 1, dt)
            gm.rhs(d, nxt, rhs)
            # the residual the stage returns: one rounding of the difference, the product and the sum each
            L = rhs.download()
            tol = 4 * 2.0 ** -53 * (np.abs(before) + np.abs(first) + np.abs(dt * L))
            assert (np.abs(res.download() - ((before - first) + dt * L)) <= tol).all()
        np.testing.assert_array_equal(run.download(), cur.download())
