"""The FP64 Euler fluxes over the whole range of their square roots: gas at rest whose pressures reach down to the smallest
numbers and to zero.  The density's right-hand side is then the sound speed times the jumps of the density, far from zero
beside what it is formed from, so a root that is wrong for small arguments shows in full."""
import numpy as np
import pytest

from hopefoam_amd import DGH_EQ_EULER, DGH_FLUX_LF, DGH_FLUX_ROE, DGH_PREC_FP64, Context, RhsDesc
from hopefoam_amd.cases import rel_l2
from meshgen import split_quads
from oracle_lib import OracleMesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 4, 8])
@pytest.mark.parametrize("kind,scale", [(k, s) for k in ("lf", "roe") for s in (1e-280, 1e-299, 1e-301, 1e-304, 1e-307)] +
                         [("lf", 1e-310), ("lf", 0.0)])   # (the Roe average divides by the square of the sound speed)
def test_sound_speed_of_small_pressures(N, kind, scale):
    vxy, vid = split_quads(5, 5, 0.0, 2.0, 0.0, 1.5)
    om = OracleMesh(N, vxy, vid, extended=True)
    rng = np.random.default_rng(N)
    q = np.zeros((4, om.K, om.Np))
    q[0] = rng.uniform(0.5, 2.0, (om.K, 1))   # constant in each element: its volume terms are zero
    q[3] = scale * rng.uniform(1.0, 3.0, (om.K, 1))
    ref = om.rhs_euler(q, 1.4, 1 if kind == "lf" else 0)[0]
    d = RhsDesc(DGH_EQ_EULER, DGH_FLUX_LF if kind == "lf" else DGH_FLUX_ROE, DGH_PREC_FP64, 0, 0.0, 0.0, 1.4)
    with Context(0) as ctx:
        gm = ctx.mesh(N, vxy, vid)
        fq, fr = gm.field(4, q), gm.field(4)
        gm.rhs(d, fq, fr)
        got = fr.download()[0]
    if scale == 0.0:
        assert (ref == 0.0).all() and (got == 0.0).all()
        return
    # the parity bar of one right-hand side; beneath the normal numbers the pressure itself holds fewer digits
    assert rel_l2(got / np.sqrt(scale), ref / np.sqrt(scale)) <= max(1e-12, 8 * 2.0 ** -1074 / scale)
