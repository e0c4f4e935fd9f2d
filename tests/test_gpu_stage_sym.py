"""The FP64 stage kernel on the mirror halves of the operators, at every order, on meshes whose last element group is
ragged, with every boundary type, both Euler fluxes and both advection fluxes, against the extended-precision oracle."""
import numpy as np
import pytest

from hopefoam_amd import (DGH_EQ_ADVECT, DGH_EQ_EULER, DGH_FLUX_AVERAGE, DGH_FLUX_LF, DGH_FLUX_ROE, DGH_FLUX_UPWIND,
                          DGH_PREC_FP64, Context, RhsDesc)
from hopefoam_amd.cases import rel_l2
from meshgen import split_quads
from oracle_lib import OracleMesh

pytestmark = pytest.mark.gpu


def _mesh(nx, ny):
    """open split-quad mesh: the left side fixedValue, the right zeroGradient, bottom and top reflective walls"""
    vxy, vid = split_quads(nx, ny, 0.0, 2.0, 0.0, 1.5, periodic=(False, False))
    v = np.asarray(vxy).reshape(-1, 3, 2)
    mid = 0.5 * (v + np.roll(v, -1, axis=1))
    tag = np.zeros((v.shape[0], 3), np.int32)
    tag[(mid[:, :, 1] == 0.0) | (mid[:, :, 1] == 1.5)] = 3
    tag[mid[:, :, 0] == 0.0] = 1
    tag[mid[:, :, 0] == 2.0] = 2
    return vxy, vid, tag


def _state(x, y):
    rho = 1.0 + 0.2 * np.sin(2 * x + y)
    u, v = 0.5 + 0.3 * np.cos(x - 2 * y), -0.2 + 0.3 * np.sin(x * y)
    p = 1.0 + 0.2 * np.cos(3 * x)
    return np.stack([rho, rho * u, rho * v, p / 0.4 + 0.5 * rho * (u * u + v * v)])


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("kind", ["lf", "roe", "upwind", "average"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (5, 5)])   # K = 2 and 50: one short group; three whole ones and two elements
def test_rhs_and_stage_against_oracle(N, kind, nx, ny):
    vxy, vid, tag = _mesh(nx, ny)
    om, xp = OracleMesh(N, vxy, vid, tag), OracleMesh(N, vxy, vid, tag, extended=True)
    x, y = om.nodes()
    q = _state(x, y)
    euler = kind in ("lf", "roe")
    q = q if euler else q[0]
    nvar = 4 if euler else 1
    rng = np.random.default_rng(N)
    bcq = np.zeros((nvar, om.K, 3, om.Nfp)) + np.array([1.1, 0.4, -0.1, 2.7])[:nvar, None, None, None] \
        + 0.05 * rng.random((nvar, om.K, 3, om.Nfp))
    if euler:
        flux = DGH_FLUX_LF if kind == "lf" else DGH_FLUX_ROE
        d = RhsDesc(DGH_EQ_EULER, flux, DGH_PREC_FP64, 0, 0.0, 0.0, 1.4)
        ref, own = (m.rhs_euler(q, 1.4, 1 if kind == "lf" else 0, bcq) for m in (xp, om))
    else:
        flux = DGH_FLUX_UPWIND if kind == "upwind" else DGH_FLUX_AVERAGE
        d = RhsDesc(DGH_EQ_ADVECT, flux, DGH_PREC_FP64, 0, 0.7, -0.4, 0.0)
        ref, own = (m.rhs_advect(q, 0.7, -0.4, bcq, kind == "average") for m in (xp, om))
    # the parity bar of one right-hand side, or twice what the reference algorithm itself rounds in FP64
    bar = max(1e-12, 2.0 * rel_l2(own, ref))
    dt = 1e-3
    with Context(0) as ctx:
        gm = ctx.mesh(N, vxy, vid, tag)
        gm.set_bc_values(bcq)
        fq, fr, fo = gm.field(nvar, q), gm.field(nvar), gm.field(nvar)
        gm.rhs(d, fq, fr)
        assert rel_l2(fr.download(), ref) <= bar
        res0 = 0.1 * q
        fr.upload(res0)
        gm.lserk4_stage(d, fq, fo, fr, 1, dt)
        a, b = -567301805773.0 / 1357537059087.0, 5161836677717.0 / 13612068292357.0
        res = a * res0 + dt * ref
        # the update adds the right-hand side's error times dt and a few roundings of the registers
        assert rel_l2(fr.download(), res) <= bar * dt * np.linalg.norm(ref) / np.linalg.norm(res) + 1e-15
        assert rel_l2(fo.download(), q + b * res) <= bar * dt * np.linalg.norm(ref) / np.linalg.norm(q) + 1e-15
