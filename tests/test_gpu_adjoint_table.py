"""The adjoint kernel of transfer-table calls (n_ell >= 64) at the edges of its
blocks: node groups that end early, single nodes, multipole chunks and slices
with a remainder, every tracer count's padding, against the closed-form
adjoint (which runs over (cosmology, ell) columns).  The closed form's EH98
derivative and the table's interpolated one differ by below 1e-4 of a term
(piecewise linear interpolation on the same nodes would give 8e-5), so the
bound is 1e-4 of the sum of the terms' magnitudes."""
import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context
from jax_cosmo_amd.autograd import AngularClFunction
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wl,nc", [(1, 0), (0, 2), (3, 1), (2, 3), (4, 4), (5, 5)])
@pytest.mark.parametrize("n_ell,n_z,B", [(64, 2, 1), (65, 62, 3), (97, 64, 2), (129, 126, 40), (201, 254, 3)])
def test_table_adjoint_edges(wl, nc, n_ell, n_z, B):
    ctx = default_context()
    probes = make_probes(wl, nc)
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))
    P = (wl + nc) * (wl + nc + 1) // 2
    params = PARAMS[np.arange(B) % 3]
    ell = np.geomspace(2.0, 6000.0, n_ell)
    cl = ctx.angular_cl(params, sid, ell, n_z, P)
    cbar = (np.random.default_rng(n_ell).normal(size=cl.shape) / cl).astype(np.float32)
    th = ctx.angular_cl_vjp(params, sid, ell, n_z, cbar)
    try:
        ctx.set_forward_options(transfer_table=0)
        ref = ctx.angular_cl_vjp(params[:3], sid, ell, n_z, cbar[:3])
        scale = np.empty_like(ref)
        for d in range(7):
            t = np.zeros((len(ref), 7))
            t[:, d] = 1.0
            dot = ctx.angular_cl_jvp(params[:3], t, sid, ell, n_z, P)[1]
            scale[:, d] = np.abs(cbar[:3].astype(np.float64) * dot).sum(axis=(1, 2))
    finally:
        ctx.set_forward_options(transfer_table=1)
    assert th.shape == (B, 7) and np.isfinite(th).all()
    assert (np.abs(th[:3] - ref) <= 1e-4 * scale).all()


def test_a_bad_cosmology_stays_alone():
    ctx = default_context()
    ell, probes = np.geomspace(10.0, 5000.0, 70), make_probes(2, 2)
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))

    def grad(p):
        th = torch.tensor(p[:, [0, 1, 2, 3, 4, 6, 7]], device="cuda", requires_grad=True)
        AngularClFunction.apply(th, torch.as_tensor(p[:, 5], device="cuda"), ell, sid, 256, 10).sum().backward()
        return th.grad.cpu().numpy()

    good = grad(PARAMS)
    p = PARAMS.copy()
    p[1, 4] = np.nan
    out = grad(p)
    assert np.isnan(out[1]).any()
    assert np.array_equal(out[[0, 2]], good[[0, 2]])
