"""The Jacobian's one pass over all seven directions against seven directional
derivatives (the same kernels, another split of the sum over a: relative to the
largest entry of a direction, 1e-5), over one cosmology, several chunks of
cosmologies, one and ten tracers, and with and without slices."""
import numpy as np
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd import autograd as jag
from jax_cosmo_amd._native import default_context
from test_gpu_forward_table import PARAMS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,wl,nc,n_ell,n_z", [(1, 1, 0, 1, 62), (3, 5, 5, 65, 130), (149, 0, 1, 33, 62),
                                               (2, 1, 1, 40000, 62)])
def test_jacobian_against_directional_derivatives(B, wl, nc, n_ell, n_z):
    ctx = default_context()
    ell = np.geomspace(20.0, 2000.0, n_ell)
    probes = []
    if wl:
        probes.append(jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, z) for z in np.linspace(0.5, 1.2, wl)]))
    if nc:
        probes.append(jc.probes.NumberCounts([jc.redshift.gaussian_nz(z, 0.1) for z in np.linspace(0.4, 1.2, nc)],
                                             jc.bias.constant_linear_bias(1.5)))
    params = PARAMS[np.arange(B) % 3]
    jac = jag.angular_cl_jacobian(params, ell, probes, n_z=n_z)
    P = (wl + nc) * (wl + nc + 1) // 2
    assert jac.shape == (B, P, n_ell, 7) and jac.dtype == np.float32
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))
    for d in range(7):
        t = np.zeros((B, 7))
        t[:, d] = 1.0
        dot = ctx.angular_cl_jvp(params, t, sid, ell, n_z, P)[1]
        scale = np.abs(dot).max(axis=2, keepdims=True)
        assert (np.abs(jac[..., d] - dot) <= 1e-5 * scale).all()


def test_a_direction_at_a_time(monkeypatch):
    """More multipoles than seven rows of a launch hold: the same Jacobian by
    single directions."""
    ell = np.geomspace(20.0, 2000.0, 9)
    probes = [jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, 0.7)])]
    ref = jag.angular_cl_jacobian(PARAMS, ell, probes, n_z=62)
    monkeypatch.setattr(jag, "MAX_COLUMNS", 62)
    jac = jag.angular_cl_jacobian(PARAMS, ell, probes, n_z=62)
    assert jac.shape == ref.shape and jac.dtype == ref.dtype
    assert (np.abs(jac - ref) <= 1e-5 * np.abs(ref).max(axis=2, keepdims=True)).all()
