"""The forward Limber kernel of transfer-table calls (n_ell >= 64) at the
edges of its tiles: column groups of 64 that straddle two cosmologies or end
early, a-ranges that leave single nodes and empty waves, and every padded
tracer width, against the closed-form kernel.  Both are float32 with float64
tables; the transfer table alone may differ from the closed form by 2e-6, so
2e-5 bounds the pair."""
import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context

pytestmark = pytest.mark.gpu

PARAMS = np.array([[0.2589, 0.0486, 0.6774, 0.9667, 0.8159, 0.0, -1.0, 0.0],
                   [0.31, 0.045, 0.72, 0.95, 0.78, 0.0, -0.9, 0.2],
                   [0.22, 0.055, 0.63, 0.98, 0.87, 0.02, -1.1, -0.3]])


def make_probes(wl, nc):
    z0 = (0.5, 0.75, 1.0, 1.25, 1.5)
    out = []
    if wl:
        out.append(jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, z) for z in z0[:wl]]))
    if nc:
        out.append(jc.probes.NumberCounts([jc.redshift.gaussian_nz(0.3 * (i + 1), 0.1) for i in range(nc)],
                                          jc.bias.constant_linear_bias(1.5)))
    return out


def both(params, ell, probes, n_z):
    ctx = default_context()
    try:
        tab = jc.cl.angular_cl_batch(params, ell, probes, n_z=n_z)
        ctx.set_forward_options(transfer_table=0)
        ref = jc.cl.angular_cl_batch(params, ell, probes, n_z=n_z)
    finally:
        ctx.set_forward_options(transfer_table=1)
    return tab, ref


@pytest.mark.parametrize("wl,nc", [(1, 0), (0, 2), (3, 1), (2, 3), (4, 4), (5, 5)])
@pytest.mark.parametrize("n_ell,n_z,B", [(64, 2, 1), (65, 30, 3), (97, 62, 3), (128, 256, 2), (201, 66, 3)])
def test_table_kernel_edges(wl, nc, n_ell, n_z, B):
    tab, ref = both(PARAMS[:B], np.geomspace(2.0, 6000.0, n_ell), make_probes(wl, nc), n_z)
    assert tab.shape == ref.shape and np.isfinite(tab).all()
    np.testing.assert_allclose(tab, ref, rtol=2e-5, atol=0)


def test_a_bad_cosmology_stays_alone():
    # columns of a NaN cosmology share their group with both neighbours'
    ell, probes = np.geomspace(10.0, 5000.0, 70), make_probes(2, 2)
    p = torch.as_tensor(PARAMS, device="cuda")
    good = jc.cl.angular_cl_batch(p, ell, probes, n_z=256).cpu().numpy()
    p[1, 4] = float("nan")
    out = jc.cl.angular_cl_batch(p, ell, probes, n_z=256).cpu().numpy()
    assert np.isnan(out[1]).all()
    assert np.array_equal(out[[0, 2]], good[[0, 2]])
