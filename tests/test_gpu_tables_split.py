"""Table kernels of a few cosmologies, whose directions are apart, and of many,
whose directions are together: the same gradients and directional derivatives
row by row, at the numbers of cosmologies where the shapes change on 256 compute
units, with and without transfer tables, under every model.  The FP64 tables agree
to rounding; the float32 sums over a are split differently, so 1e-5 of the
largest component bounds the pair."""
import numpy as np
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_ell,n_z", [(9, 62), (70, 130)])
@pytest.mark.parametrize("model", [(0, 0, None), (1, 0, None), (0, 1, None), (0, 0, 0.55)])
def test_rows_of_small_and_large_batches(n_ell, n_z, model):
    ctx = default_context()
    ell = np.geomspace(20.0, 2000.0, n_ell)
    probes = make_probes(2, 2)
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))
    rng = np.random.default_rng(n_ell)
    n = 300
    params = PARAMS[np.arange(n) % 3]
    saved = ctx.models()
    try:
        ctx.set_models(model[0], model[1])
        ctx.set_growth(model[2])
        cl = ctx.angular_cl(params[:3], sid, ell, n_z, 10)
        u = (rng.uniform(0.5, 1.5, (1, 10, n_ell)) / np.abs(cl).max(axis=(0, 2), keepdims=True)).astype(np.float32)
        v = rng.normal(size=(1, 7))

        def both(b):
            th = ctx.angular_cl_vjp(params[:b], sid, ell, n_z, np.repeat(u, b, axis=0))
            dot = ctx.angular_cl_jvp(params[:b], np.repeat(v, b, axis=0), sid, ell, n_z, 10)[1]
            return th, dot

        th, dot = both(n)
        assert np.isfinite(th).all()
        for b in (1, 36, 37, 256, 257):
            t, d = both(b)
            assert (np.abs(t - th[:b]) <= 1e-5 * np.abs(th[:b]).max(axis=1, keepdims=True)).all()
            assert (np.abs(d - dot[:b]) <= 1e-5 * np.abs(dot[:b]).max(axis=2, keepdims=True)).all()
            lhs = (d[0].astype(np.float64) * u[0]).sum()
            assert abs(lhs - t[0] @ v[0]) <= 1e-3 * np.abs(t[0] * v[0]).sum()
    finally:
        ctx.set_models(saved[0], saved[1])
        ctx.set_growth(saved[2])
