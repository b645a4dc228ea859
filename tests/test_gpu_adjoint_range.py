"""The adjoint is linear in its cotangents over most of float32's exponents:
cotangents times a power of two give the gradient times that power.  Products of
a cotangent, two kernels and the weight are normal numbers from 2^-80 (lensing) to
2^100 (counts), so only denormal remainders of the smallest multipoles'
terms may differ: 1e-6."""
import numpy as np
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wl,nc", [(1, 0), (0, 1), (5, 5)])
@pytest.mark.parametrize("lo,hi", [(2.0, 1e4), (100.0, 3000.0)])
def test_scaled_cotangents(wl, nc, lo, hi):
    ctx = default_context()
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(make_probes(wl, nc)))
    T, ell = wl + nc, np.geomspace(lo, hi, 100)
    cb = np.random.default_rng(T).normal(size=(1, T * (T + 1) // 2, 100)).astype(np.float32)
    th = ctx.angular_cl_vjp(PARAMS[:1], sid, ell, 512, cb)
    for k in (-80, 80, 100):
        got = ctx.angular_cl_vjp(PARAMS[:1], sid, ell, 512, np.ldexp(cb, k))
        np.testing.assert_allclose(np.ldexp(got, -k), th, rtol=1e-6)
