"""Triangular solves and likelihoods of dense covariances around the 512-row
blocks of the solves against LAPACK: the tolerance of test_gpu_dense_blocks
(errors of a few 1e-16 N times a condition number of 1e3), 1e-10 for N < 1600."""
import numpy as np
import pytest
import torch

from jax_cosmo_amd._native import default_context
from test_gpu_dense_blocks import spd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [257, 511, 513, 768, 1023, 1024, 1025, 1300, 1537])
def test_solves_around_blocks(n):
    ctx = default_context()
    C = spd(n, n)
    ref = np.linalg.cholesky(C)
    Lr = torch.as_tensor(ref, device="cuda")
    rng = np.random.default_rng(n)
    for nrhs in (1, 64, 130):
        R = rng.normal(size=(nrhs, n))
        z = np.linalg.solve(ref, R.T).T
        y = np.linalg.solve(ref.T, R.T).T
        scale = max(1.0, np.abs(z).max(), np.abs(y).max())
        np.testing.assert_allclose(ctx.dense_solve(Lr, R, mode=0), z, rtol=0, atol=1e-10 * scale)
        np.testing.assert_allclose(ctx.dense_solve(Lr, R, mode=1), y, rtol=0, atol=1e-10 * scale)
        mu = R.astype(np.float32)
        data = rng.normal(size=n)
        d = np.linalg.solve(ref, (data - mu.astype(np.float64)).T)
        ll, dmu = ctx.gaussian_loglike_dense(mu, data, Lr, want_dmu=True)
        np.testing.assert_allclose(ll, -0.5 * (d ** 2).sum(0), rtol=1e-10)
        x = np.linalg.solve(ref.T, d).T
        np.testing.assert_allclose(dmu, x, rtol=0, atol=2.0 ** -23 * np.abs(x).max())


@pytest.mark.parametrize("n", [1, 2, 33, 63, 64, 65])
@pytest.mark.parametrize("nrhs", [1, 4, 5, 130])
def test_solves_of_few_rows(n, nrhs):
    ctx = default_context()
    ref = np.linalg.cholesky(spd(n, n))
    Lr = torch.as_tensor(ref, device="cuda")
    R = np.random.default_rng(n).normal(size=(nrhs, n))
    z = np.linalg.solve(ref, R.T)
    for mode, want in ((0, z.T), (1, np.linalg.solve(ref.T, R.T).T), (2, np.linalg.solve(ref.T, z).T)):
        atol = 1e-10 * max(1.0, np.abs(want).max())
        np.testing.assert_allclose(ctx.dense_solve(Lr, R, mode=mode), want, rtol=0, atol=atol)
        Rd = torch.as_tensor(R, device="cuda")  # solved in place
        np.testing.assert_allclose(ctx.dense_solve(Lr, Rd, mode=mode).cpu().numpy(), want, rtol=0, atol=atol)
