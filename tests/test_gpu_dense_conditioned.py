"""The dense factorisation of correlated covariances (condition 1e9 to 1e13, as
of Gaussian processes with a small nugget).  The backward error of a Cholesky
factorisation does not depend on the condition number: |L L^T - C| is at most
(N + 1) 2^-53 |L| |L|^T, and (|L| |L|^T)_ij <= max C_ii; the check itself adds
the rounding of its own product, of the same size."""
import numpy as np
import pytest

from jax_cosmo_amd._native import default_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("length,nugget", [(5, 1e-8), (20, 1e-8), (5, 1e-11), (20, 1e-11), (50, 1e-12)])
@pytest.mark.parametrize("n", [128, 577, 1024])
def test_residual_does_not_grow_with_condition(n, length, nugget):
    x = np.arange(float(n))
    C = np.exp(-0.5 * ((x[:, None] - x) / length) ** 2) + nugget * np.eye(n)
    np.linalg.cholesky(C)  # positive definite in 64 bits
    L, _ = default_context().dense_cholesky(C)
    L = L.cpu().numpy()
    assert np.array_equal(L, np.tril(L))
    assert np.abs(L @ L.T - C).max() <= 2 * (n + 1) * 2.0**-53 * C.max()


@pytest.mark.parametrize("at", [(5,), (0, 63, 64, 199), tuple(range(60, 130))])
def test_infinite_variance_takes_a_datum_out(at):
    # against the algebra of the other data alone; condition 1e3 as in the
    # tests of the blocks' edges, and so their 1e-10
    n = 200
    rng = np.random.default_rng(3)
    a = rng.normal(size=(n, n + 4)) / np.sqrt(n + 4)
    C = a @ a.T + 1e-2 * np.eye(n)
    keep = np.setdiff1d(np.arange(n), at)
    sub = C[np.ix_(keep, keep)]
    C[at, at] = np.inf
    ctx = default_context()
    L, logdet = ctx.dense_cholesky(C)
    assert logdet == np.inf
    Lh = L.cpu().numpy()
    np.testing.assert_allclose(Lh[np.ix_(keep, keep)], np.linalg.cholesky(sub), rtol=0, atol=1e-10)
    assert np.isinf(Lh[at, at]).all()
    mu, data = rng.normal(size=(3, n)).astype(np.float32), rng.normal(size=n)
    r = (data - mu.astype(np.float64))[:, keep]
    x = np.linalg.solve(sub, r.T).T
    ll, dmu = ctx.gaussian_loglike_dense(mu, data, L, want_dmu=True)
    np.testing.assert_allclose(ll, -0.5 * (r * x).sum(1), rtol=1e-10)
    np.testing.assert_allclose(dmu[:, keep], x, rtol=1e-6, atol=1e-6 * np.abs(x).max())
    assert (dmu[:, at] == 0).all()
    sol = ctx.dense_solve(L, data[None], mode=2)[0]
    np.testing.assert_allclose(sol[keep], np.linalg.solve(sub, data[keep]), rtol=0, atol=1e-10 * np.abs(sol).max())
    assert (sol[list(at)] == 0).all()
