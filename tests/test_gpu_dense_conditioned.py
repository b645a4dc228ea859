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
