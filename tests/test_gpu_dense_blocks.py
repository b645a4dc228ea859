"""The dense factorisation and triangular solves at the edges of their blocks
(16, 64 and 256 rows) against LAPACK.  Entries are O(1) and the matrices'
condition number is about 1e3, so both sides carry errors of a few 1e-16 N
times 1e3 at most: 1e-10 bounds them for N < 1000."""
import numpy as np
import pytest
import torch

from jax_cosmo_amd._native import default_context

pytestmark = pytest.mark.gpu


def spd(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, n + 4)) / np.sqrt(n + 4)
    return a @ a.T + 1e-2 * np.eye(n)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 191, 255, 256, 257, 301, 512, 577, 775])
def test_factor_and_solves(n):
    ctx = default_context()
    C = spd(n, n)
    ref = np.linalg.cholesky(C)
    L, logdet = ctx.dense_cholesky(C)
    np.testing.assert_allclose(L.cpu().numpy(), ref, rtol=0, atol=1e-10)
    assert logdet == pytest.approx(np.linalg.slogdet(C)[1], rel=1e-10, abs=1e-10)
    Lr = torch.as_tensor(ref, device="cuda")
    for nrhs in (1, 16, 67):
        R = np.random.default_rng(nrhs).normal(size=(nrhs, n))
        z = np.linalg.solve(ref, R.T).T
        y = np.linalg.solve(ref.T, R.T).T
        scale = max(1.0, np.abs(z).max(), np.abs(y).max())
        np.testing.assert_allclose(ctx.dense_solve(Lr, R, mode=0), z, rtol=0, atol=1e-10 * scale)
        np.testing.assert_allclose(ctx.dense_solve(Lr, R, mode=1), y, rtol=0, atol=1e-10 * scale)
        x = ctx.dense_solve(Lr, R, mode=2)
        np.testing.assert_allclose(x @ C, R, rtol=0, atol=1e-10 * max(1.0, np.abs(x).max()))


@pytest.mark.parametrize("n,at", [(65, 64), (80, 3), (200, 150)])
def test_not_positive_definite_is_reported(n, at):
    C = spd(n, 5)
    C[at, at] = -1.0
    with pytest.raises(ValueError):
        default_context().dense_cholesky(C)
