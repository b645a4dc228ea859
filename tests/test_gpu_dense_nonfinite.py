"""Right-hand sides with an element that is not finite: a triangular solve
leaves the unknowns that do not depend on it as they are.  Against the same
solve without it, whose values take part in the same sums: 1e-10 as in the tests
of the blocks' edges."""
import numpy as np
import pytest

from jax_cosmo_amd._native import default_context
from test_gpu_dense_blocks import spd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [50, 300, 1100])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_only_the_dependent_unknowns_are_lost(n, bad):
    ctx = default_context()
    L, _ = ctx.dense_cholesky(spd(n, n))
    at = [0, 5, 16, n // 2, n - 2, n - 1]
    clean = np.random.default_rng(n).normal(size=(len(at) + 1, n))
    R = clean.copy()
    R[np.arange(len(at)), at] = bad
    for mode in (0, 1):
        ref, x = ctx.dense_solve(L, clean, mode=mode), ctx.dense_solve(L, R, mode=mode)
        for b, k in enumerate(at):
            keep = slice(0, k) if mode == 0 else slice(k + 1, n)
            np.testing.assert_allclose(x[b, keep], ref[b, keep], rtol=0, atol=1e-10 * np.abs(ref).max())
            assert not np.isfinite(x[b, k])
        assert np.array_equal(x[-1], ref[-1])
