"""Dense solves on device arrays take no memory of the context: solves on
several streams side by side, a captured solve replayed between eager ones, and
the library's own in-place form, against LAPACK to 1e-10 as in the tests of the
blocks' edges."""
import ctypes

import numpy as np
import pytest
import torch

from jax_cosmo_amd._native import JC_DEVICE_PTRS, check, default_context
from test_gpu_dense_blocks import spd

pytestmark = pytest.mark.gpu


def factor(n, seed):
    L = np.linalg.cholesky(spd(n, seed))
    return L, torch.as_tensor(L, device="cuda")


def solution(L, R, mode):
    y = np.linalg.solve(L, R.T) if mode != 1 else R.T
    return (np.linalg.solve(L.T, y) if mode else y).T


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n", [64, 65, 127, 128, 200, 577])
def test_in_place_form(n, mode):
    ctx = default_context()
    L, Lt = factor(n, n)
    for nrhs in (1, 16, 17, 67):
        R = np.random.default_rng(nrhs).normal(size=(nrhs, n))
        want = solution(L, R, mode)
        for inplace in (True, False):
            Rt = torch.as_tensor(R, device="cuda")
            X = Rt if inplace else torch.full_like(Rt, float("nan"))
            torch.cuda.synchronize()
            check(ctx.lib.jc_dense_solve(ctx.handle, ctypes.c_void_p(Lt.data_ptr()), n, ctypes.c_void_p(Rt.data_ptr()),
                                         nrhs, mode, ctypes.c_void_p(X.data_ptr()), JC_DEVICE_PTRS))
            check(ctx.lib.jc_synchronize(ctx.handle))
            np.testing.assert_allclose(X.cpu().numpy(), want, rtol=0, atol=1e-10 * max(1.0, np.abs(want).max()))


def test_too_small_a_workspace_is_refused():
    ctx = default_context()
    n = ctypes.c_int64()
    check(ctx.lib.jc_dense_solve_workspace(100, 3, 2, ctypes.byref(n)))
    _, Lt = factor(100, 1)
    X = torch.zeros((3, 100), dtype=torch.float64, device="cuda")
    work = torch.empty(n.value, dtype=torch.float64, device="cuda")
    args = [ctypes.c_void_p(t.data_ptr()) for t in (Lt, X, work)]
    with pytest.raises(ValueError):
        check(ctx.lib.jc_dense_solve_work(ctx.handle, args[0], 100, args[1], 3, 2, args[1], args[2], n.value - 1))


def test_two_streams_side_by_side():
    ctx = default_context()
    n, nrhs = 1500, 200
    rng = np.random.default_rng(0)
    cases = []
    for k in range(4):
        L, Lt = factor(n, k)
        R = rng.normal(size=(nrhs, n))
        cases.append((Lt, torch.as_tensor(R, device="cuda"), solution(L, R, 2)))
    streams = [torch.cuda.Stream() for _ in cases]
    torch.cuda.synchronize()
    for (Lt, R, _), s in zip(cases, streams):
        with torch.cuda.stream(s):
            ctx.dense_solve(Lt, R, mode=2)
    torch.cuda.synchronize()
    for _, x, want in cases:
        np.testing.assert_allclose(x.cpu().numpy(), want, rtol=0, atol=1e-10 * np.abs(want).max())


@pytest.mark.parametrize("n", [40, 300])
def test_captured_solve(n):
    ctx = default_context()
    L, Lt = factor(n, 2)
    _, L2 = factor(n, 3)
    rng = np.random.default_rng(1)
    X = torch.zeros((5, n), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.dense_solve(Lt, X, mode=2)
    for _ in range(4):
        R = rng.normal(size=(5, n))
        X.copy_(torch.as_tensor(R))
        ctx.dense_solve(L2, torch.as_tensor(R, device="cuda"), mode=2)  # the program's own work in between
        graph.replay()
        torch.cuda.synchronize()
        want = solution(L, R, 2)
        np.testing.assert_allclose(X.cpu().numpy(), want, rtol=0, atol=1e-10 * max(1.0, np.abs(want).max()))
