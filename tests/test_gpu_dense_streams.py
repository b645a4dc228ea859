"""Dense solves on device arrays take no memory of the context: solves on
several streams side by side, a captured solve replayed between eager ones,
calls that wait for their result beside an unfinished one on another stream, and
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


def test_factorisation_beside_a_pending_likelihood():
    # the likelihoods of many device means are queued on one stream; the call
    # returns, and covariances are factored on another meanwhile
    ctx = default_context()
    n, B = 1200, 512
    rng = np.random.default_rng(5)
    L, Lt = factor(n, 7)
    mu, data = rng.normal(size=(B, n)).astype(np.float32), rng.normal(size=n)
    want = -0.5 * (solution(L, data - mu.astype(np.float64), 0) ** 2).sum(1)
    mut, dt = torch.as_tensor(mu, device="cuda"), torch.as_tensor(data, device="cuda")
    C = spd(700, 8)
    ref = np.linalg.cholesky(C)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(5):
        ll = torch.zeros(B, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        with ctx._lock:
            ctx.set_stream(a.cuda_stream)
            check(ctx.lib.jc_gaussian_loglike_dense(
                ctx.handle, ctypes.c_void_p(mut.data_ptr()), B, n, ctypes.c_void_p(dt.data_ptr()),
                ctypes.c_void_p(Lt.data_ptr()), 0.0, ctypes.c_void_p(ll.data_ptr()), None, JC_DEVICE_PTRS))
            ctx.reset_stream()
        with torch.cuda.stream(b):
            F, _ = ctx.dense_cholesky(C)
        torch.cuda.synchronize()
        np.testing.assert_allclose(ll.cpu().numpy(), want, rtol=1e-10)
        np.testing.assert_allclose(F.cpu().numpy(), ref, rtol=0, atol=1e-10)


def test_host_means_beside_a_pending_gradient():
    # log-likelihoods and gradients of a batch under a block-diagonal covariance
    # are queued on one stream; host means take the dense algebra on another
    import jax_cosmo_amd as jc
    from test_gpu_forward_table import PARAMS, make_probes

    ctx = default_context()
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    probes, ell, n_z, B = make_probes(2, 2), np.geomspace(20.0, 2000.0, 70), 256, 256
    sid, P = ctx.tracer_set(jc.cl.tracer_entries(probes)), 10
    params = PARAMS[np.arange(B) % 3]
    cl = ctx.angular_cl(PARAMS[:1], sid, ell, n_z, P)[0].astype(np.float64)
    prec = np.ascontiguousarray(np.eye(P)[..., None] / (0.1 * np.abs(cl[None])) ** 2)
    data = 1.05 * cl
    ll0, g0 = ctx.gaussian_loglike_grad(params, sid, ell, n_z, data, prec)
    n = 900
    L, Lt = factor(n, 4)
    mu, d = np.random.default_rng(2).normal(size=(64, n)).astype(np.float32), np.ones(n)
    want = -0.5 * (solution(L, d - mu.astype(np.float64), 0) ** 2).sum(1)
    dev = [torch.as_tensor(x, device="cuda") for x in (params, ell, data, prec)]
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(5):
        ll = torch.zeros(B, dtype=torch.float64, device="cuda")
        g = torch.zeros((B, 7), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ctx.gaussian_loglike_grad_dev(dev[0].data_ptr(), B, sid, dev[1].data_ptr(), len(ell), n_z, dev[2].data_ptr(),
                                      dev[3].data_ptr(), 0.0, ll.data_ptr(), g.data_ptr(), stream=a.cuda_stream)
        with torch.cuda.stream(b):
            got, dmu = ctx.gaussian_loglike_dense(mu, d, Lt, want_dmu=True)
        torch.cuda.synchronize()
        ctx.reset_stream()
        np.testing.assert_allclose(got, want, rtol=1e-10)
        np.testing.assert_array_equal(ll.cpu().numpy(), ll0)  # the same sums in the same order
        np.testing.assert_array_equal(g.cpu().numpy(), g0)
