"""The adjoint over long multipole lists, whose sums are FP32 over at most 512
multipoles: against the same cotangents taken 100 multipoles at a time and added
in FP64.  Both sums round 25 to 128 positive terms per wave in FP32, each by
2^-24 of the running sum, and the rounded halves cancel in part: 2.5e-7 of the
terms' magnitudes (4 units in the last place) bounds the difference, where one
running sum of 20000 differs by 7e-6."""
import numpy as np
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd import serving
from jax_cosmo_amd._native import default_context
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


def cotangents(sid, n, n_z, P):
    ctx = default_context()
    ell = np.geomspace(10.0, 5000.0, n)
    cl = ctx.angular_cl(PARAMS[:1], sid, ell, n_z, P)[0]
    cb = (np.random.default_rng(n).uniform(0.5, 1.5, (P, n)) / np.abs(cl)).astype(np.float32)
    parts = [ctx.angular_cl_vjp(PARAMS[:1], sid, ell[a:a + 100], n_z, np.ascontiguousarray(cb[None, :, a:a + 100]))[0]
             for a in range(0, n, 100)]
    return ell, cb, np.sum(parts, 0), np.abs(parts).sum(0)


@pytest.mark.parametrize("n", [511, 513, 1025, 5000, 20000])
def test_long_lists(n):
    ctx = default_context()
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(make_probes(2, 2)))
    ell, cb, ref, mag = cotangents(sid, n, 512, 10)
    for B in (1, 150):
        params = np.repeat(PARAMS[:1], B, 0)
        th = ctx.angular_cl_vjp(params, sid, ell, 512, np.broadcast_to(cb, (B,) + cb.shape).copy())
        assert (np.abs(th - ref) <= 2.5e-7 * mag).all()


def test_served_requests_of_uneven_lengths():
    # more live blocks than the chip holds, so only the bound splits a list;
    # against the same server's answers to the lists cut into requests of 100
    ctx = default_context()
    probes = make_probes(2, 2)
    lens = [4096, 1, 700, 513, 512, 3000] * 20
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))
    case = {n: cotangents(sid, n, 512, 10)[:2] for n in set(lens)}

    def serve(lists):
        prep = srv.prepare([dict(cosmo=PARAMS[0], tracers=[0, 1, 2, 3], ell=ell, n_z=512, cl_bar=cb)
                            for ell, cb in lists])
        srv.submit_prepared(prep)
        srv.wait(0)
        return np.array([th for _, th in prep.outs])

    with serving.Server(probes, max_batch=128, max_grad=128, max_ell=4096, slots=1, n_z=(512,)) as srv:
        got = serve([case[n] for n in lens])
        parts = {n: serve([(ell[a:a + 100], cb[:, a:a + 100]) for a in range(0, n, 100)])
                 for n, (ell, cb) in case.items()}
    for n, th in zip(lens, got):
        assert (np.abs(th - parts[n].sum(0)) <= 2.5e-7 * np.abs(parts[n]).sum(0)).all()
