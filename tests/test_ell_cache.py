"""The kept device copies of host multipole lists: threads that evict at once,
memory of an evicted list that another stream may still read, and captures."""
import threading
import time

import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd import angular_cl as acl
from jax_cosmo_amd import autograd as jag


def test_two_threads_evict(monkeypatch):
    class Slow(dict):  # widens the gap between choosing the entry and dropping it
        def pop(self, *a):
            time.sleep(0.05)
            return dict.pop(self, *a)

    cpu = torch.device("cpu")
    monkeypatch.setattr(acl, "_ELL_CACHE", Slow())
    for k in range(acl._ELL_CACHE_MAX):
        acl._device_ell(np.array([float(k)]), cpu)
    errors, gate = [], threading.Barrier(4)

    def work(k):
        try:
            gate.wait()
            for j in range(3):
                ell = np.array([1000.0 + 10 * k + j, 5.0])
                assert torch.equal(acl._device_ell(ell, cpu), torch.as_tensor(ell))
        except BaseException as e:  # noqa: B902
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors
    assert len(acl._ELL_CACHE) == acl._ELL_CACHE_MAX


@pytest.mark.gpu
def test_evicted_list_waits_for_the_other_stream():
    dev = torch.device("cuda", 0)
    n = 77
    acl._device_ell(np.full(n, 3.0), dev)  # belongs to the default stream
    side = torch.cuda.Stream()
    x = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        ptr = acl._device_ell(np.full(n, 3.0), dev).data_ptr()  # as a call on `side` takes it
        for _ in range(60):
            x = (x @ x).clamp_(-1, 1)
    for k in range(acl._ELL_CACHE_MAX):
        acl._device_ell(np.array([7.0 + k]), dev)
    assert not side.query(), "the side stream was meant to be busy still"
    others = [torch.empty(n, dtype=torch.float64, device=dev) for _ in range(300)]
    assert ptr not in {t.data_ptr() for t in others}
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_gradient_calls_are_not_captured():
    ctx = jc._native.default_context()
    sid = ctx.tracer_set(jc.cl.tracer_entries([jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, 0.8)])]))
    theta = torch.tensor([[0.25, 0.05, 0.7, 0.96, 0.8, -0.95, 0.1]], dtype=torch.float64, device="cuda")
    ell = np.geomspace(20.0, 800.0, 70)
    jag.AngularClFunction.apply(theta, 0.0, ell, sid, 64, 1)
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            theta * 2.0
            jag.AngularClFunction.apply(theta, 0.0, ell, sid, 64, 1)
