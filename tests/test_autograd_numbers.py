"""angular_cl_torch of a cosmology that holds numbers, all or but for one
parameter: the vector that reaches the device call, and its values against
angular_cl (the same kernels)."""
import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd import autograd as jag

VALUES = (0.25, 0.05, 0.7, 0.96, 0.8, 0.01, -0.95, 0.1)


class FakeContext:
    def tracer_set(self, entries):
        return 1


@pytest.mark.parametrize("tensor", [None, 0, 5, 7])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_vector_of_the_call(monkeypatch, tensor, dtype):
    calls = []

    class Record:
        @staticmethod
        def apply(theta, omega_k, *a):
            calls.append((theta, omega_k))

    monkeypatch.setattr(jag, "default_context", FakeContext)
    monkeypatch.setattr(jag, "AngularClFunction", Record)
    params = [torch.tensor(v, dtype=dtype) if i == tensor else v for i, v in enumerate(VALUES)]
    jag.angular_cl_torch(params, np.array([10.0]), [jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, 0.8)])])
    theta, omega_k = calls[0]
    want = [float(params[i]) for i in jag.GRAD_INDEX]
    assert theta.dtype == torch.float64 and theta.device.type == "cpu"
    assert theta.tolist() == [want] and omega_k == float(params[5])


@pytest.mark.gpu
def test_numbers_give_the_spectra():
    ell = np.geomspace(20.0, 800.0, 9)
    probes = [jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, 0.8)])]
    ref = jc.cl.angular_cl(jc.Cosmology(*VALUES), ell, probes, n_z=64)
    out = jag.angular_cl_torch(VALUES, ell, probes, n_z=64)
    assert out.device.type == "cpu"
    np.testing.assert_array_equal(out[0].numpy(), ref)
