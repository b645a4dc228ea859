"""Host-pointer calls whose inputs and results lie just inside and just outside
the pinned buffers (128 KB in, 512 KB out): the same bits as the device-pointer
calls, which pass through neither."""
import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,n_ell", [(1, 1), (99, 437), (100, 437), (50, 437), (2040, 64), (2040, 65), (1, 16377)])
def test_host_and_device_pointers_agree(B, n_ell):
    ctx = default_context()
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(make_probes(1, 1)))
    params = np.ascontiguousarray(PARAMS[np.arange(B) % 3])
    ell = np.geomspace(20.0, 2000.0, n_ell)
    tan = np.random.default_rng(B).normal(size=(B, 7))
    cbar = np.random.default_rng(B + 1).normal(size=(B, 3, n_ell)).astype(np.float32)
    dev = [torch.as_tensor(x, device="cuda") for x in (params, ell, tan, cbar)]
    out, dot = (torch.empty((B, 3, n_ell), device="cuda") for _ in range(2))
    th = torch.empty((B, 7), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.angular_cl_dev(dev[0].data_ptr(), B, sid, dev[1].data_ptr(), n_ell, 62, out.data_ptr())
    ctx.synchronize()
    np.testing.assert_array_equal(ctx.angular_cl(params, sid, ell, 62, 3), out.cpu().numpy())
    ctx.angular_cl_jvp_dev(dev[0].data_ptr(), dev[2].data_ptr(), B, sid, dev[1].data_ptr(), n_ell, 62,
                           out.data_ptr(), dot.data_ptr())
    ctx.synchronize()
    for got, want in zip(ctx.angular_cl_jvp(params, tan, sid, ell, 62, 3), (out, dot)):
        np.testing.assert_array_equal(got, want.cpu().numpy())
    ctx.angular_cl_vjp_dev(dev[0].data_ptr(), B, sid, dev[1].data_ptr(), n_ell, 62, dev[3].data_ptr(), th.data_ptr())
    ctx.synchronize()
    np.testing.assert_array_equal(ctx.angular_cl_vjp(params, sid, ell, 62, cbar), th.cpu().numpy())
