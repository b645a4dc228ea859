"""The weak-lensing kernel over its launch shapes (few blocks with many waves,
one or two cosmologies a block, up to 5 and up to 10 bins), at node counts that
end inside a block of 64 and with and without nodes nearer than 1 Mpc/h, whose
clips act, against the FP64 oracle: C_ell to 1e-4, derivatives to 1e-3 (the
library's stated tolerances)."""
import numpy as np
import pytest
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd._native import default_context
from oracle import jc_oracle as O
from test_gpu_forward_table import PARAMS

pytestmark = pytest.mark.gpu

IDX = [0, 1, 2, 3, 4, 6, 7]


@pytest.mark.parametrize("nb,zmax,n_z", [(1, 0.01, 62), (5, 4.0, 130), (6, 4.0, 62), (10, 0.01, 66)])
def test_wl_shapes_against_oracle(nb, zmax, n_z):
    ctx = default_context()
    z0 = np.linspace(0.4, 0.9, nb) * zmax / 3
    ell = np.geomspace(20.0, 800.0, 5)
    P = nb * (nb + 1) // 2
    probes = [jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, z, zmax=zmax) for z in z0])]
    pv = torch.tensor(PARAMS[0], requires_grad=True)
    ref = O.angular_cl(O.Cosmo.from_vector(pv), torch.tensor(ell),
                       [O.WeakLensing([O.smail_nz(1.0, 2.0, z, zmax=zmax) for z in z0])], N=n_z)
    rng = np.random.default_rng(nb)
    u = (rng.uniform(0.5, 1.5, (P, 5)) / ref.detach().numpy()).astype(np.float32)
    (ref * torch.tensor(u.astype(np.float64))).sum().backward()
    grad = pv.grad.numpy()[IDX]
    jc.cl._check_fns(jc.transfer.Eisenstein_Hu, jc.power.halofit)
    sid = ctx.tracer_set(jc.cl.tracer_entries(probes))
    for B in (1, 300, 515):  # on 256 compute units: each launch shape at n_z 62
        params = PARAMS[np.arange(B) % 3]
        cl = ctx.angular_cl(params, sid, ell, n_z, P)
        np.testing.assert_allclose(cl[0], ref.detach().numpy(), rtol=1e-4)
        np.testing.assert_allclose(cl[3:], cl[:-3][: max(B - 3, 0)], rtol=1e-6)
        th = ctx.angular_cl_vjp(params, sid, ell, n_z, np.broadcast_to(u, (B, P, 5)).copy())
        np.testing.assert_allclose(th[0], grad, rtol=1e-3)
        np.testing.assert_allclose(th[3:], th[:-3][: max(B - 3, 0)], rtol=1e-5)
        v = rng.normal(size=7)
        dot = ctx.angular_cl_jvp(params, np.broadcast_to(v, (B, 7)).copy(), sid, ell, n_z, P)[1]
        lhs = (dot[0].astype(np.float64) * u).sum()
        assert abs(lhs - grad @ v) <= 1e-3 * np.abs(grad * v).sum()
