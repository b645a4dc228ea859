"""Served batches whose live requests lie on both sides of the lensing kernel's
switch between two and more cosmologies a block (256 at n_z 256 on 256 compute
units) and whose column tiles leave a part of the XCDs without one, against the
batch path: float32 sums over a split differently, 5e-6 of a spectrum's largest
value."""
import numpy as np
import pytest

import jax_cosmo_amd as jc
from jax_cosmo_amd import serving
from test_gpu_forward_table import PARAMS, make_probes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ctile", [0, 1, 8, 16])
@pytest.mark.parametrize("n,n_ell", [(1, 20), (3, 200), (256, 30), (300, 64)])
def test_served_against_batch(n, n_ell, ctile):
    probes = make_probes(5, 2)
    srv = serving.Server(probes, max_batch=320, max_grad=1, max_ell=200, slots=1, n_z=(256,), wl_ctile=ctile)
    ell = np.geomspace(15.0, 3000.0, n_ell)
    reqs = [dict(cosmo=PARAMS[i % 3], tracers=list(range(7)), ell=ell, n_z=256) for i in range(n)]
    prep = srv.prepare(reqs)
    srv.submit_prepared(prep)
    srv.wait(0)
    done = 0
    while done < n:
        done += srv.poll_array(n).size
    ref = jc.cl.angular_cl_batch(PARAMS, ell, probes, n_z=256)
    scale = np.abs(ref).max(axis=2, keepdims=True)
    for i, (cl, _) in enumerate(prep.outs):
        assert (np.abs(cl - ref[i % 3]) <= 5e-6 * scale[i % 3]).all()
