"""Performance cases of the Limber C_ell framework.

Each case is one call (or one queue of requests) that a program using
jax_cosmo_amd makes, through the public entry points: single spectra, batches,
gradients, Jacobians, Gaussian likelihoods with block-diagonal and dense
covariances, and a served queue of uneven requests.

``prepare`` makes what the program holds before the call, ``run`` is one pass,
``work`` counts what the pass cannot do without, and ``exact`` evaluates the
same quantities in 64 bits with plain torch, from the published formulae and
the discretisation of jax_cosmo (its tables, interpolation rule and quadrature
nodes).
"""
import math

import numpy as np
import torch

import jax_cosmo_amd as jc
from jax_cosmo_amd import autograd as jag
from jax_cosmo_amd import likelihood as jlk
from jax_cosmo_amd import serving
from jax_cosmo_amd._native import default_context

# the parameter box of the seeded cosmologies: Omega_c, Omega_b, h, n_s,
# sigma8, w0, wa
BOX_LO = np.array([0.2, 0.04, 0.6, 0.9, 0.7, -1.3, -0.5])
BOX_HI = np.array([0.35, 0.06, 0.8, 1.0, 0.9, -0.7, 0.5])
FREE = [0, 1, 2, 3, 4, 6, 7]  # columns of the box in Cosmology(...) order; 5 is Omega_k = 0
WL_Z0 = (0.5, 0.75, 1.0, 1.25, 1.5)
NC_MU = (0.3, 0.6, 0.9, 1.2, 1.5)
ZMAX = 10.0


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one cosmology, one lensing bin, as in an interactive session or a scalar sampler
        dict(name="shear_one", kind="single", wl=1, nc=0, ell=50, n_z=256),
        # one cosmology of a full 3x2pt survey: a sampler that evaluates point by point
        dict(name="survey_one", kind="single", wl=5, nc=5, ell=100, n_z=512),
        # C_ell and the 7-parameter gradient of one cosmology with torch scalars: a gradient-based sampler (HMC)
        dict(name="grad_one", kind="grad_one", wl=2, nc=2, ell=50, n_z=512),
        # dC/dtheta of one cosmology: a Fisher forecast
        dict(name="jacobian_one", kind="jacobian", wl=5, nc=5, ell=100, n_z=512, batch=1),
        # an ensemble sampler's walkers, odd sizes, few multipoles
        dict(name="batch_walkers", kind="batch", wl=4, nc=3, ell=45, n_z=256, batch=37),
        # the batch workload of the benchmark
        dict(name="batch_1024", kind="batch", wl=5, nc=5, ell=100, n_z=512, batch=1024),
        # training set of an emulator: more cosmologies, multipoles and a finer grid
        dict(name="batch_large", kind="batch", wl=5, nc=5, ell=200, n_z=1024, batch=2048),
        # C_ell and gradients of a batch through torch: variational inference, many HMC chains
        dict(name="grad_256", kind="grad", wl=5, nc=5, ell=100, n_z=512, batch=256),
        # an uneven request queue, drained by the continuous-batching server
        dict(name="served_300", kind="serve", requests=300),
        # log-likelihoods of a batch of means under a block-diagonal covariance
        dict(name="loglike_sparse", kind="sparse", tracers=10, ell=100, batch=256),
        # the same under a dense covariance whose factor is resident
        dict(name="loglike_dense", kind="dense", tracers=10, ell=100, batch=256),
        # factorising a dense covariance, once per analysis
        dict(name="cholesky", kind="cholesky", tracers=10, ell=50),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["single", "grad_one", "jacobian", "batch", "batch", "batch", "grad", "serve", "sparse", "dense",
                       "cholesky"])
    wl, nc = rng.randint(0, 5), rng.randint(0, 5)
    if wl + nc == 0:
        wl = 1
    spectra = dict(kind=kind, wl=wl, nc=nc, ell=_log_int(rng, 20, 200), n_z=rng.choice([256, 300, 512, 770, 1024]))
    if kind in ("single", "grad_one"):
        return spectra
    if kind == "jacobian":
        return dict(spectra, batch=_log_int(rng, 1, 6))
    if kind == "batch":
        return dict(spectra, batch=_log_int(rng, 2, 2048))
    if kind == "grad":
        return dict(spectra, batch=_log_int(rng, 2, 128))
    if kind == "serve":
        return dict(kind=kind, requests=_log_int(rng, 8, 300))
    t = rng.randint(2, 10)
    if kind == "cholesky":
        return dict(kind=kind, tracers=t, ell=_log_int(rng, 20, 50))
    return dict(kind=kind, tracers=t, ell=_log_int(rng, 20, 100), batch=_log_int(rng, 1, 256))


# ---------------------------------------------------------------- inputs
def _cosmologies(seed, n):
    p = np.zeros((n, 8))
    p[:, FREE] = BOX_LO + (BOX_HI - BOX_LO) * np.random.default_rng(seed).random((n, 7))
    return p


def _ell(case):
    return np.geomspace(10.0, 5000.0, case["ell"])


def _probes(wl, nc):
    out = []
    if wl:
        out.append(jc.probes.WeakLensing([jc.redshift.smail_nz(1.0, 2.0, z, gals_per_arcmin2=10.0) for z in WL_Z0[:wl]],
                                         sigma_e=0.26))
    if nc:
        out.append(jc.probes.NumberCounts([jc.redshift.gaussian_nz(m, 0.1, gals_per_arcmin2=10.0) for m in NC_MU[:nc]],
                                          jc.bias.constant_linear_bias(1.5)))
    return out


def _pairs(t):
    return t * (t + 1) // 2


def _cotangent(case, seed, n):
    """A loss's dL/dC_ell: noise weighted as l (l + 1) C_ell / 2 pi is."""
    p = _pairs(case["wl"] + case["nc"])
    w = np.random.default_rng(seed + 1).normal(size=(n, p, case["ell"]))
    ell = _ell(case)
    return (w * ell * (ell + 1.0) / (2.0 * math.pi)).astype(np.float32)


def _requests(case, seed):
    """Uneven requests: 1..10 bins of the pool, 20..200 multipoles, one of
    three Simpson sizes.  The shapes go with the case, the cosmologies with
    the seed."""
    rng = np.random.default_rng(case["requests"])
    reqs = []
    for c in _cosmologies(seed, case["requests"]):
        t = int(rng.integers(1, 11))
        reqs.append(dict(cosmo=c, tracers=np.sort(rng.choice(10, size=t, replace=False)).tolist(),
                         ell=np.geomspace(10.0, 5000.0, int(rng.integers(20, 201))),
                         n_z=int(rng.choice([256, 512, 1024]))))
    return reqs


def _gaussian_problem(case, seed):
    """Observed spectra, their Gaussian covariance, a data vector and a batch
    of means near it, from the seed alone: correlated power-law spectra plus
    shot noise on the auto-spectra, f_sky = 0.25."""
    rng = np.random.default_rng(seed)
    t, n_ell = case["tracers"], case["ell"]
    p = _pairs(t)
    ell = np.geomspace(10.0, 5000.0, n_ell)
    amp = 1e-8 * 10.0 ** rng.uniform(0.0, 1.0, t)
    slope = rng.uniform(0.8, 1.4, t)
    root = np.sqrt(amp)[:, None] * (ell / 100.0) ** (-0.5 * slope[:, None])
    corr = 0.85 ** np.abs(np.arange(t)[:, None] - np.arange(t)[None, :])
    signal = corr[:, :, None] * root[:, None, :] * root[None, :, :]
    obs = signal + 1e-9 * np.eye(t)[:, :, None]
    i, j = np.triu_indices(t)
    norm = (2.0 * ell + 1.0) * np.gradient(ell) * 0.25
    cov = (obs[i[:, None], i[None, :]] * obs[j[:, None], j[None, :]]
           + obs[i[:, None], j[None, :]] * obs[j[:, None], i[None, :]]) / norm  # [P, P, n_ell]
    mean = signal[i, j]  # [P, n_ell]
    scatter = np.sqrt(np.einsum("ppl->pl", cov))
    data = mean + scatter * rng.normal(size=mean.shape)
    mu = (mean + 0.5 * scatter * rng.normal(size=(case.get("batch", 1), p, n_ell))).astype(np.float32)
    return cov, data.reshape(-1), mu, rng


def _dense_cov(cov, rng):
    """The dense form of a block-diagonal covariance plus two modes common to
    all multipoles (a super-sample term)."""
    p, _, n_ell = cov.shape
    n = p * n_ell
    scale = np.sqrt(np.einsum("ppl->pl", cov)).reshape(-1)
    modes = 0.3 * scale[:, None] * rng.normal(size=(n, 2))
    dense = modes @ modes.T
    view = dense.reshape(p, n_ell, p, n_ell)
    diag = np.arange(n_ell)
    view[:, diag, :, diag] += np.transpose(cov, (2, 0, 1))
    return dense


def prepare(case, seed):
    k = case["kind"]
    if k in ("sparse", "dense", "cholesky"):
        cov, data, mu, rng = _gaussian_problem(case, seed)
        if k == "sparse":
            return dict(kind=k, data=data, mu=mu, cov=cov)
        dense = _dense_cov(cov, rng)
        if k == "cholesky":
            return dict(kind=k, cov=dense)
        # the factor is the plan that the program keeps
        return dict(kind=k, data=data, mu=mu.reshape(mu.shape[0], -1), factor=jlk.cholesky(dense))
    if k == "serve":
        srv = serving.Server(_probes(5, 5), max_batch=512, max_grad=160, max_ell=200, slots=2, n_z=(256, 512, 1024))
        return dict(kind=k, server=srv, prep=srv.prepare(_requests(case, seed)))
    s = dict(kind=k, ell=_ell(case), probes=_probes(case["wl"], case["nc"]), n_z=case["n_z"])
    n = case.get("batch", 1)
    params = _cosmologies(seed, n)
    if k == "single":
        s["cosmo"] = jc.Cosmology(*[float(v) for v in params[0]])
    elif k == "batch":
        s["params"] = torch.as_tensor(params, device="cuda")
    elif k == "jacobian":
        s["params"] = params
    else:
        # torch's default dtype for the parameters, so float32 gradients
        theta = torch.as_tensor(params[:, FREE], device="cuda").to(torch.float32)
        cbar = torch.as_tensor(_cotangent(case, seed, n), device="cuda")
        if k == "grad_one":
            s["theta"] = [theta[0, i].clone().requires_grad_(True) for i in range(7)]
            s["cbar"] = cbar[0]
        else:
            s["theta"] = theta.requires_grad_(True)
            s["cbar"] = cbar
            s["set_id"] = default_context().tracer_set(jc.cl.tracer_entries(s["probes"]))
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    k = s["kind"]
    if k == "single":
        return jc.cl.angular_cl(s["cosmo"], s["ell"], s["probes"], n_z=s["n_z"])
    if k == "batch":
        return jc.cl.angular_cl_batch(s["params"], s["ell"], s["probes"], n_z=s["n_z"])
    if k == "jacobian":
        return jag.angular_cl_jacobian(s["params"], s["ell"], s["probes"], n_z=s["n_z"])
    if k == "grad_one":
        t = s["theta"]
        cosmo = jc.Cosmology(t[0], t[1], t[2], t[3], t[4], 0.0, t[5], t[6])
        cl = jc.cl.angular_cl(cosmo, s["ell"], s["probes"], n_z=s["n_z"])
        return cl.detach(), torch.stack(torch.autograd.grad(cl, t, s["cbar"]))
    if k == "grad":
        cl = jag.AngularClFunction.apply(s["theta"], 0.0, s["ell"], s["set_id"], s["n_z"], s["cbar"].shape[1])
        return cl.detach(), torch.autograd.grad(cl, s["theta"], s["cbar"])[0]
    if k == "serve":
        srv, n = s["server"], len(s["prep"].keeps)
        srv.submit_prepared(s["prep"])
        srv.wait(0)
        done = 0
        while done < n:
            done += srv.poll_array(n).size
        return np.concatenate([cl.ravel() for cl, _ in s["prep"].outs])
    if k == "sparse":
        return jlk.log_likelihood_batch(s["data"], s["mu"], s["cov"])
    if k == "dense":
        return jlk.log_likelihood_batch(s["data"], s["mu"], s["factor"])
    f = jlk.cholesky(s["cov"])
    return f.L, f.logdet


# ---------------------------------------------------------------- what a pass cannot do without
def _spectra_work(n, t, wl, n_ell, n_z, columns):
    """Bytes and operations of C_ell for n cosmologies.  A (cosmology, ell, a)
    point is about 60 operations of P_nl and a multiply-add per pair (and per
    derivative `columns`); a cosmology's tables are the halofit moments (four
    multiply-adds on 257 x 256 nodes) and, per lensing bin, a multiply-add on
    n_z x 256 nodes after about 8 operations for the lensing efficiency."""
    p = _pairs(t)
    point = n * n_ell * (n_z + 1)
    flops = point * (60.0 * columns + 2.0 * p * columns)
    tables = 257 * 256 * 8.0 + (n_z * 256 * (8.0 + 2.0 * wl) if wl else 0.0) + 200.0 * n_z + 1e5
    return n * 8 * 8 + n_ell * 8, flops + n * tables * columns, n * p * n_ell * 4


def work(case):
    k = case["kind"]
    if k in ("single", "batch", "jacobian", "grad_one", "grad"):
        n = case.get("batch", 1)
        t = case["wl"] + case["nc"]
        # a derivative in 7 directions: 7 tangents forwards, about 3 passes in reverse
        cols = 8 if k == "jacobian" else (4 if k.startswith("grad") else 1)
        rd, fl, wr = _spectra_work(n, t, case["wl"], case["ell"], case["n_z"], cols)
        if k == "jacobian":
            wr *= 7
        if k.startswith("grad"):
            rd += wr  # the cotangent
            wr += n * 7 * 4
        return {"bytes": rd + wr, "flops": fl}
    if k == "serve":
        total = {"bytes": 0.0, "flops": 0.0}
        # the queue's mean request: 5.5 bins, 110 multipoles, n_z 597
        rd, fl, wr = _spectra_work(case["requests"], 6, 3, 110, 597, 1)
        total["bytes"] += rd + wr
        total["flops"] += fl
        return total
    p = _pairs(case["tracers"])
    n = p * case["ell"]
    if k == "cholesky":
        return {"bytes": 16.0 * n * n, "flops": n ** 3 / 3.0}
    b = case["batch"]
    if k == "sparse":
        return {"bytes": 8.0 * p * n + 8.0 * n + 4.0 * b * n + 8.0 * b,
                "flops": case["ell"] * p ** 3 / 3.0 + 2.0 * b * p * n}
    return {"bytes": 4.0 * n * n + 8.0 * n + 4.0 * b * n + 8.0 * b, "flops": float(b) * n * n}


# ---------------------------------------------------------------- 64 bits, plain torch
RH, H0, C_KMS, TCMB = 2997.92458, 100.0, 299792.458, 2.726


def _simpson(n, h, dev):
    w = torch.full((n + 1,), 2.0, dtype=torch.float64, device=dev)
    w[1::2] = 4.0
    w[0] = w[-1] = 1.0
    return w * (h / 3.0)


def _lin(a, b, n, dev):
    return torch.linspace(a, b, n, dtype=torch.float64, device=dev)


def _segments(x, xp):
    """Nearest-node linear interpolation of jax_cosmo: the node next to x
    (clipped to the interior), and the neighbour on x's side of it."""
    hi = torch.searchsorted(xp, x.contiguous()).clamp(1, xp.numel() - 1)
    near = torch.where((x - xp[hi - 1]) ** 2 <= (x - xp[hi]) ** 2, hi - 1, hi).clamp(1, xp.numel() - 2)
    xc = torch.minimum(torch.maximum(x, xp[1]), xp[-2])
    other = torch.where(xc - xp[near] < 0, near - 1, near + 1)
    return near, other, (x - xp[near]) / (xp[other] - xp[near])


def _at(f, seg):
    """f [B, nodes] interpolated at the segments' points: [B, ...]."""
    i, j, t = seg
    fi = f[:, i.reshape(-1)].reshape(f.shape[0], *i.shape)
    fj = f[:, j.reshape(-1)].reshape(f.shape[0], *i.shape)
    return fi + (fj - fi) * t


class _Model:
    """C_ell in 64 bits for the cosmologies th [B, 8]."""

    def __init__(self, th):
        self.dev = th.device
        oc, ob, h, ns, s8, ok, w0, wa = [th[:, i:i + 1] for i in range(8)]
        self.ob, self.h, self.ns, self.ok, self.w0, self.wa = ob, h, ns, ok, w0, wa
        self.om = oc + ob
        self.ode = 1.0 - ok - self.om
        self._background()
        self._transfer_constants()
        # sigma_8: Romberg on 129 samples of ln k in [-4, 3]
        lk = _lin(-4.0, 3.0, 129, self.dev)
        k = lk.exp()
        x = 8.0 * k
        win = 3.0 * (x.sin() - x * x.cos()) / x ** 3
        f = k * (k * win) ** 2 * self.transfer(k[None]) ** 2 * (ns * lk).exp()
        rows = []
        for lev in range(8):
            g = f[:, ::128 >> lev]
            row = [(g.sum(1) - 0.5 * (g[:, 0] + g[:, -1])) * (7.0 / (1 << lev))]
            for q in range(lev):
                row.append((4.0 ** (q + 1) * row[q] - rows[-1][q]) / (4.0 ** (q + 1) - 1.0))
            rows.append(row)
        self.norm = s8 ** 2 / (rows[-1][-1][:, None] / (2.0 * math.pi ** 2))
        # halofit: Gaussian moments of the a = 1 linear power
        self.lk = _lin(math.log(1e-4), math.log(1e4), 257, self.dev)
        self.kh = self.lk.exp()
        g1 = _at(self.grow, _segments(torch.ones(1, dtype=torch.float64, device=self.dev), self.a_g)).clamp(0.0, 1.0)
        p1 = (ns * self.lk).exp() * self.transfer(self.kh[None]) ** 2 * g1 ** 2 * self.norm
        dx = (math.log(1e4) - math.log(1e-4)) / 256
        self.wp = _simpson(256, dx, self.dev) * p1 * self.kh ** 3 / (2.0 * math.pi ** 2)
        self.lr = _lin(math.log(1e-4), math.log(1e1), 256, self.dev)
        self.sig = self.wp @ (-(self.kh[:, None] * self.lr.exp()) ** 2).exp()

    def e2(self, a):
        fde = -3.0 * (1.0 + self.w0 + self.wa) * a.log() + 3.0 * self.wa * (a - 1.0)
        self.de = self.ode * fde.exp()
        return self.om * a ** -3 + self.ok * a ** -2 + self.de

    def _background(self):
        # chi: cumulative Simpson in ln a with midpoints on 256 nodes
        la = (10.0 ** _lin(-3.0, 0.0, 256, self.dev)).log()
        self.a_c = 10.0 ** _lin(-3.0, 0.0, 256, self.dev)

        def f(t):
            a = t.exp()
            return RH / (a * self.e2(a).sqrt())

        h = la[1:] - la[:-1]
        step = h / 6.0 * (f(la[:-1]) + 4.0 * f(la[:-1] + h / 2.0) + f(la[1:]))
        c = torch.cat([torch.zeros_like(step[:, :1]), step.cumsum(1)], 1)
        self.chi = c[:, -1:] - c
        # growth: RK4 in a on 128 nodes from (a_0, 1)
        self.a_g = 10.0 ** _lin(-3.0, 0.0, 128, self.dev)
        mid = self.a_g[:-1] + (self.a_g[1:] - self.a_g[:-1]) / 2.0

        def qr(x):
            e2 = self.e2(x)
            w = self.w0 + (1.0 - x) * self.wa
            omx = self.om * x ** -3 / e2
            return (2.0 - 0.5 * (omx + (1.0 + 3.0 * w) * self.de / e2)) / x, 1.5 * omx / x ** 2

        qn, rn = qr(self.a_g)
        qm, rm = qr(mid)
        y = torch.zeros_like(self.om[:, 0]) + self.a_g[0]
        v = torch.ones_like(y)
        ds = [y]
        for i in range(1, 128):
            s = self.a_g[i] - self.a_g[i - 1]
            k1, l1 = v, rn[:, i - 1] * y - qn[:, i - 1] * v
            ya, va = y + s / 2 * k1, v + s / 2 * l1
            k2, l2 = va, rm[:, i - 1] * ya - qm[:, i - 1] * va
            ya, va = y + s / 2 * k2, v + s / 2 * l2
            k3, l3 = va, rm[:, i - 1] * ya - qm[:, i - 1] * va
            ya, va = y + s * k3, v + s * l3
            k4, l4 = va, rn[:, i] * ya - qn[:, i] * va
            y = y + s / 6.0 * (k1 + 2 * k2 + 2 * k3 + k4)
            v = v + s / 6.0 * (l1 + 2 * l2 + 2 * l3 + l4)
            ds.append(y)
        d = torch.stack(ds, 1)
        self.grow = d / d[:, -1:]

    def _transfer_constants(self):
        """Eisenstein & Hu (1998), eqs. 2-7, 11, 12, 14, 15, 23, 24."""
        t2 = (TCMB / 2.7) ** 2
        wm, wb = self.om * self.h ** 2, self.ob * self.h ** 2
        self.fb = self.ob / self.om
        self.keq = 7.46e-2 * wm / t2 / self.h
        zeq = 2.5e4 * wm / t2 ** 2
        b1 = 0.313 * wm ** -0.419 * (1.0 + 0.607 * wm ** 0.674)
        zd = 1291.0 * wm ** 0.251 / (1.0 + 0.659 * wm ** 0.828) * (1.0 + b1 * wb ** (0.238 * wm ** 0.223))
        rd, req = 31.5 * wb / t2 ** 2 * 1e3 / zd, 31.5 * wb / t2 ** 2 * 1e3 / zeq
        self.s = 2.0 / (3.0 * self.keq) * (6.0 / req).sqrt() * (
            ((1.0 + rd).sqrt() + (rd + req).sqrt()) / (1.0 + req.sqrt())).log()
        self.ksilk = 1.6 * wb ** 0.52 * wm ** 0.73 * (1.0 + (10.4 * wm) ** -0.95) / self.h
        fc = 1.0 - self.fb
        a1 = (46.9 * wm) ** 0.670 * (1.0 + (32.1 * wm) ** -0.532)
        a2 = (12.0 * wm) ** 0.424 * (1.0 + (45.0 * wm) ** -0.582)
        self.ac = a1 ** -self.fb * a2 ** -(self.fb ** 3)
        self.bc = 1.0 / (1.0 + 0.944 / (1.0 + (458.0 * wm) ** -0.708) * (fc ** ((0.395 * wm) ** -0.0266) - 1.0))
        y = (1.0 + zeq) / (1.0 + zd)
        x = (1.0 + y).sqrt()
        self.ab = 2.07 * self.keq * self.s * (1.0 + rd) ** -0.75 * y * (
            -6.0 * x + (2.0 + 3.0 * y) * ((x + 1.0) / (x - 1.0)).log())
        self.bn = 8.41 * wm ** 0.435
        self.bb = 0.5 + self.fb + (3.0 - 2.0 * self.fb) * ((17.2 * wm) ** 2 + 1.0).sqrt()

    def transfer(self, k, b=slice(None)):
        """T(k) at k [b, ...] of the cosmologies b."""
        def of(v):
            return v[b].reshape(-1, *([1] * (k.dim() - 1)))

        q = k / (13.41 * of(self.keq))
        c0 = 386.0 / (1.0 + 69.9 * q ** 1.08)

        def t0(inv_alpha, beta):
            ln = (math.e + 1.8 * beta * q).log()
            return ln / (ln + (14.2 * inv_alpha + c0) * q ** 2)

        ks = k * of(self.s)
        f = 1.0 / (1.0 + (ks / 5.4) ** 4)
        tc = f * t0(1.0, of(self.bc)) + (1.0 - f) * t0(1.0 / of(self.ac), of(self.bc))
        kt = ks / (1.0 + (of(self.bn) / ks) ** 3) ** (1.0 / 3.0)
        tb = (t0(1.0, 1.0) / (1.0 + (ks / 5.2) ** 2)
              + of(self.ab) / (1.0 + (of(self.bb) / ks) ** 3) * (-(k / of(self.ksilk)) ** 1.4).exp()) * kt.sin() / kt
        fb = of(self.fb)
        return fb * tb + (1.0 - fb) * tc

    def spectra(self, b, ell, wl, nc, n_z):
        """C [len(b), P, n_ell] of the cosmologies b (a slice), with the
        lensing bins wl and the clustering bins nc by index."""
        one = _Model.__new__(_Model)
        for n, v in self.__dict__.items():
            setattr(one, n, v[b] if isinstance(v, torch.Tensor) and v.dim() == 2 else v)
        one._limber_setup(n_z)
        rows = [one._lensing(WL_Z0[i], n_z) for i in wl] + [one._clustering(NC_MU[i]) for i in nc]
        r = torch.stack(rows, 1)  # [b, T, Na]
        # P_nl at k = (ell + 1/2) / chi
        chi1 = one.chia.clamp(min=1.0)[:, :, None]
        k = (ell + 0.5) / chi1
        lin = k ** one.ns[:, :, None] * one.transfer(k) ** 2 * (one.d ** 2 * one.norm)[:, :, None]
        d2 = k ** 3 * lin / (2.0 * math.pi ** 2)
        hf = {n: v[:, :, None] for n, v in one.hf.items()}
        y = k * hf["rnl"]
        dq = d2 * (1.0 + d2) ** hf["beta"] / (1.0 + hf["alpha"] * d2) * (-(y / 4.0 + y ** 2 / 8.0)).exp()
        dh = hf["a"] * y ** (3.0 * hf["f1"]) / (
            1.0 + hf["b"] * y ** hf["f2"] + (hf["c"] * hf["f3"] * y) ** (3.0 - hf["gamma"]))
        m = 2.0 * math.pi ** 2 / k ** 3 * (dq + dh / (1.0 + hf["nu"] / y ** 2)) * one.weight[:, :, None]
        fac = (ell * (ell - 1.0) * (ell + 1.0) * (ell + 2.0)).sqrt() / (ell + 0.5) ** 2
        t = len(rows)
        i, j = torch.triu_indices(t, t, device=self.dev)
        scale = torch.where(torch.arange(t, device=self.dev)[:, None] < len(wl), fac[None], torch.ones_like(fac)[None])
        return torch.matmul((r[:, i] * r[:, j]).contiguous(), m) * (scale[i] * scale[j])

    def _limber_setup(self, n_z):
        a = _lin(1.0 / (1.0 + ZMAX), 1.0, n_z + 1, self.dev)
        self.a, self.z = a, 1.0 / a - 1.0
        self.chia = _at(self.chi, _segments(a, self.a_c)).clamp(min=0.0)
        self.d = _at(self.grow, _segments(a, self.a_g)).clamp(0.0, 1.0)
        e2 = self.e2(a)
        omx, dex = self.om * a ** -3 / e2, self.de / e2
        self.hub = H0 * e2.sqrt()
        w = _simpson(n_z, (1.0 - 1.0 / (1.0 + ZMAX)) / n_z, self.dev)
        self.weight = w * RH / (a ** 2 * e2.sqrt()) / (self.chia ** 2).clamp(min=1.0) / C_KMS ** 2
        # nonlinear scale: the interpolation rule above on the decreasing
        # table sigma^2(R, a), at sigma^2 = 1
        sig = self.d[:, :, None] ** 2 * self.sig[:, None, :]
        sv = sig.detach()
        ind = ((1.0 - sv) ** 2).argmin(2, keepdim=True).clamp(1, 254)
        left = (sv[:, :, 254:255] - sv.gather(2, ind)) < 0
        oth = torch.where(left, ind - 1, ind + 1)
        si, so = sig.gather(2, ind), sig.gather(2, oth)
        slope = (self.lr[oth] - self.lr[ind]) / (so - si)
        rnl = (self.lr[ind] + slope * (1.0 - si)).exp().clamp(min=1e-6)  # [b, Na, 1]
        y2 = (self.kh * rnl) ** 2
        e = self.wp[:, None, :] * (-y2).exp() * self.d[:, :, None] ** 2
        s1, s2 = (e * y2).sum(2), (e * y2 ** 2).sum(2)
        n = 2.0 * s1 - 3.0
        c = (2.0 * s1) ** 2 + 4.0 * (s1 - s2)
        # Takahashi et al. (2012)
        wde = dex * (1.0 + self.w0 + (1.0 - a) * self.wa)
        ten = math.log(10.0)
        self.hf = dict(
            rnl=rnl[:, :, 0],
            a=(ten * (1.5222 + 2.8553 * n + 2.3706 * n ** 2 + 0.9903 * n ** 3 + 0.2250 * n ** 4 - 0.6038 * c
                      + 0.1749 * wde)).exp(),
            b=(ten * (-0.5642 + 0.5864 * n + 0.5716 * n ** 2 - 1.5474 * c + 0.2279 * wde)).exp(),
            c=(ten * (0.3698 + 2.0404 * n + 0.8161 * n ** 2 + 0.5869 * c)).exp(),
            gamma=0.1971 - 0.0843 * n + 0.8460 * c,
            alpha=(6.0835 + 1.3373 * n - 0.1959 * n ** 2 - 5.5274 * c).abs(),
            beta=2.0379 - 0.7354 * n + 0.3157 * n ** 2 + 1.2490 * n ** 3 + 0.3980 * n ** 4 - 0.1682 * c,
            nu=(ten * (5.2105 + 3.6902 * n)).exp(),
            f1=omx ** -0.0307, f2=omx ** -0.0585, f3=omx ** 0.0743)

    def _nz(self, f):
        """n(z) normalised by a 256-interval Simpson rule over [0, zmax]."""
        zn = _lin(0.0, ZMAX, 257, self.dev)
        norm = (_simpson(256, ZMAX / 256, self.dev) * f(zn)).sum()
        return lambda z: f(z) / norm

    def _clustering(self, mu):
        nz = self._nz(lambda z: (-0.5 * ((z - mu) / 0.1) ** 2).exp())
        return nz(self.z) * 1.5 * self.hub

    def _lensing(self, z0, n_z):
        nz = self._nz(lambda z: z * (-(z / z0) ** 2).exp())
        u = _lin(0.0, 1.0, 257, self.dev)
        zi = self.z[:, None] + (ZMAX - self.z[:, None]) * u  # [Na, 257]
        w = _simpson(256, 1.0, self.dev) * (ZMAX - self.z[:, None]) / 256
        if not hasattr(self, "_eff"):
            ci = _at(self.chi, _segments(1.0 / (1.0 + zi), self.a_c))
            self._eff = (ci - self.chia[:, :, None]).clamp(min=0.0) / ci.clamp(min=1.0)
        q = (self._eff * (w * nz(zi))).sum(2)
        return 3.0 * H0 ** 2 * self.om / (2.0 * C_KMS) * (1.0 + self.z) * self.chia * q


def _spectra64(th, ell, wl, nc, n_z, chunk_points=3_000_000):
    m = _Model(th)
    step = max(1, int(chunk_points // ((n_z + 1) * max(len(ell), 257))))
    return torch.cat([m.spectra(slice(s, s + step), ell, wl, nc, n_z) for s in range(0, th.shape[0], step)])


def _tangent64(th, d, *args):
    """(C, dC/dtheta_d) by forward-mode differentiation."""
    import torch.autograd.forward_ad as fwd

    e = torch.zeros_like(th)
    e[:, FREE[d]] = 1.0
    with fwd.dual_level():
        c = _spectra64(fwd.make_dual(th, e), *args)
        v, t = fwd.unpack_dual(c)
        return v.clone(), t.clone()


def exact(case, seed):
    k = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def dbl(x):
        return torch.as_tensor(x, device=dev).to(torch.float64)

    if k in ("sparse", "dense", "cholesky"):
        cov, data, mu, rng = _gaussian_problem(case, seed)
        if k == "sparse":
            blocks = dbl(np.ascontiguousarray(np.transpose(cov, (2, 0, 1))))
            low = torch.linalg.cholesky(blocks)
            r = dbl(data).reshape(1, *mu.shape[1:]) - dbl(mu)  # [B, P, L]
            z = torch.linalg.solve_triangular(low, r.permute(2, 1, 0).contiguous(), upper=False)
            logdet = 2.0 * torch.diagonal(low, dim1=1, dim2=2).log().sum()
            return (-0.5 * ((z ** 2).sum((0, 1)) - logdet)).cpu().numpy()
        low = torch.linalg.cholesky(dbl(_dense_cov(cov, rng)))
        logdet = 2.0 * low.diagonal().log().sum()
        if k == "cholesky":
            return low, float(logdet)
        r = dbl(data) - dbl(mu).reshape(mu.shape[0], -1)
        z = torch.linalg.solve_triangular(low, r.T.contiguous(), upper=False)
        return (-0.5 * ((z ** 2).sum(0) - logdet)).cpu().numpy()
    if k == "serve":
        reqs = _requests(case, seed)
        m = _Model(dbl(np.array([q["cosmo"] for q in reqs])))
        out = []
        for i, q in enumerate(reqs):
            wl, nc = [t for t in q["tracers"] if t < 5], [t - 5 for t in q["tracers"] if t >= 5]
            out.append(m.spectra(slice(i, i + 1), dbl(q["ell"]), wl, nc, q["n_z"]).reshape(-1))
        return torch.cat(out).cpu().numpy()
    params = _cosmologies(seed, case.get("batch", 1))
    args = (dbl(_ell(case)), list(range(case["wl"])), list(range(case["nc"])), case["n_z"])
    if k == "single":
        return _spectra64(dbl(params), *args)[0].cpu().numpy()
    if k == "batch":
        return _spectra64(dbl(params), *args)
    if k == "jacobian":
        return torch.stack([_tangent64(dbl(params), d, *args)[1] for d in range(7)], -1).cpu().numpy()
    # the gradients are taken at the float32 parameters that the program holds
    params[:, FREE] = params[:, FREE].astype(np.float32)
    cbar = dbl(_cotangent(case, seed, params.shape[0]))
    grad = []
    for d in range(7):
        cl, dot = _tangent64(dbl(params), d, *args)
        grad.append((cbar * dot).sum((1, 2)))
    grad = torch.stack(grad, 1)
    return (cl[0], grad[0]) if k == "grad_one" else (cl, grad)
