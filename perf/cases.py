"""Workloads of the ISDF-Lanczos GW path, each as a user's program runs it.

A case is one call, or one short sequence of calls, of the package's public
entry points (``nanogw_amd.lanczos.IsdfContext``, ``nanogw_amd.batch.GwBatch``)
on seeded synthetic inputs.  The sizes are those of ``synth.CONFIGS`` (c1: 480
points, 8 x 56 pairs; c2: 2000 points, 40 x 400; c3: 5000 points, 100 x 1500)
and of the batched molecules (``synth.c4_specs``: nv 8..60, nc = 10 nv, 12 nv
points, 16 states), with Lanczos runs cut to a few steps: every step costs the
same.  Odd nv and nc are the rule for the batched molecules, not the exception.

Operators: Gaussian-envelope Hermite orbitals at random points (as
``synth.orbitals``), orbital energies drawn as ``synth.energies`` does, and a
positive definite softened Coulomb kernel for M, scaled so that the Casida
operator's spectrum stays inside the interval of the square-root fit.
"""
import math

import numpy as np
import torch

from nanogw_amd.batch import GwBatch
from nanogw_amd.lanczos import IsdfContext

NPOLY = 12          # the driver's default degree of the square-root polynomial
RYD = 13.60569193   # eV
DELTAE, ECUTS = 4.0, 0.02   # energy_range and resolution (Ry) of the benchmark workloads
RIDGE = 1e-6        # ridge of the zeta fit, relative to tr(A) / n_intp
F64 = torch.float64


def listed():
    return [
        # The drop-in of NanoGW's single-vector routines: one FP64 vector.
        # The smallest molecule (launches and latency count) ...
        {"name": "apply_f64_one_c1", "kind": "apply", "prec": "f64", "nmu": 480, "nv": 8, "nc": 56, "nvec": 1, "tda": False},
        # ... and the largest (one read of M, two GEMM-like passes with 100 columns).
        {"name": "apply_f64_one_c3", "kind": "apply", "prec": "f64", "nmu": 5000, "nv": 100, "nc": 1500, "nvec": 1, "tda": False},
        # The BLOCK operator of the parity path, one 200-column call (the
        # column count per call of the FP64 reference runs) of the middle molecule.
        {"name": "apply_f64_block_c2", "kind": "apply", "prec": "f64", "nmu": 2000, "nv": 40, "nc": 400, "nvec": 200, "tda": False},
        # A batched molecule's operator, eight states' columns, TDA; nv is odd.
        {"name": "apply_bf16x3_nv37_tda", "kind": "apply", "prec": "bf16x3", "nmu": 444, "nv": 37, "nc": 370, "nvec": 3256, "tda": True},
        # The mixed-precision operator on all bands of one state of the largest molecule.
        {"name": "apply_f16_c3", "kind": "apply", "prec": "f16", "nmu": 5000, "nv": 100, "nc": 1500, "nvec": 1600, "tda": False},
        # The BLOCK Lanczos drop-in on host vectors, ragged in every size.
        {"name": "lanczos_f64_ragged", "kind": "lanczos", "prec": "f64", "nmu": 731, "nv": 13, "nc": 129, "nvec": 37, "niter": 12, "nz": 101, "tda": False},
        # Sigma_c of the four states around the gap of the smallest molecule: the parity path's whole call.
        {"name": "sigma_f64_c1", "kind": "sigma", "prec": "f64", "nmu": 480, "nv": 8, "nc": 56, "nqp": 4, "niter": 16, "nen": 200, "tda": False},
        # Batched serving: three molecules of the 64-molecule workload, 16
        # states each, admitted together, stepped to the end in one graph.
        {"name": "serve_bf16x3_small", "kind": "serve", "prec": "bf16x3", "nvs": "9,23,38", "ncr": 10, "nmur": 12, "nqp": 16, "niter": 4, "nen": 200},
        # Served mixed precision on the largest molecule (the headline's
        # path): one state, all 1600 bands in every launch.
        {"name": "serve_f16_c3", "kind": "serve", "prec": "f16", "nvs": "100", "ncr": 15, "nmur": 50, "nqp": 1, "niter": 2, "nen": 200},
        # Coulomb kernel M from a device zeta, the middle molecule's grid (114^3 box).
        {"name": "vbuild_c2", "kind": "vbuild", "radius": 10.0, "h": 0.35, "nmu": 2000},
        # Interpolation vectors of the same molecule.
        {"name": "zeta_c2", "kind": "zeta", "radius": 10.0, "h": 0.35, "nmu": 2000, "nv": 40, "nc": 400},
        # The QP roots of a batch's states from their Sigma_c tables.
        {"name": "newton_64", "kind": "newton", "nqp": 64, "nen": 200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["one", "one", "f64", "low", "low", "lanczos", "sigma", "serve", "serve", "vbuild", "zeta", "newton"])
    tda = rng.random() < 0.25
    if kind == "one":
        nv = _log_int(rng, 5, 100)
        return {"kind": "apply", "prec": "f64", "nmu": rng.randint(12 * nv, 50 * nv), "nv": nv, "nc": rng.randint(7 * nv, 15 * nv), "nvec": 1, "tda": tda}
    if kind == "f64":
        nv = _log_int(rng, 6, 40)
        return {"kind": "apply", "prec": "f64", "nmu": rng.randint(12 * nv, 50 * nv), "nv": nv, "nc": rng.randint(7 * nv, 10 * nv), "nvec": _log_int(rng, 8, 200), "tda": tda}
    if kind == "low":
        nv = _log_int(rng, 8, 60)
        return {"kind": "apply", "prec": rng.choice(["bf16x3", "f16"]), "nmu": rng.randint(12 * nv, 50 * nv), "nv": nv, "nc": rng.randint(8 * nv, 12 * nv), "nvec": _log_int(rng, 60, 3000), "tda": tda}
    if kind == "lanczos":
        nv = rng.randint(5, 24)
        return {"kind": "lanczos", "prec": "f64", "nmu": rng.randint(12 * nv, 50 * nv), "nv": nv, "nc": rng.randint(7 * nv, 12 * nv), "nvec": rng.randint(3, 80), "niter": rng.randint(6, 12), "nz": rng.randint(50, 201), "tda": tda}
    if kind == "sigma":
        nv = rng.randint(5, 14)
        return {"kind": "sigma", "prec": "f64", "nmu": rng.randint(20 * nv, 60 * nv), "nv": nv, "nc": rng.randint(6 * nv, 10 * nv), "nqp": rng.randint(1, 4), "niter": rng.randint(8, 16), "nen": rng.randint(60, 200), "tda": tda}
    if kind == "serve":
        n = rng.randint(1, 4)
        return {"kind": "serve", "prec": rng.choice(["bf16x3", "f16"]), "nvs": ",".join(str(rng.randint(8, 44)) for _ in range(n)), "ncr": 10, "nmur": 12, "nqp": rng.randint(2, 16), "niter": rng.randint(2, 5), "nen": rng.randint(100, 200)}
    if kind == "vbuild":
        return {"kind": "vbuild", "radius": round(rng.uniform(6.0, 10.0), 2), "h": round(rng.uniform(0.36, 0.48), 3), "nmu": _log_int(rng, 100, 1600)}
    if kind == "zeta":
        nv = rng.randint(8, 36)
        return {"kind": "zeta", "radius": round(rng.uniform(6.0, 10.0), 2), "h": round(rng.uniform(0.36, 0.48), 3), "nmu": rng.randint(12 * nv, 48 * nv), "nv": nv, "nc": rng.randint(7 * nv, 10 * nv)}
    return {"kind": "newton", "nqp": _log_int(rng, 1, 1000), "nen": rng.randint(50, 400)}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _orbitals(pts, nb, g):
    """Gaussian envelope (2.5 bohr) x random Hermite products, one column per band."""
    dev = pts.device
    span = float(pts.norm(dim=1).max())
    centre = torch.randn(nb, 3, generator=g, device=dev, dtype=F64)
    centre = centre / centre.norm(dim=1, keepdim=True) * torch.rand(nb, 1, generator=g, device=dev, dtype=F64) * (0.5 * span)
    coef = torch.randn(nb, 6, generator=g, device=dev, dtype=F64)
    out = torch.empty(nb, pts.shape[0], device=dev, dtype=F64)
    for b0 in range(0, nb, 64):
        u = (pts[None, :, :] - centre[b0:b0 + 64, None, :]) / 2.5
        x, y, z = u[..., 0], u[..., 1], u[..., 2]
        c = coef[b0:b0 + 64, :, None]
        poly = c[:, 0] + 2 * c[:, 1] * x + 2 * c[:, 2] * y + 2 * c[:, 3] * z + c[:, 4] * (4 * x * y) + c[:, 5] * (4 * z * z - 2)
        out[b0:b0 + 64] = poly * torch.exp(-0.5 * (u * u).sum(-1))
    return out / out.norm(dim=1, keepdim=True)   # (nb, points)


def _energies(nv, nc, rng):
    ev = np.sort(rng.uniform(-0.9, -0.25, nv))
    ec = np.sort(rng.uniform(-0.15, 2.0, nc))
    return 2.0 * np.concatenate([ev, ec])


def _operator(nmu, nv, nc, seed):
    """psi (nband, nmu) and M (nmu, nmu) on the GPU, energies (Ry)."""
    g, rng = _gen(seed), np.random.default_rng(seed)
    nb = nv + nc
    pts = torch.randn(nmu, 3, generator=g, device="cuda", dtype=F64) * (2.0 + 0.02 * nv)
    psi = _orbitals(pts, nb, g)
    e1 = _energies(nv, nc, rng)
    d2 = ((pts[:, None, :] - pts[None, :, :]) ** 2).sum(-1) if nmu <= 2500 else torch.cdist(pts, pts) ** 2
    m = 1.0 / torch.sqrt(d2 + 0.5)
    m = 0.5 * (m + m.T)
    # scale M: largest eigenvalue of 4 R^1/2 C^T M C R^1/2 at a tenth of e_max
    e = torch.as_tensor(e1, device="cuda")
    s = (e[nv:, None] - e[None, :nv]).sqrt()   # (nc, nv)
    x = torch.rand(nc, nv, generator=g, device="cuda", dtype=F64)
    lam = 1.0
    for _ in range(8):
        x = x / x.norm()
        t = (((s * x).T.contiguous() @ psi[nv:]) * psi[:nv]).sum(0)
        u = m @ t
        x = s * (psi[nv:] @ (psi[:nv] * u).T.contiguous())
        lam = float(x.norm())
    emax = 1.25 * (e1[-1] - e1[0]) ** 2
    m *= 0.1 * emax / (4.0 * lam)
    return psi, m, e1


def _polynomial(e1, nv):
    """Degree-12 approximation of sqrt on the driver's interval, highest order first."""
    lo, hi = (e1[nv] - e1[nv - 1]) ** 2 / 1.25, 1.25 * (e1[-1] - e1[0]) ** 2
    k = np.arange(64)
    t = np.cos(np.pi * (k + 0.5) / 64)
    c = np.polynomial.chebyshev.chebfit(t, np.sqrt(0.5 * (hi - lo) * t + 0.5 * (hi + lo)), NPOLY)
    p = np.polynomial.Polynomial(np.polynomial.chebyshev.cheb2poly(c))
    return p(np.polynomial.Polynomial([-(hi + lo) / (hi - lo), 2.0 / (hi - lo)])).coef[::-1].copy()


def _host(psi, m):
    """(n_intp, nband) and (n_intp, n_intp) Fortran-ordered host arrays."""
    return psi.cpu().numpy().T, m.cpu().numpy().T


def _vectors(case, seed):
    """Normalised vectors, (nvec, ncv) on the GPU: columns of the transition space."""
    g = _gen(seed + 1_000_003)
    ncv = case["nv"] * case["nc"]
    x = torch.empty(case["nvec"], ncv, device="cuda", dtype=F64)
    for b in range(0, case["nvec"], 256):
        x[b:b + 256].normal_(generator=g)
    x /= x.norm(dim=1, keepdim=True)
    return x


def _qp(nv, nb, nqp):
    lo = max(0, min(nv - (nqp + 1) // 2, nb - nqp))
    return list(range(lo, lo + nqp))


def _systems(case):
    return [(case["nmur"] * nv, nv, case["ncr"] * nv) for nv in map(int, case["nvs"].split(","))]


def _grid(case):
    """Grid points of the sphere, FFT box and truncation radius (r_max rules of the wave-function reader)."""
    h, radius = case["h"], case["radius"]
    n = int(radius / h) + 1
    ax = np.arange(-n, n + 1)
    z, y, x = np.meshgrid(ax, ax, ax, indexing="ij")
    pts = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    g = np.ascontiguousarray(pts[((pts * h) ** 2).sum(1) <= radius * radius + 1e-12].astype(np.int32))
    rmax = float(np.sqrt(((g * h) ** 2).sum(1).max()))
    nf = int(np.rint(4.0 * rmax / h))
    nf += nf % 2
    return g, (nf, nf, nf), 2.0 * rmax


def _points(ngrid, n, seed):
    return np.sort(np.random.default_rng(seed).choice(ngrid, n, replace=False)).astype(np.int64)


def _zeta_inputs(case, seed):
    """Localised interpolation vectors (n_intp, ngrid) on the GPU."""
    gidx, nfft, trunc = _grid(case)
    g = _gen(seed)
    r = torch.as_tensor(gidx, device="cuda", dtype=F64) * case["h"]
    c = r[torch.as_tensor(_points(len(gidx), case["nmu"], seed), device="cuda")]
    zeta = torch.empty(case["nmu"], len(gidx), device="cuda", dtype=F64)
    for k in range(0, case["nmu"], 64):
        d2 = ((r[None] - c[k:k + 64, None, :]) ** 2).sum(-1)
        noise = torch.randn(d2.shape, generator=g, device="cuda", dtype=F64)
        zeta[k:k + 64] = torch.exp(-d2 / 1.5) * (1.0 + 0.05 * noise)
    return gidx, nfft, trunc, zeta


def _fit_inputs(case, seed):
    """Grid orbitals (nband, ngrid) on the GPU and the interpolation points."""
    gidx, _, _ = _grid(case)
    r = torch.as_tensor(gidx, device="cuda", dtype=F64) * case["h"]
    psi = _orbitals(r, case["nv"] + case["nc"], _gen(seed))
    return psi, _points(len(gidx), case["nmu"], seed)


def _newton_inputs(case, seed):
    """Sigma_c tables (eV) as sums over broadened poles, and the other terms of the QP equation."""
    rng = np.random.default_rng(seed)
    nqp, nen = case["nqp"], case["nen"]
    width = DELTAE * RYD
    en = rng.uniform(-16.0, 4.0, nqp)
    e = en[None, :] - 0.5 * width + width / (nen - 1) * np.arange(nen)[:, None]
    sig = np.zeros((nen, nqp), np.complex128, order="F")
    for _ in range(24):
        pole = en + rng.choice([-1.0, 1.0], nqp) * rng.uniform(8.0, 40.0, nqp)
        sig += rng.uniform(0.2, 3.0, nqp) / (e - pole[None, :] + 1j * np.where(pole > en, 1.0, -1.0) * rng.uniform(0.5, 3.0, nqp))
    sigx = rng.uniform(-18.0, -4.0, nqp)
    return sig, width, en, en.copy(), sigx, sigx + rng.uniform(-2.0, 2.0, nqp)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "newton":
        return {"kind": kind, "ctx": IsdfContext(0), "args": _newton_inputs(case, seed)}
    if kind == "vbuild":
        gidx, nfft, trunc, zeta = _zeta_inputs(case, seed)
        return {"kind": kind, "ctx": IsdfContext(0), "case": case, "grid": (gidx, nfft, trunc), "zeta": zeta}
    if kind == "zeta":
        psi, intp = _fit_inputs(case, seed)
        return {"kind": kind, "ctx": IsdfContext(0), "case": case, "psi": psi, "intp": intp, "out": torch.empty(case["nmu"], psi.shape[1], device="cuda", dtype=F64)}
    if kind == "serve":
        ctx = IsdfContext(0)
        ctx.set_precision(case["prec"])
        batch = GwBatch(ctx)
        jobs = []
        for k, (nmu, nv, nc) in enumerate(_systems(case)):
            psi, m, e1 = _operator(nmu, nv, nc, seed + 7919 * k)
            jobs.append((batch.add_system(*_host(psi, m), e1, nv), _qp(nv, nv + nc, case["nqp"]), _polynomial(e1, nv)))
        return {"kind": kind, "ctx": ctx, "batch": batch, "jobs": jobs, "case": case}
    psi, m, e1 = _operator(case["nmu"], case["nv"], case["nc"], seed)
    ctx = IsdfContext(0)
    ctx.set_isdf(*_host(psi, m), e1, case["nv"])
    ctx.set_precision(case["prec"])
    state = {"kind": kind, "ctx": ctx, "case": case}
    if kind == "apply":
        state["x"] = _vectors(case, seed)
        state["y"] = torch.empty_like(state["x"])
        torch.cuda.synchronize()   # the context works on its own stream
    elif kind == "lanczos":
        v = _vectors(case, seed)
        state["v0"] = (3.0 * v).cpu().numpy().T
        state["zz"] = _lanczos_grid(case, e1)
        state["poly"] = _polynomial(e1, case["nv"])
    else:
        state["qp"] = _qp(case["nv"], case["nv"] + case["nc"], case["nqp"])
        state["poly"] = _polynomial(e1, case["nv"])
    return state


def _lanczos_grid(case, e1):
    """Complex energies of each column: a window of excitation energies with the resolution's width."""
    z = np.linspace(0.1, e1[-1] - e1[0], case["nz"]) + 1j * ECUTS
    return np.asfortranarray(np.repeat(z[:, None], case["nvec"], axis=1))


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "apply":
        c, x, y = state["case"], state["x"], state["y"]
        ctx.matvec_dev(x.data_ptr(), y.data_ptr(), x.shape[1], x.shape[0], c["tda"])
        ctx.synchronize()   # the caller's own stream reads y next
        return y
    if kind == "lanczos":
        c = state["case"]
        return ctx.lanczos_spectra_isdf_BLOCK(state["v0"], np.full(c["nvec"], 3.0), state["zz"], c["niter"], state["poly"], c["tda"])
    if kind == "sigma":
        c = state["case"]
        return ctx.calculate_sigma_lanczos(state["qp"], c["nen"], DELTAE, ECUTS, c["niter"], state["poly"], c["tda"])
    if kind == "serve":
        c, batch = state["case"], state["batch"]
        rids = [batch.submit(sid, qp, c["nen"], DELTAE, ECUTS, c["niter"], poly) for sid, qp, poly in state["jobs"]]
        batch.step(c["niter"])
        out = [batch.result(rid, c["nen"], len(job[1])) for rid, job in zip(rids, state["jobs"])]
        for rid in rids:
            batch.release(rid)
        return out
    if kind == "vbuild":
        c, zeta = state["case"], state["zeta"]
        gidx, nfft, trunc = state["grid"]
        return ctx.isdf_coulomb_kernel_dev(zeta.data_ptr(), zeta.shape[1], zeta.shape[1], zeta.shape[0], gidx, nfft, c["h"], trunc)
    if kind == "zeta":
        c, psi, out = state["case"], state["psi"], state["out"]
        used_lu = ctx.isdf_zeta_dev(psi.data_ptr(), psi.shape[1], psi.shape[1], psi.shape[0], c["nv"], state["intp"], RIDGE, out.data_ptr(), psi.shape[1])
        return {"zeta": out, "used_lu": used_lu}
    return ctx.qp_newton(*state["args"])


# ---------------------------------------------------------------- counts
def _matvec_flops(nmu, nv, nc):
    return 4.0 * nmu * nv * nc + 2.0 * nmu * nmu


def _sigma_work(nmu, nv, nc, nqp, niter, nen):
    """One state: P vectors, then niter steps of NPOLY applications, for every band."""
    cols = nqp * (nv + nc)
    flops = cols * (niter * NPOLY * _matvec_flops(nmu, nv, nc) + 2.0 * nmu * nmu + 2.0 * nmu * nv * nc)
    return 8.0 * (nmu * (nv + nc) + nmu * nmu) + 16.0 * nen * nqp, flops


def work(case):
    kind = case["kind"]
    if kind == "newton":
        n = case["nqp"] * case["nen"]
        return {"bytes": 16.0 * n + 80.0 * case["nqp"], "flops": 60.0 * n}
    if kind in ("vbuild", "zeta"):
        gidx, nfft, _ = _grid(case)
        ng, n, box = float(len(gidx)), float(case["nmu"]), float(np.prod(nfft))
        if kind == "vbuild":   # two real transforms per vector, half of the symmetric product
            return {"bytes": 8.0 * (ng * n + n * n), "flops": n * n * ng + n * 5.0 * box * math.log2(box)}
        nb, nv = case["nv"] + case["nc"], case["nv"]
        return {"bytes": 8.0 * (ng * nb + ng * n), "flops": 2.0 * ng * n * n + 2.0 * ng * n * (nb + nv) + n ** 3}
    if kind == "serve":
        parts = [_sigma_work(*s, case["nqp"], case["niter"], case["nen"]) for s in _systems(case)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    nmu, nv, nc = case["nmu"], case["nv"], case["nc"]
    if kind == "sigma":
        b, f = _sigma_work(nmu, nv, nc, case["nqp"], case["niter"], case["nen"])
        return {"bytes": b, "flops": f}
    op = 8.0 * (nmu * (nv + nc) + nmu * nmu)
    ncv, b = float(nv * nc), case["nvec"]
    if kind == "apply":
        return {"bytes": op + 16.0 * ncv * b, "flops": b * _matvec_flops(nmu, nv, nc)}
    return {"bytes": op + 8.0 * ncv * b + 32.0 * case["nz"] * b, "flops": b * case["niter"] * NPOLY * _matvec_flops(nmu, nv, nc)}


# ---------------------------------------------------------------- 64-bit values
def _apply64(psi, m, e, nv, x, tda):
    """y (B, ncv) = H x in plain torch."""
    nb, nmu = psi.shape
    nc = nb - nv
    r = (e[nv:, None] - e[None, :nv]).reshape(-1)   # pair index v + nv c
    s = torch.ones_like(r) if tda else r.sqrt()
    y = torch.empty_like(x)
    step = max(1, int(4e8 // (8 * nv * nmu)))
    for b0 in range(0, x.shape[0], step):
        xb = s * x[b0:b0 + step]
        n = xb.shape[0]
        xt = xb.reshape(n, nc, nv).transpose(1, 2).contiguous().reshape(n * nv, nc)
        t = ((xt @ psi[nv:]).reshape(n, nv, nmu) * psi[None, :nv]).sum(1)
        w = (psi[None, :nv] * (t @ m)[:, None, :]).reshape(n * nv, nmu)
        g = (w @ psi[nv:].T.contiguous()).reshape(n, nv, nc).transpose(1, 2).reshape(n, nc * nv)
        y[b0:b0 + step] = r * x[b0:b0 + step] + 2.0 * g if tda else r * r * x[b0:b0 + step] + 4.0 * s * g
    return y


def _lanczos64(op, nv, q, poly, niter, tda):
    """Recurrence coefficients (B, niter) of the normalised columns q."""
    psi, m, e = op
    a, b = [], [torch.ones(q.shape[0], device=q.device, dtype=F64)]

    def p(v):
        out = poly[0] * _apply64(psi, m, e, nv, v, tda) + poly[1] * v
        for c in poly[2:]:
            out = _apply64(psi, m, e, nv, out, tda) + c * v
        return out

    w = p(q)
    for k in range(niter):
        al = (w * q).sum(1)
        a.append(al)
        if k == niter - 1:
            break
        w = w - al[:, None] * q
        be = w.norm(dim=1)
        b.append(be)
        q, w = w / be[:, None], -be[:, None] * q
        w = w + p(q)
    return torch.stack(a, 1), torch.stack(b, 1)


def _spectra64(a, b, zz):
    """Continued fraction at zz (nz, B)."""
    s = torch.zeros_like(zz)
    for j in reversed(range(a.shape[1])):
        en = torch.ones_like(b[:, 0]) if j == 0 else b[:, j] ** 2
        s = en / (zz - a[:, j] - s)
    return s


def _sigma64(psi, m, e1, nv, qp, poly, niter, nen, tda):
    """Sigma_c (nen, nqp) of the Lanczos driver."""
    e = torch.as_tensor(e1, device="cuda")
    nb, nc = psi.shape[0], psi.shape[0] - nv
    s = torch.ones(nc * nv, device="cuda", dtype=F64) if tda else (e[nv:, None] - e[None, :nv]).sqrt().reshape(-1)
    out = np.zeros((nen, len(qp)), np.complex128, order="F")
    for iq, mb in enumerate(qp):
        total = torch.zeros(nen, device="cuda", dtype=torch.complex128)
        for n0 in range(0, nb, 400):
            bands = torch.arange(n0, min(nb, n0 + 400), device="cuda")
            u = (psi[mb][None] * psi[bands]) @ m
            pv = torch.empty(len(bands), nc * nv, device="cuda", dtype=F64)
            for k in range(0, len(bands), 100):
                w = (psi[None, :nv] * u[k:k + 100, None, :]).reshape(-1, psi.shape[1])
                g = (w @ psi[nv:].T.contiguous()).reshape(-1, nv, nc).transpose(1, 2)
                pv[k:k + 100] = s * g.reshape(-1, nc * nv)
            pn = pv.norm(dim=1)
            a, b = _lanczos64((psi, m, e), nv, pv / pn[:, None], poly, niter, tda)
            z = DELTAE / (nen - 1) * torch.arange(nen, device="cuda", dtype=F64) + (e1[mb] - 0.5 * DELTAE)
            sign = torch.where(bands < nv, -1.0, 1.0).to(F64)
            zeta = torch.complex(sign[None, :] * (z[:, None] - e[bands][None, :]), torch.full((nen, len(bands)), ECUTS, device="cuda", dtype=F64))
            sp = _spectra64(a, b, zeta)
            if tda:
                inc = sp * sign * float(np.float32(2.0) ** np.float32(0.5)) * pn ** 2
            else:
                s0 = _spectra64(a, b, torch.zeros(1, len(bands), device="cuda", dtype=torch.complex128))
                inc = 2.0 * pn ** 2 / (sign * zeta) * (sp - s0)
            total += inc.sum(1)
        out[:, iq] = total.cpu().numpy()
    return out


def _spline64(x, y, at):
    """Cubic spline with clamped slopes through columns y(n, q) at x(n, q): values at `at` (q)."""
    n = x.shape[0]
    slope0, slope1 = (y[1] - y[0]) / (x[1] - x[0]), (y[-1] - y[-2]) / (x[-1] - x[-2])
    x, y = x[1:-1], y[1:-1]
    n -= 2
    y2, u = np.zeros_like(y), np.zeros_like(y)
    y2[0] = -0.5
    u[0] = 3.0 / (x[1] - x[0]) * ((y[1] - y[0]) / (x[1] - x[0]) - slope0)
    for i in range(1, n - 1):
        sg = (x[i] - x[i - 1]) / (x[i + 1] - x[i - 1])
        p = sg * y2[i - 1] + 2.0
        y2[i] = (sg - 1.0) / p
        u[i] = (6.0 * ((y[i + 1] - y[i]) / (x[i + 1] - x[i]) - (y[i] - y[i - 1]) / (x[i] - x[i - 1])) / (x[i + 1] - x[i - 1]) - sg * u[i - 1]) / p
    un = 3.0 / (x[-1] - x[-2]) * (slope1 - (y[-1] - y[-2]) / (x[-1] - x[-2]))
    y2[-1] = (un - 0.5 * u[-2]) / (0.5 * y2[-2] + 1.0)
    for k in range(n - 2, -1, -1):
        y2[k] = y2[k] * y2[k + 1] + u[k]
    q = np.arange(x.shape[1])

    def value(t):
        hi = np.clip((x <= t[None, :]).sum(0), 1, n - 1)
        lo = hi - 1
        h = x[hi, q] - x[lo, q]
        a, b = (x[hi, q] - t) / h, (t - x[lo, q]) / h
        return a * y[lo, q] + b * y[hi, q] + ((a ** 3 - a) * y2[lo, q] + (b ** 3 - b) * y2[hi, q]) * h * h / 6.0

    return value(at), (value(at + 0.01) - value(at - 0.01)) / 0.02


def _newton64(sig, width, edft, en0, sigx, vxc):
    nen, nqp = sig.shape
    x = en0[None, :] - 0.5 * width + width / (nen - 1) * np.arange(nen)[:, None]
    f = sigx + sig.real - vxc + edft - x
    e, done = en0.copy(), np.zeros(nqp, bool)
    for _ in range(20):
        fx, df = _spline64(x, f, e)
        dx = np.where(done, 0.0, fx / df)
        e = e - dx
        done |= np.abs(dx) < 0.01
    slope = _spline64(x, f, e)[1]
    s0 = _spline64(x, f, edft)[0] + vxc
    return {"eqp": e, "zfac": -1.0 / slope, "sigma0": s0 + 0j, "imsig": _spline64(x, np.ascontiguousarray(sig.imag), e)[0], "ierr": None}


def _coulomb64(case, seed):
    gidx, nfft, trunc, zeta = _zeta_inputs(case, seed)
    n, h = nfft[0], case["h"]
    k = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=F64) * (2.0 * math.pi / (n * h))
    kr = torch.arange(n // 2 + 1, device="cuda", dtype=F64) * (2.0 * math.pi / (n * h))
    g2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + kr[None, None, :] ** 2
    v = torch.where(g2 < 1e-12, torch.full_like(g2, 0.5 * trunc * trunc), (1.0 - torch.cos(trunc * g2.sqrt())) / g2.clamp_min(1e-12)) * (8.0 * math.pi)
    at = torch.as_tensor(np.mod(gidx, n), device="cuda", dtype=torch.long)
    flat = (at[:, 2] * n + at[:, 1]) * n + at[:, 0]
    vz = torch.empty_like(zeta)
    for c in range(zeta.shape[0]):
        box = torch.zeros(n ** 3, device="cuda", dtype=F64)
        box[flat] = zeta[c]
        vz[c] = torch.fft.irfftn(torch.fft.rfftn(box.reshape(n, n, n)) * v, s=(n, n, n)).reshape(-1)[flat]
    return np.asfortranarray(((zeta @ vz.T.contiguous()) / h ** 3).cpu().numpy())


def _zeta64(case, seed):
    psi, intp = _fit_inputs(case, seed)
    pi = psi[:, torch.as_tensor(intp, device="cuda")].contiguous()
    nv = case["nv"]
    a = ((pi[:nv].T.contiguous() @ pi[:nv]) * (pi.T.contiguous() @ pi)).cpu().numpy()
    a += RIDGE * np.trace(a) / len(a) * np.eye(len(a))
    b = (pi[:nv].T.contiguous() @ psi[:nv]) * (pi.T.contiguous() @ psi)
    return {"zeta": np.linalg.solve(a, b.cpu().numpy()), "used_lu": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "newton":
        return _newton64(*_newton_inputs(case, seed))
    if kind == "vbuild":
        return _coulomb64(case, seed)
    if kind == "zeta":
        return _zeta64(case, seed)
    if kind == "serve":
        out = []
        for k, (nmu, nv, nc) in enumerate(_systems(case)):
            psi, m, e1 = _operator(nmu, nv, nc, seed + 7919 * k)
            out.append(_sigma64(psi, m, e1, nv, _qp(nv, nv + nc, case["nqp"]), _polynomial(e1, nv), case["niter"], case["nen"], False))
        return out
    nv = case["nv"]
    psi, m, e1 = _operator(case["nmu"], nv, case["nc"], seed)
    e = torch.as_tensor(e1, device="cuda")
    if kind == "apply":
        return _apply64(psi, m, e, nv, _vectors(case, seed), case["tda"])
    if kind == "sigma":
        return _sigma64(psi, m, e1, nv, _qp(nv, nv + case["nc"], case["nqp"]), _polynomial(e1, nv), case["niter"], case["nen"], case["tda"])
    a, b = _lanczos64((psi, m, e), nv, _vectors(case, seed), _polynomial(e1, nv), case["niter"], case["tda"])
    zz = torch.as_tensor(_lanczos_grid(case, e1), device="cuda")
    return _spectra64(a, b, zz).cpu().numpy(), a.cpu().numpy().T, b.cpu().numpy().T
