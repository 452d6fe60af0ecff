"""The work whose speed is measured: what a user has the framework do, over the
sizes, directions and options it is used with.

Every case is one call (or one short chain of calls) of the public entry
points: the tomography and ptychography operators, the two CG subproblems, an
ADMM run, and the warm-start network's forward and backward pass.  Inputs are
made from a seed alone with plain torch: projections of random balls in closed
form, far-field intensities with Poisson noise, and iterates part of the way
between the initial guess and the object, as a reconstruction holds them
between iterations.  ``exact`` restates each call in 64 bits with plain torch.
"""
import math

import numpy as np
import torch

from ptychotomo_amd import Solver, gaussian_probe, jittered_raster, make_theta
from ptychotomo_amd.unet import UNet3D

VOXEL, ENERGY, ALPHA = 1e-6, 8.8, 3e-7          # [cm], [keV], TV weight of the demo
RHO, TAU = 0.5, 0.5
WAVE = 2 * math.pi / (2 * math.pi * 6.58211928e-19 * 299792458e+2 / ENERGY)
C64, C128, F32, F64 = torch.complex64, torch.complex128, torch.float32, torch.float64


def _smooth(m):
    for f in (2, 3, 5):
        while m % f == 0:
            m //= f
    return m == 1


# object sizes the tomography accepts, up to the largest workload's
SIZES = [n for n in range(32, 513, 4) if _smooth(3 * n // 2)]

# (output, input) channels of the warm-start network's layers
NET = dict(e1a=(16, 2), e1b=(16, 16), e2a=(32, 16), e2b=(32, 32), bna=(64, 32), bnb=(64, 64),
           d2a=(32, 96), d2b=(32, 32), d1a=(16, 48), d1b=(16, 16), head=(2, 16))


def listed():
    return [
        # a thin slab of a small object: the smallest call, launches and latency
        dict(name="tomo_fwd_32", kind="tomo_fwd", n=32, nz=8, ntheta=48),
        # an object whose size is no power of two, odd slab and angle counts
        dict(name="tomo_adj_180", kind="tomo_adj", n=180, nz=21, ntheta=201),
        # the production volume, projected and backprojected once each per CG step
        dict(name="tomo_fwd_256", kind="tomo_fwd", n=256, nz=256, ntheta=384),
        dict(name="tomo_adj_256", kind="tomo_adj", n=256, nz=256, ntheta=384),
        # simulating a data set: far-field intensities of all angles
        dict(name="ptycho_fwd_128", kind="ptycho_fwd", n=128, nz=128, ntheta=192, det=16,
             nprb=16, step=4, jitter=1.0, photons=1e3),
        # backpropagating far fields of the large scan's 32 x 32 frames
        dict(name="ptycho_adj_256_det32", kind="ptycho_adj", n=256, nz=256, ntheta=24, det=32,
             nprb=32, step=8, jitter=2.0, photons=1e2),
        # one angle chunk of the 512^3 workload's ptychography subproblem
        dict(name="cg_ptycho_512_det32", kind="cg_ptycho", n=512, nz=512, ntheta=32, ptheta=32,
             det=32, nprb=32, step=8, jitter=2.0, photons=1e2, model="poisson", piter=4),
        # the demo script's scan: 64 x 64 detector, 16 x 16 probe, step 8
        dict(name="cg_ptycho_128_det64", kind="cg_ptycho", n=128, nz=128, ntheta=64, ptheta=32,
             det=64, nprb=16, step=8, jitter=1.0, photons=1e3, model="gaussian", piter=4),
        # the tomography subproblem at the demo script's size
        dict(name="cg_tomo_128", kind="cg_tomo", n=128, nz=128, ntheta=192, titer=4),
        # a steady-state ADMM iteration: the small workload, where launches count,
        # and the production one.  One iteration, since rounding travels: after two
        # the 64-bit twin is already 2e-5 away in psi and 3e-4 in the dual lamd
        dict(name="admm_64", kind="admm", n=64, nz=64, ntheta=96, ptheta=32, det=16, nprb=16,
             step=4, jitter=1.0, photons=1e3, model="poisson", piter=4, titer=4, niter=1),
        dict(name="admm_256", kind="admm", n=256, nz=256, ntheta=384, ptheta=32, det=16, nprb=16,
             step=4, jitter=1.0, photons=1e3, model="poisson", piter=4, titer=4, niter=1),
        # one training pass of the warm-start network: forward, loss, all gradients
        dict(name="unet_grad_64", kind="unet", nz=64, ny=64, nx=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tomo_fwd", "tomo_adj", "ptycho_fwd", "ptycho_adj", "cg_ptycho", "cg_tomo",
                       "admm", "unet"])
    if kind == "unet":
        return dict(kind=kind, **{k: 4 * _log(rng, 4, 20) for k in ("nz", "ny", "nx")})
    hi = {"tomo_fwd": 512, "tomo_adj": 512, "cg_tomo": 160, "admm": 128}.get(kind, 512)
    want = _log(rng, 32, hi)
    n = min(SIZES, key=lambda m: abs(m - want))
    if kind in ("tomo_fwd", "tomo_adj", "cg_tomo"):
        nz = _log(rng, 8, min(n, 2 ** 24 // n ** 2))
        c = dict(kind=kind, n=n, nz=nz, ntheta=_log(rng, max(8, n // 4), 3 * n // 2))
        return dict(c, titer=rng.choice([1, 4, 4])) if kind == "cg_tomo" else c
    det = 16 if kind == "admm" else rng.choice([8, 16, 16, 32, 64])
    nprb = rng.choice([det, det, rng.randint(max(4, det // 2), det)]) if det < 64 else 16
    step = max(2, nprb // 4) if det < 64 else 8
    if kind == "admm":
        nprb, step = 16, 4
    n = max(n, 2 * nprb)
    n = min((m for m in SIZES if m >= n), default=512)
    nz = n if kind == "admm" else _log(rng, max(nprb + 1, n // 4), n)
    frames = ((nz - nprb) // step + 1) * ((n - nprb) // step + 1)
    ptheta = 8
    chunks = rng.randint(1, max(1, min(12, 160_000_000 // (frames * det * det * ptheta))))
    ntheta = ptheta * chunks
    if kind in ("ptycho_fwd", "ptycho_adj"):
        ntheta = max(1, ntheta - rng.randint(0, 7))
        return dict(kind=kind, n=n, nz=nz, ntheta=ntheta, det=det, nprb=nprb, step=step,
                    jitter=step / 4, photons=1e3)
    if kind == "admm":
        return dict(kind=kind, n=n, nz=nz, ntheta=max(ntheta, n // 8 * 8), ptheta=ptheta, det=det,
                    nprb=nprb, step=step, jitter=1.0, photons=1e3, model="poisson", piter=4,
                    titer=4, niter=1)
    return dict(kind=kind, n=n, nz=nz, ntheta=ntheta, ptheta=ptheta, det=det, nprb=nprb, step=step,
                jitter=step / 4, photons=rng.choice([1e2, 1e3]),
                model=rng.choice(["poisson", "gaussian"]), piter=rng.choice([2, 4]))


# ---------------------------------------------------------------- inputs
def _gen(seed, k):
    return torch.Generator(device="cuda").manual_seed(1000 * int(seed) + k)


def _cnoise(shape, seed, k, amp):
    g = _gen(seed, k)
    re = torch.randn(shape, generator=g, device="cuda")
    return torch.complex(re, torch.randn(shape, generator=g, device="cuda")) * amp


def _balls(case, seed):
    rng = np.random.default_rng([int(seed), 5])
    n, nz = case["n"], case["nz"]
    out = []
    for _ in range(24):
        r = rng.uniform(n / 40 + 1, n / 10 + 1)
        rad, ang = (n / 2 - r - 2) * math.sqrt(rng.uniform()), rng.uniform(0, 2 * math.pi)
        out.append((rng.uniform(0, nz), rad * math.sin(ang), rad * math.cos(ang), r,
                    rng.uniform(0.2, 1)))
    return out


def _projections(case, seed):
    """Chord lengths of the balls [ntheta, nz, n], scaled to a largest
    projected phase of 1 rad, and that scale."""
    n, nz = case["n"], case["nz"]
    th = torch.from_numpy(make_theta(case["ntheta"])).cuda()[:, None, None]
    z = torch.arange(nz, device="cuda", dtype=F32)[None, :, None]
    s = torch.arange(n, device="cuda", dtype=F32)[None, None, :] - n // 2
    p = torch.zeros((case["ntheta"], nz, n), device="cuda")
    for cz, cy, cx, r, v in _balls(case, seed):
        s0 = cx * torch.cos(th) - cy * torch.sin(th)
        p += 2 * v * torch.sqrt(torch.clamp(r * r - (s - s0) ** 2 - (z - cz) ** 2, min=0))
    sc = 1.0 / (VOXEL * WAVE * max(float(p.max()), 1e-3))
    return p * sc, sc


def _object(case, seed, sc):
    n, nz = case["n"], case["nz"]
    z = torch.arange(nz, device="cuda", dtype=F32)[:, None, None]
    y = (torch.arange(n, device="cuda", dtype=F32) - n // 2)[None, :, None]
    x = (torch.arange(n, device="cuda", dtype=F32) - n // 2)[None, None, :]
    u = torch.zeros((nz, n, n), device="cuda")
    for cz, cy, cx, r, v in _balls(case, seed):
        u += v * ((z - cz) ** 2 + (y - cy) ** 2 + (x - cx) ** 2 <= r * r)
    return torch.complex(u, 0.1 * u) * sc


def _wave(p, part=1.0):
    return torch.exp(torch.complex(-0.1 * p, p) * (VOXEL * WAVE * part)).to(C64)


def _jgrad(u):
    """Forward differences times 2/sqrt(3), last plane 0: [3, nz, n, n]."""
    e = torch.zeros((3, *u.shape), dtype=u.dtype, device=u.device)
    e[0, :, :, :-1] = u[:, :, 1:] - u[:, :, :-1]
    e[1, :, :-1, :] = u[:, 1:, :] - u[:, :-1, :]
    e[2, :-1, :, :] = u[1:, :, :] - u[:-1, :, :]
    return e * (2 / math.sqrt(3))


def _scan(case, seed):
    return jittered_raster(case["ntheta"], case["nz"], case["n"], case["nprb"], case["step"],
                           case["jitter"], np.random.default_rng([int(seed), 7]))


def _frame_index(case, scan, a0, a1):
    """Flat object index [angles, scan, ix, iy] of each probe pixel of angles a0..a1."""
    pos = np.sign(scan[:, a0:a1]) * np.floor(np.abs(scan[:, a0:a1].astype(np.float64)) + 0.5)
    pos = torch.from_numpy(pos.astype(np.int64)).cuda()
    i = torch.arange(case["nprb"], device="cuda")
    x, y = pos[0][..., None, None] + i[:, None], pos[1][..., None, None] + i[None, :]
    t = torch.arange(a0, a1, device="cuda")[:, None, None, None]
    return (t * case["nz"] + y) * case["n"] + x


def _frames(case, scan, prb, psi, a0, a1):
    """probe x object patch in the detector frame, [angles, scan, det, det]."""
    d, p = case["det"], case["nprb"]
    o = (d - p) // 2
    v = psi.reshape(-1)[_frame_index(case, scan, a0, a1)] * prb
    return torch.nn.functional.pad(torch.view_as_real(v), (0, 0, o, d - p - o, o, d - p - o)) \
        if d > p else torch.view_as_real(v)


def _angle_step(case, scan):
    return max(1, 32_000_000 // (scan.shape[2] * case["det"] ** 2))


def _make_data(case, seed, scan, psi):
    """Unit-peak probe scaled to the wanted counts, and the noisy intensities."""
    prb = torch.from_numpy(gaussian_probe(case["nprb"], case["nprb"] / 4)).cuda()
    d = case["det"]
    data = torch.empty((case["ntheta"], scan.shape[2], d, d), device="cuda")
    for a in range(0, case["ntheta"], _angle_step(case, scan)):
        b = min(a + _angle_step(case, scan), case["ntheta"])
        f = torch.fft.fft2(torch.view_as_complex(_frames(case, scan, prb, psi, a, b)))
        data[a:b] = f.real ** 2 + f.imag ** 2
    s = case["photons"] / float(data.max())
    g = _gen(seed, 3)
    for a in range(0, case["ntheta"], _angle_step(case, scan)):
        b = a + _angle_step(case, scan)
        data[a:b] = torch.poisson(data[a:b] * s, generator=g)
    return (prb * math.sqrt(s)).cpu().numpy().astype(np.complex64), data


def _far(case, seed, shape):
    return _cnoise(shape, seed, 4, 1.0)


def _solver(case, scan, prb):
    return Solver(prb, scan, make_theta(case["ntheta"]), [case["det"]] * 2, VOXEL, ENERGY,
                  case["ntheta"], case["nz"], case["n"], case.get("ptheta", case["ntheta"]),
                  case["nz"])


def _inputs(case, seed):
    """The arrays of a case, all on the GPU (probe and scan on the host)."""
    k, sh = case["kind"], (case.get("ntheta"), case["nz"], case.get("n"))
    if k == "unet":
        d = (case["nz"], case["ny"], case["nx"])
        x = torch.randn((*d, 2), generator=_gen(seed, 1), device="cuda")
        for ax in (0, 1, 2):            # smooth, like a reconstruction
            x = (x + torch.roll(x, 1, ax) + torch.roll(x, 2, ax) + torch.roll(x, 3, ax)) / 2
        y = x + 0.3 * torch.roll(x, 1, 0)
        w = {}
        rng = np.random.default_rng([int(seed), 11])
        for name, (co, ci) in NET.items():
            taps = (27,) if name != "head" else ()
            w[name + ".w"] = (rng.standard_normal((co, *taps, ci)) *
                              math.sqrt(2 / (27 * ci))).astype(np.float32)
            w[name + ".b"] = (0.01 * rng.standard_normal(co)).astype(np.float32)
        m = x.abs().max()
        return dict(x=(x / m).contiguous(), y=(y / m).contiguous(), weights=w)
    if "det" in case:
        scan = _scan(case, seed)
    else:                               # tomography alone: a token scan of one position
        case = dict(case, det=8, nprb=8)
        scan, prb = np.zeros((2, case["ntheta"], 1), np.float32), gaussian_probe(8, 2.0)
    p, sc = _projections(case, seed)
    I = dict(scan=scan)
    n, ct = case["n"], _coeftomo(case)
    sgn = 1.0 if (3 * n // 4) % 2 == 0 else -1.0    # sign convention of the transform
    if k in ("ptycho_fwd", "ptycho_adj"):
        prb = gaussian_probe(case["nprb"], case["nprb"] / 4) * np.float32(3.0)
        I["psi"] = _wave(p)
        if k == "ptycho_adj":
            I["far"] = _far(case, seed, (case["ntheta"], scan.shape[2], case["det"], case["det"]))
    elif k in ("cg_ptycho", "admm"):
        prb, I["data"] = _make_data(case, seed, scan, _wave(p))
        I["psi"] = _wave(p, 0.8) * (1 + _cnoise(sh, seed, 1, 0.02))
        I["h"] = _wave(p, 0.9)
        I["lamd"] = _cnoise(sh, seed, 2, 0.05)
    if k in ("tomo_fwd", "cg_tomo", "admm"):
        u = _object(case, seed, sc)
        I["u"] = 0.8 * u + _cnoise(u.shape, seed, 5, 0.02 * sc)
        if k == "tomo_fwd":
            I["u"] = u + _cnoise(u.shape, seed, 5, 0.02 * sc)
    if k == "tomo_adj":
        I["g"] = torch.complex(p, 0.1 * p) * ct + _cnoise(sh, seed, 6, 0.02 * ct * float(p.max()))
    if k == "cg_tomo":
        K = 1j * _wave(p) * (1 - 0.02 * torch.rand(sh, generator=_gen(seed, 7), device="cuda"))
        I["K"] = K.to(C64)
        I["xi0"] = K * torch.complex(p, 0.1 * p) * (ct * sgn)
        I["xi1"] = 0.9 * _jgrad(u) + _cnoise((3, *u.shape), seed, 8, 0.01 * sc)
        I["xi0"], I["xi1"] = I["xi0"].to(C64), I["xi1"].to(C64)
    if k == "admm":
        I["e"] = _jgrad(I["u"]).to(C64)
        I["phi"] = 0.95 * I["e"]
        I["mu"] = _cnoise(I["e"].shape, seed, 9, 0.5 * ALPHA)
    I["prb"] = prb
    return I


def prepare(case, seed):
    I = _inputs(case, seed)
    if case["kind"] == "unet":
        net = UNet3D()
        net.load_state_dict(I.pop("weights"))
        return dict(case=case, net=net, **I)
    c = case if "det" in case else dict(case, det=8)
    slv = _solver(c, I["scan"], I["prb"])
    if case["kind"] == "ptycho_adj":
        slv.cl_ptycho.setobj(slv.scan.data_ptr(), slv.prb.data_ptr())
    I.pop("scan"), I.pop("prb")
    return dict(case=case, slv=slv, **I)


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "unet":
        net = s["net"]
        out = net.forward(s["x"])
        loss, gr = net.loss(out, s["y"])
        net.backward(gr)
        return dict(out=out, loss=loss, gw=dict(net.g), gb=dict(net.gb))
    slv = s["slv"]
    if k == "tomo_fwd":
        return slv.fwd_tomo_batch(s["u"])
    if k == "tomo_adj":
        return slv.adj_tomo_batch(s["g"])
    if k == "ptycho_fwd":
        return slv.fwd_ptycho_batch_dev(s["psi"])
    if k == "ptycho_adj":
        return slv.adj_ptycho(s["far"])
    if k == "cg_ptycho":
        return slv.cg_ptycho_batch(s["data"], s["psi"], s["h"], s["lamd"], RHO, c["piter"],
                                   c["model"])
    if k == "cg_tomo":
        return slv.cg_tomo(s["xi0"], s["xi1"], s["K"], s["u"], RHO, TAU, c["titer"])
    u, psi = slv.admm(s["data"], s["h"], s["e"], s["psi"], s["phi"], s["lamd"], s["mu"], s["u"],
                      ALPHA, c["piter"], c["titer"], c["niter"], c["model"], m0=2, rho=RHO,
                      tau=TAU, lagr_every=0, verbose=False)
    st = slv.state
    return dict(u=u, psi=psi, h=st["h"], e=st["e"], phi=st["phi"], lamd=st["lamd"], mu=st["mu"],
                rho=float(st["rho"]), tau=float(st["tau"]))


# ---------------------------------------------------------------- necessary work
def work(case):
    k = case["kind"]
    if k == "unet":
        v = case["nz"] * case["ny"] * case["nx"]
        macs = v * 27 * (2 * 16 + 16 * 16 + (16 * 32 + 32 * 32) / 8 + (32 * 64 + 64 * 64) / 64 +
                         (96 * 32 + 32 * 32) / 8 + 48 * 16 + 16 * 16)
        return dict(bytes=v * 2 * 4 * 3, flops=6 * macs)
    n, nz, nt = case["n"], case["nz"], case["ntheta"]
    vol, prj = 8 * nz * n * n, 8 * nt * nz * n
    # a transform of the volume and one of the projection lines, per operator call
    tomo = 5 * nz * (n * n * 2 + nt * n) * math.log2(n)
    if k in ("tomo_fwd", "tomo_adj"):
        return dict(bytes=vol + prj, flops=tomo)
    if k == "cg_tomo":
        return dict(bytes=5 * vol + 2 * prj, flops=(2 * case["titer"] + 1) * tomo)
    d, p, st = case["det"], case["nprb"], case["step"]
    pix = nt * ((nz - p) // st + 1) * ((n - p) // st + 1) * d * d
    fft = 10 * pix * math.log2(d)
    if k == "ptycho_fwd":
        return dict(bytes=prj + 4 * pix, flops=fft)
    if k == "ptycho_adj":
        return dict(bytes=prj + 8 * pix, flops=fft)
    # per CG step: psi and the direction forward, the residual back
    cg = dict(bytes=4 * prj + 4 * pix, flops=3 * case["piter"] * fft)
    if k == "cg_ptycho":
        return cg
    it = case["niter"]
    return dict(bytes=4 * pix + 6 * prj + 20 * vol,
                flops=it * (cg["flops"] + (2 * case["titer"] + 1) * tomo))


# ---------------------------------------------------------------- 64-bit restatement
def _coeftomo(case):
    return float(np.float32(1 / np.sqrt(case["ntheta"] * case["n"] / 2)))


class _Tomo:
    """The Radon transform of the framework in 64 bits: for every angle the
    projection's N = 3n/2 frequencies as direct nonuniform Fourier sums at the
    operator's float32 sample positions (k cos, -k sin)/N, k in [-N/2, N/2),
    then the centred inverse DFT, cropped to the n detector pixels.  The object
    is extended to N x N by its edge values inside the circle of radius N/2;
    the adjoint extends the projections to N by their edge values."""

    def __init__(self, case):
        self.n, self.N, self.ct = case["n"], 3 * case["n"] // 2, _coeftomo(case)
        n, N = self.n, self.N
        th = make_theta(case["ntheta"]).astype(np.float64)
        k = np.arange(N) - N // 2
        x = (k / N * np.cos(th)[:, None]).astype(np.float32)
        y = (-k / N * np.sin(th)[:, None]).astype(np.float32)
        lim = np.float32(0.5 - 1e-5)
        x[x >= np.float32(0.5)] = lim
        y[y >= np.float32(0.5)] = lim
        f = lambda a: torch.from_numpy(a.astype(np.float64)).cuda()  # noqa: E731
        self.x, self.y, self.k = f(x), f(y), f(k)
        i = np.arange(N)
        self.pad = torch.from_numpy(np.clip(i - N // 6, 0, n - 1)).cuda()
        c = (i - N // 2).astype(np.float32) / np.float32(N)
        self.mask = f((np.float32(4) * c[None] * c[None] + np.float32(4) * c[:, None] * c[:, None]
                       < np.float32(1) - np.float32(1) / np.float32(N)))
        self.s = f(i - N // 2)
        self.sgn = (-1.0) ** (N // 2) / N * self.ct

    def _e(self, a, b, sign):
        ph = 2 * math.pi * torch.outer(a, b)
        return torch.complex(torch.cos(ph), sign * torch.sin(ph))

    def fwd(self, u):
        n, N, nz = self.n, self.N, u.shape[0]
        ft = (u.to(C128)[:, self.pad[:, None], self.pad[None, :]] * self.mask).reshape(nz * N, N)
        o = N // 2 - n // 2
        inv = self._e(self.k, self.s[o:o + n] / N, 1) * self.sgn
        out = torch.empty((len(self.x), nz, n), dtype=C128, device="cuda")
        for t in range(len(self.x)):
            g = (ft @ self._e(self.s, self.x[t], -1)).reshape(nz, N, N)
            out[t] = (g * self._e(self.s, self.y[t], -1)).sum(1) @ inv
        return out

    def adj(self, g):
        n, N = self.n, self.N
        nz, o = g.shape[1], N // 2 - n // 2
        c = self.s[o:o + n]
        dft = self._e(self.s / N, self.k, -1) * self.sgn
        out = torch.zeros((nz * n, n), dtype=C128, device="cuda")
        for t in range(len(self.x)):
            H = g[t].to(C128)[:, self.pad] @ dft
            a = (H[:, None, :] * self._e(c, self.y[t], 1)[None]).reshape(nz * n, N)
            out += a @ self._e(self.x[t], c, 1)
        return out.reshape(nz, n, n) * self.mask[o:o + n, o:o + n]


class _Ptycho:
    """Probe x patch, unitary 2D DFT, the phase of the sub-pixel position."""

    def __init__(self, case, scan, prb):
        self.case, self.scan = case, scan
        self.prb = torch.from_numpy(prb).cuda().to(C128)
        top = np.abs(prb).max().astype(np.float32)
        self.cp = float(np.float32(1) / top)
        self.cd = float(np.float32(1) / (np.float32(case["det"] ** 2) *
                                         (np.abs(prb) ** 2).max().astype(np.float32)))
        self.shape = (case["ntheta"], case["nz"], case["n"])

    def fwd(self, psi, a0=0, a1=None):
        a1 = self.case["ntheta"] if a1 is None else a1
        f = torch.view_as_complex(_frames(self.case, self.scan, self.prb, psi, a0, a1).contiguous())
        return torch.fft.fft2(f, norm="ortho") * self.cp

    def adj(self, g, a0=0, a1=None):
        c = self.case
        a1 = c["ntheta"] if a1 is None else a1
        o = (c["det"] - c["nprb"]) // 2
        v = torch.fft.ifft2(g, norm="ortho")[..., o:o + c["nprb"], o:o + c["nprb"]]
        v = torch.view_as_real(v * (self.prb.conj() * self.cp)).reshape(-1, 2)
        out = torch.zeros((self.shape[0] * self.shape[1] * self.shape[2], 2), dtype=F64,
                          device="cuda")
        out.index_add_(0, _frame_index(c, self.scan, a0, a1).reshape(-1), v)
        return torch.view_as_complex(out).reshape(self.shape)

    def phase(self):
        fr = self.scan.astype(np.float64)
        fr = fr - np.sign(fr) * np.floor(np.abs(fr) + 0.5)
        return torch.from_numpy(np.exp(2j * np.pi * (fr[0] + fr[1]))).cuda()[..., None, None]


def _n2(x):
    return float((x.real ** 2 + x.imag ** 2).sum())


def _halve(change, gamma):
    """The halving rule on change(gamma) = f(gamma) - f(0)."""
    while change(gamma) > 0 and gamma > 1e-12:
        gamma *= 0.5
    return 0.0 if gamma <= 1e-12 else gamma


def _direction(grad, grad0, d):
    if grad0 is None:
        return -grad
    den = (d.conj() * (grad - grad0)).sum()
    beta = _n2(grad) / den if abs(complex(den)) > 0 else 0.0
    return -grad + beta * d


def _jadj(g):
    r = torch.zeros_like(g[0])
    r[:, :, 0] = g[0, :, :, 0]
    r[:, :, 1:] = g[0, :, :, 1:] - g[0, :, :, :-1]
    r[:, 0] += g[1, :, 0]
    r[:, 1:] += g[1, :, 1:] - g[1, :, :-1]
    r[0] += g[2, 0]
    r[1:] += g[2, 1:] - g[2, :-1]
    return r * (-2 / math.sqrt(3))


def _cg_tomo(R, xi0, xi1, K, u, rho, tau, titer):
    grad0, d, gamma = None, None, 2.0
    for _ in range(titer):
        r0, g0 = K * R.fwd(u) - xi0, _jgrad(u) - xi1
        grad = rho * R.adj(K.conj() * r0) + tau * _jadj(g0)
        d = _direction(grad, grad0, d)
        grad0 = grad
        dr, dg = K * R.fwd(d), _jgrad(d)
        a = rho * _n2(dr) + tau * _n2(dg)
        b = 2 * (rho * float((r0.conj() * dr).sum().real) +
                 tau * float((g0.conj() * dg).sum().real))
        gamma = _halve(lambda t: t * t * a + t * b, gamma)
        u = u + gamma * d
    return u


def _cg_chunk(F, a0, a1, data, psi, h, lamd, rho, piter, model):
    """CG on the angles a0..a1 of full-size arrays (zero elsewhere)."""
    sl = slice(a0, a1)
    grad0, d, gamma = None, None, 2.0
    q = data[sl].to(F64) * F.cd

    def place(x):
        full = torch.zeros(F.shape, dtype=C128, device="cuda")
        full[sl] = x
        return full
    for _ in range(piter):
        a = F.fwd(place(psi), a0, a1)
        m = a.abs()
        r = a - q * a / (m ** 2 + 1e-32) if model == "poisson" else \
            a - torch.sqrt(q) * torch.exp(1j * torch.angle(a))
        e0 = h - psi + lamd / rho
        grad = F.adj(r, a0, a1)[sl] - rho * e0
        d = _direction(grad, grad0, d)
        grad0 = grad
        b = F.fwd(place(d), a0, a1)
        floor = torch.clamp(m, min=1e-32)

        def change(t):
            mt = (a + t * b).abs()
            if model == "poisson":
                f = (mt ** 2 - m ** 2 - 2 * q * torch.log(torch.clamp(mt, min=1e-32) / floor)).sum()
            else:
                f = ((mt - torch.sqrt(q)) ** 2 - (m - torch.sqrt(q)) ** 2).sum()
            return float(f) + rho * (t * t * _n2(d) - 2 * t * float((e0.conj() * d).sum().real))
        gamma = _halve(change, gamma)
        psi = psi + gamma * d
    return psi


def _cg_ptycho(F, case, data, psi, h, lamd, rho):
    out = psi.to(C128).clone()
    for a in range(0, case["ntheta"], case["ptheta"]):
        b = a + case["ptheta"]
        out[a:b] = _cg_chunk(F, a, b, data, psi[a:b].to(C128), h[a:b].to(C128),
                             lamd[a:b].to(C128), rho, case["piter"], case["model"])
    return out


def _balance(r, s, v):
    return v * 2 if r > 10 * s else v * 0.5 if s > 10 * r else v


def _admm(case, I, F, R):
    c1, ct, rho, tau = VOXEL * WAVE, R.ct, RHO, TAU
    S = {k: I[k].to(C128) for k in ("h", "e", "psi", "phi", "lamd", "mu", "u")}
    n, r = case["n"], case["nprb"] // 2
    for _ in range(case["niter"]):
        S["psi"] = psi = _cg_ptycho(F, case, I["data"], S["psi"], S["h"], S["lamd"], rho)
        ang = torch.angle(psi)
        ps = float((ang[:, :, r:2 * r].mean() + ang[:, :, n - 2 * r:n - r].mean()) / 2)
        t = (psi - S["lamd"] / rho) * np.exp(-1j * ps)
        lt = torch.complex(torch.log(torch.clamp(t.abs(), min=1e-32)), torch.angle(t))
        K = 1j * t / t.abs().max()
        S["u"] = u = _cg_tomo(R, K * (-1j * lt / c1) * ct, S["phi"] - S["mu"] / tau, K, S["u"],
                              rho, tau, case["titer"])
        e = _jgrad(u)
        z = e + S["mu"] / tau
        za = torch.sqrt((z.real ** 2 + z.imag ** 2).sum(0))
        S["phi"] = z * torch.clamp(1 - ALPHA / tau / torch.clamp(za, min=1e-300), min=0)
        h = torch.exp(1j * R.fwd(u) * (c1 / ct)) * np.exp(1j * ps)
        S["lamd"] = S["lamd"] + rho * (h - psi)
        S["mu"] = S["mu"] + tau * (e - S["phi"])
        rho, tau = _balance(_n2(psi - h), rho * rho * _n2(h - S["h"]), rho), \
            _balance(_n2(S["phi"] - e), tau * tau * _n2(e - S["e"]), tau)
        S["h"], S["e"] = h, e
    return dict({k: S[k] for k in ("u", "psi", "h", "e", "phi", "lamd", "mu")}, rho=rho, tau=tau)


def _unet(I):
    par = {k: [torch.from_numpy(I["weights"][k + x]).cuda().to(F64).requires_grad_()
               for x in (".w", ".b")] for k in NET}

    def conv(x, name):
        w, b = par[name]
        d, h, w_ = x.shape[:3]
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b
        for i in range(27):
            z, yy, xx = i // 9, i // 3 % 3, i % 3
            y = y + xp[z:z + d, yy:yy + h, xx:xx + w_] @ w[:, i].T
        return torch.relu(y)

    def pool(x):
        d, h, w, c = x.shape
        return x.reshape(d // 2, 2, h // 2, 2, w // 2, 2, c).mean((1, 3, 5))

    def up(x):
        for ax in (0, 1, 2):
            x = x.repeat_interleave(2, ax)
        return x
    x, y = I["x"].to(F64), I["y"].to(F64)
    e1 = conv(conv(x, "e1a"), "e1b")
    e2 = conv(conv(pool(e1), "e2a"), "e2b")
    bn = conv(conv(pool(e2), "bna"), "bnb")
    d2 = conv(conv(torch.cat([up(bn), e2], -1), "d2a"), "d2b")
    d1 = conv(conv(torch.cat([up(d2), e1], -1), "d1a"), "d1b")
    out = x + d1 @ par["head"][0].T + par["head"][1]
    loss = ((out - y) ** 2).mean()
    loss.backward()
    return dict(out=out.detach(), loss=loss.detach(), gw={k: par[k][0].grad for k in NET},
                gb={k: par[k][1].grad for k in NET})


def exact(case, seed):
    k = case["kind"]
    I = _inputs(case, seed)
    if k == "unet":
        return _unet(I)
    # cost of the direct sums of one operator call; beyond this the answer takes too long
    ops = 8.0 * case["nz"] * (1.5 * case["n"]) ** 3 * case["ntheta"]
    calls = {"tomo_fwd": 1, "tomo_adj": 1, "cg_tomo": 2 * case.get("titer", 0),
             "admm": (2 * case.get("titer", 0) + 1) * case.get("niter", 0)}.get(k, 0)
    if ops * calls > 1.2e14:
        return None
    if k == "tomo_fwd":
        return _Tomo(case).fwd(I["u"])
    if k == "tomo_adj":
        return _Tomo(case).adj(I["g"])
    if k == "cg_tomo":
        v = [I[x].to(C128) for x in ("xi0", "xi1", "K", "u")]
        return _cg_tomo(_Tomo(case), *v, RHO, TAU, case["titer"])
    F = _Ptycho(case, I["scan"], I["prb"])
    st = _angle_step(case, I["scan"])
    blocks = [(a, min(a + st, case["ntheta"])) for a in range(0, case["ntheta"], st)]
    if k == "ptycho_fwd":
        return torch.cat([F.fwd(I["psi"].to(C128), a, b).abs() ** 2 / F.cd for a, b in blocks])
    if k == "ptycho_adj":
        g = I["far"]
        return sum(F.adj(g[a:b].to(C128) * F.phase().conj()[a:b], a, b) for a, b in blocks)
    if k == "cg_ptycho":
        return _cg_ptycho(F, case, I["data"], I["psi"], I["h"], I["lamd"], RHO)
    return _admm(case, I, F, _Tomo(case))
