"""Drop-in ``Solver`` for joint ptycho-tomography by ADMM on MI355X.

Mirrors the reference class ``Solver`` (src/ptychotomo/solver.py:19-336):
same constructor, method names, argument meaning, shapes, dtypes and
normalisation.  Arrays are PyTorch tensors on the GPU (complex64 / float32);
NumPy inputs are copied to the device.  Every computation runs in the HIP
library through its C ABI; PyTorch only holds the buffers.

Implementation notes (mathematically identical to the reference, different
in rounding only):
* ``fwd_tomo_batch`` / ``adj_tomo_batch`` and ``cg_ptycho_batch`` process the
  whole volume in one native call; the angle chunking of ``ptheta`` is kept
  where it changes the mathematics (per-chunk CG step and Dai-Yuan beta,
  solver.py:245-254), as segmented reductions.
* ``cg_tomo`` updates R u by linearity (R(u + g d) = R u + g R d) instead of
  a fresh transform per CG iteration; ``admm`` transforms the new u once per
  ADMM iteration for the h update (solver.py:323) and the next cg_tomo.
* The line searches evaluate up to 7 halving candidates per sweep in one
  fused pass (``cg_ptycho``: far field and rho term; ``cg_tomo``: K R and J
  terms).  Each candidate is formed as the reference forms it -- x + g*dx
  element-wise in FP32 -- so a step below FP32 resolution reproduces the
  gamma = 0 value exactly and the halving rule stops where the reference's
  does instead of collapsing to gamma = 0.
* Scalars (norms, dots, steps) are accumulated in FP64, and the scalar rules
  (Dai-Yuan beta, the halving decisions, the takexi phase, the penalty
  update) run as FP64 device kernels, so an ADMM iteration is enqueued
  without host round trips and can be replayed as a HIP graph.  After a zero
  step the reference's Dai-Yuan beta is 0/0; here it is 0 (restart).
"""
import contextlib
import ctypes
import sys

import numpy as np
import torch

from . import _lib
from ._dev import c64, device, empty, f32, f64, ptr, stream, to_dev, zeros
from .objects import wavenumber as _wavenumber
from .ptychofft import ptychofft
from .radonusfft import radonusfft

PLANCK_CONSTANT = 6.58211928e-19  # [keV*s]   solver.py:15
SPEED_OF_LIGHT = 299792458e+2     # [cm/s]    solver.py:16

_MAXGAM = 8      # candidate slots of the line-search buffers (gamma = 0 + 7 halvings)
# halvings per sweep of cg_ptycho's device line searches; every schedule covers at
# least 41 halvings (2 -> below 1e-12), so the halving rule is followed to its end
# (cg_tomo's search is one call, pt_k_tomo_linesearch).  The first CG step starts
# at gamma = 2 and usually accepts after 3-4 halvings (one sweep of 5); the later
# steps start from the previous step, accept it about three times in four
# (256^3: 212 of 288 chunk searches), and otherwise mostly within 5 more
# halvings (sweeps of 1, 5, then 7).  A sweep costs the two far-field
# transforms of every open chunk plus each candidate's sums (about a fifth of
# the transforms' cost each)
_PSCHED_FIRST = (5,) + (7,) * 6
_PSCHED_LATER = (1, 5) + (7,) * 6
# device scalar block (FP64): 1, rho, tau, takexi {pshift, cos, sin, kfac},
# takexi statistics, penalty norms, max |angle psi|
_ONE, _RHO, _TAU, _PRM, _STATS, _NORMS, _MAXANG, _NSC = 0, 1, 2, 3, 8, 12, 16, 24


def _call(name, *args):
    return _lib.call(name, *args)


class Solver(object):
    """solver.py:19-46."""

    def __init__(self, prb, scan, theta, det, voxelsize, energy, ntheta, nz, n, ptheta, pnz):
        self.voxelsize = voxelsize
        self.energy = energy
        self.scan = to_dev(scan, f32)
        self.prb = to_dev(prb, c64)
        self.theta = to_dev(theta, f32)
        self.ntheta = int(ntheta)
        self.nz = int(nz)
        self.n = int(n)
        self.nscan = int(self.scan.shape[2])
        self.ndety = int(det[0])
        self.ndetx = int(det[1])
        self.nprb = int(self.prb.shape[0])
        self.ptheta = int(ptheta)
        self.pnz = int(pnz)
        if self.ntheta % self.ptheta:
            raise ValueError("ntheta must be a multiple of ptheta")
        if self.nz % self.pnz:
            raise ValueError("nz must be a multiple of pnz")
        self.nchunk = self.ntheta // self.ptheta
        # chunk-sized ptychography operator (solver.py:35-36; det[0] -> detx)
        self.cl_ptycho = ptychofft(self.ptheta, self.nz, self.n, self.ptheta, self.nscan,
                                   self.ndety, self.ndetx, self.nprb)
        # slab-sized tomography operator (solver.py:39-40)
        self.cl_tomo = radonusfft(self.ntheta, self.pnz, self.n)
        self.cl_tomo.setobj(self.theta.data_ptr())
        # whole-volume operators used by the batch methods and the solvers
        if self.pnz == self.nz:
            self._tomo = self.cl_tomo
        else:
            self._tomo = radonusfft(self.ntheta, self.nz, self.n)
            self._tomo.setobj(self.theta.data_ptr())
        self._ptycho = ptychofft(self.ntheta, self.nz, self.n, self.ntheta, self.nscan,
                                 self.ndety, self.ndetx, self.nprb)
        self._ptycho.setobj(self.scan.data_ptr(), self.prb.data_ptr())
        # normalisation coefficients (solver.py:43-46)
        prb_h = self.prb.cpu().numpy()
        self.coeftomo = np.float32(1 / np.sqrt(self.ntheta * self.n / 2))
        self.coefptycho = np.float32(1) / np.abs(prb_h).max().astype(np.float32)
        self.coefdata = np.float32(1) / (np.float32(self.ndetx * self.ndety)
                                         * (np.abs(prb_h) ** 2).max().astype(np.float32))
        self._sc = torch.zeros(64, dtype=f64, device=device())  # scalar results
        self._works = {}
        self.history = []
        self.state = None

    # ------------------------------------------------------------------ helpers
    def _scalars(self, k):
        """first k FP64 results (synchronises)."""
        return self._sc[:k].cpu().numpy()

    def _dev_data(self, data):
        """data [ntheta, nscan, ndety, ndetx] float32 on the device: a device
        tensor is used as it is; a host array is copied on every call (as the
        reference copies data[ids] per call, solver.py:250-251), so changes the
        caller makes to it between calls are always seen.  To avoid the copy,
        pass a device tensor."""
        if isinstance(data, torch.Tensor) and data.is_cuda and data.dtype == f32 \
                and data.is_contiguous():
            return data
        return to_dev(data, f32)

    # ------------------------------------------------------------------ element-wise
    def mlog(self, psi):
        """solver.py:48-52."""
        psi = to_dev(psi, c64)
        res = empty(psi.shape)
        _call("pt_k_mlog", ptr(res), ptr(psi), psi.numel(), stream())
        return res

    def wavenumber(self):
        """solver.py:55-56."""
        return 2 * np.pi / (2 * np.pi * PLANCK_CONSTANT * SPEED_OF_LIGHT / self.energy)

    def exptomo(self, psi):
        """solver.py:59-60: exp(i*psi*voxelsize*k/coeftomo)."""
        psi = to_dev(psi, c64)
        res = empty(psi.shape)
        c = self.voxelsize * self.wavenumber() / float(self.coeftomo)
        _call("pt_k_exptomo", ptr(res), ptr(psi), c, 0.0, None, psi.numel(), stream())
        return res

    def logtomo(self, psi):
        """solver.py:63-64: -i/k * mlog(psi)/voxelsize*coeftomo."""
        m = self.mlog(psi)
        a = -float(self.coeftomo) / (self.wavenumber() * self.voxelsize)
        _call("pt_k_lincomb3", ptr(m), 0.0, a, ptr(m), 0.0, 0.0, None, 0.0, 0.0, None,
              m.numel(), stream())
        return m

    # ------------------------------------------------------------------ tomography
    def fwd_tomo(self, u):
        """solver.py:67-72 (one pnz slab)."""
        u = to_dev(u, c64)
        res = empty((self.ntheta, self.pnz, self.n))
        self.cl_tomo.fwd_scaled(res.data_ptr(), u.data_ptr(), float(self.coeftomo))
        return res

    def adj_tomo(self, data):
        """solver.py:75-80 (one pnz slab)."""
        data = to_dev(data, c64)
        res = empty((self.pnz, self.n, self.n))
        self.cl_tomo.adj_scaled(res.data_ptr(), data.data_ptr(), float(self.coeftomo))
        return res

    def fwd_tomo_batch(self, u):
        """solver.py:83-89 (whole volume in one call; pnz is memory-only)."""
        u = to_dev(u, c64)
        res = empty((self.ntheta, self.nz, self.n))
        self._tomo.fwd_scaled(res.data_ptr(), u.data_ptr(), float(self.coeftomo))
        return res

    def adj_tomo_batch(self, data, scale=1.0):
        """solver.py:92-97; ``scale`` multiplies the result (fused)."""
        data = to_dev(data, c64)
        res = empty((self.nz, self.n, self.n))
        self._tomo.adj_scaled(res.data_ptr(), data.data_ptr(), float(self.coeftomo) * scale)
        return res

    def fbp_tomo_batch(self, data):
        """Filtered backprojection of projections scaled like fwd_tomo_batch:
        the adjoint with the reference's ramp filter (applyfilter,
        kernels.cuh:174-187; commented out at radonusfft.cu:121), normalised so
        that fbp_tomo_batch(fwd_tomo_batch(u)) approximates u.  The filter
        weight is about 4N|k|/N per detector frequency k, N = 3n/2, so the
        filtered backprojection over ntheta angles in [0, pi) is
        4 N ntheta / pi times the inverse Radon transform; coeftomo enters
        once from the data and once from the adjoint."""
        data = to_dev(data, c64)
        res = empty((self.nz, self.n, self.n))
        N = 3 * self.n // 2
        scale = float(np.pi / (4.0 * N * self.ntheta * float(self.coeftomo)))
        self._tomo.setfilter("ramp")
        try:
            self._tomo.adj_scaled(res.data_ptr(), data.data_ptr(), scale)
        finally:
            self._tomo.setfilter(None)
        return res

    # ------------------------------------------------------------------ ptychography
    def fwd_ptycho(self, psi):
        """solver.py:100-105 (chunk set by cl_ptycho.setobj)."""
        psi = to_dev(psi, c64)
        res = empty((self.ptheta, self.nscan, self.ndety, self.ndetx))
        self.cl_ptycho.fwd_scaled(res.data_ptr(), psi.data_ptr(), float(self.coefptycho))
        return res

    def fwd_ptycho_batch(self, psi):
        """solver.py:108-117: |F psi|^2/coefdata for all angles, returned as a
        host float32 array like the reference."""
        return self.fwd_ptycho_batch_dev(psi).cpu().numpy()

    def fwd_ptycho_batch_dev(self, psi):
        psi = to_dev(psi, c64)
        data = empty((self.ntheta, self.nscan, self.ndety, self.ndetx), f32)
        _call("pt_ptycho_intensity", self._ptycho._h, ptr(data), ptr(psi), float(self.coefptycho),
              float(1.0 / self.coefdata), stream())
        return data

    def adj_ptycho(self, data):
        """solver.py:120-125 (chunk set by cl_ptycho.setobj)."""
        data = to_dev(data, c64)
        res = empty((self.ptheta, self.nz, self.n))
        self.cl_ptycho.adj_scaled(res.data_ptr(), data.data_ptr(), float(self.coefptycho))
        return res

    # ------------------------------------------------------------------ regulariser
    def fwd_reg(self, u):
        """solver.py:128-134."""
        u = to_dev(u, c64)
        res = empty((3, *u.shape))
        _call("pt_k_reg_fwd", ptr(res), ptr(u), *u.shape, stream())
        return res

    def adj_reg(self, gr):
        """solver.py:137-146."""
        gr = to_dev(gr, c64)
        res = empty(gr.shape[1:])
        _call("pt_k_reg_adj", ptr(res), ptr(gr), *gr.shape[1:], stream())
        return res

    def solve_reg(self, u, mu, tau, alpha):
        """solver.py:257-264."""
        u = to_dev(u, c64)
        mu = to_dev(mu, c64)
        res = empty(mu.shape)
        _call("pt_k_reg_solve", ptr(res), ptr(u), ptr(mu), float(tau), None, float(alpha), *u.shape,
              stream())
        return res

    # ------------------------------------------------------------------ device scalars
    def _scalar_block(self, rho=0.5, tau=0.5):
        """FP64 device block holding the ADMM scalars (layout _ONE.._NSC)."""
        blk = torch.zeros(_NSC, dtype=f64)
        blk[_ONE], blk[_RHO], blk[_TAU] = 1.0, float(rho), float(tau)
        return blk.to(device())

    def _work(self, key, nseg, shape):
        """Per-shape CG workspace (allocated once, reused: stable addresses
        for graph replay)."""
        w = self._works.get(key)
        if w is None or w["shape"] != tuple(shape) or w["nseg"] != nseg:
            z = lambda n: torch.zeros(n, dtype=f64, device=device())
            w = {"shape": tuple(shape), "nseg": nseg,
                 "red": z(3 * nseg), "beta": z(2 * nseg), "state": z(2 * nseg),
                 "step": z(2 * nseg), "cand": z(_MAXGAM * nseg), "cand2": z(_MAXGAM * nseg),
                 "f1": z(_MAXGAM * nseg),
                 "f2": z(_MAXGAM * nseg), "sc": z(4),
                 "state0": torch.tensor([2.0, 0.0] * nseg, dtype=f64, device=device()),
                 "grad": [empty(shape), empty(shape)], "d": empty(shape)}
            self._works[key] = w
        return w

    # ------------------------------------------------------------------ takexi
    def takexi(self, psi, phi, lamd, mu, rho, tau):
        """solver.py:149-168 (r = nprb // 2).  Returns (xi0, xi1, K, pshift)."""
        psi, lamd = to_dev(psi, c64), to_dev(lamd, c64)
        phi, mu = to_dev(phi, c64), to_dev(mu, c64)
        blk = self._scalar_block(rho, tau)
        xi0, K, xi1 = empty(psi.shape), empty(psi.shape), empty(phi.shape)
        self._takexi_dev(psi, phi, lamd, mu, blk, xi0, K, xi1)
        return xi0, xi1, K, float(blk[_PRM].item())

    def _takexi_dev(self, psi, phi, lamd, mu, blk, xi0, K, xi1):
        st = stream()
        r = self.nprb // 2
        _call("pt_k_takexi_stats", _dp(blk, _STATS), ptr(psi), ptr(lamd), 0.0, _dp(blk, _RHO),
              self.ntheta, self.nz, self.n, r, st)
        c1 = self.voxelsize * self.wavenumber()
        kc = c1 / float(self.coeftomo)
        _call("pt_k_takexi_dev", ptr(xi0), ptr(K), _dp(blk, _PRM), ptr(psi), ptr(lamd),
              _dp(blk, _RHO), _dp(blk, _STATS), float(self.ntheta * self.nz * r), kc, c1,
              float(self.coeftomo), psi.numel(), st)
        # xi1 = phi - mu/tau
        _call("pt_k_dual", ptr(xi1), ptr(phi), None, ptr(mu), 0.0, _dp(blk, _TAU), 1,
              phi.numel(), st)

    # ------------------------------------------------------------------ line search
    def line_search(self, minf, gamma, u, fu, d, fd):
        """solver.py:171-177 (generic form, callable minf)."""
        while (minf(u, fu) - minf(u + gamma * d, fu + gamma * fd) < 0 and gamma > 1e-12):
            gamma *= 0.5
        if gamma <= 1e-12:
            gamma = 0
        return gamma

    def _line_search_gen(self, w, nseg, weights, sched):
        """The halving rule of line_search for nseg independent segments, on
        the device: sweeps of sched[i] halvings (plus gamma = 0) until every
        segment has accepted a step (a schedule covers 2 -> 1e-12).  A
        generator: yields (cand, ngam, state, f1, f2, select) where the two
        functional terms (their change from gamma = 0) are to be evaluated at
        the ngam candidate slots per segment, skipping finished segments, and
        the sweep's selection is to be made with the arguments `select` (next
        candidates, steps, weights, ngam of the next sweep, last; by the caller,
        alone or in a group of instances); weights points to the terms' two FP64
        weights.  Consecutive sweeps alternate between two candidate buffers."""
        st = stream()
        bufs = (w["cand"], w["cand2"])
        ng = sched[0] + 1
        _call("pt_k_ls_begin", ptr(w["state"]), ptr(bufs[0]), nseg, ng, st)
        for sw in range(len(sched)):
            last = sw == len(sched) - 1
            ng_next = ng if last else sched[sw + 1] + 1
            cur, nxt = bufs[sw % 2], bufs[(sw + 1) % 2]
            yield cur, ng, w["state"], w["f1"], w["f2"], (nxt.data_ptr(), w["step"].data_ptr(),
                                                          weights.value, ng_next, int(last))
            ng = ng_next

    def _dai_yuan_dev(self, w, i, grad, grad0, L, nseg):
        """d = -grad (i = 0) or -grad + beta d (solver.py:192-196, 227-231)."""
        st = stream()
        d = w["d"]
        if i == 0:
            _call("pt_k_dy_update", ptr(d), ptr(grad), None, 1, L, nseg, st)
        else:
            _call("pt_k_dy_reduce", ptr(w["red"]), ptr(grad), ptr(grad0), ptr(d), L, nseg, st)
            _call("pt_k_dai_yuan", ptr(w["beta"]), ptr(w["red"]), nseg, st)
            _call("pt_k_dy_update", ptr(d), ptr(grad), ptr(w["beta"]), 0, L, nseg, st)

    # ------------------------------------------------------------------ cg_tomo
    def cg_tomo(self, xi0, xi1, K, init, rho, tau, titer):
        """solver.py:180-203."""
        xi0, xi1, K = to_dev(xi0, c64), to_dev(xi1, c64), to_dev(K, c64)
        u = to_dev(init, c64).clone()
        Ru = self.fwd_tomo_batch(u)
        blk = self._scalar_block(rho, tau)
        hist = torch.zeros(max(titer, 1), dtype=f64, device=device())
        self._cg_tomo_dev(xi0, xi1, K, u, Ru, blk, titer, hist)
        self._last_tomo_gammas = [float(v) for v in hist[:titer].cpu().numpy()]
        return u

    def _cg_tomo_dev(self, xi0, xi1, K, u, Ru, blk, titer, hist=None):
        """cg_tomo on u in place; Ru = R u is carried by linearity
        (R(u + g d) = R u + g R d), so a CG iteration costs one adjoint and one
        forward USFFT.  Ru is left as before the last step (nothing needs it
        then)."""
        nz, n = self.nz, self.n
        lenp, lenu = Ru.numel(), u.numel()
        st = stream()
        w = self._work("tomo", 1, u.shape)
        if "r_t" not in w or w["r_t"].shape != Ru.shape:
            w["r_t"], w["Rd"] = empty(Ru.shape), empty(Ru.shape)
        r_t, Rd, d = w["r_t"], w["Rd"], w["d"]
        w["state"].copy_(w["state0"])             # gamma = 2 (solver.py:184)
        ct = float(self.coeftomo)
        grad0 = None
        for i in range(titer):
            grad = w["grad"][i % 2]
            # grad = rho*R*(conj(K)(K Ru - xi0)) + tau*J*(J u - xi1); the previous
            # step's Ru += g R d on the way
            _call("pt_k_cg_resid", ptr(r_t), ptr(Ru), ptr(Rd) if i else None, ptr(w["step"]),
                  ptr(K), ptr(xi0), _dp(blk, _RHO), lenp, st)
            self._tomo.adj_scaled(grad.data_ptr(), r_t.data_ptr(), ct)
            _call("pt_k_cg_reg_grad", ptr(grad), ptr(u), ptr(xi1), _dp(blk, _TAU), nz, n, n, st)
            self._dai_yuan_dev(w, i, grad, grad0, lenu, 1)
            grad0 = grad
            self._tomo.fwd_scaled(Rd.data_ptr(), d.data_ptr(), ct)

            # minf = rho*|K R u - xi0|^2 + tau*|J u - xi1|^2 (solver.py:181-182)
            _call("pt_k_tomo_linesearch", ptr(w["state"]), ptr(w["step"]), ptr(K), ptr(Ru),
                  ptr(Rd), ptr(xi0), ptr(u), ptr(d), ptr(xi1), _dp(blk, _RHO), lenp, nz, n, n, st)
            _call("pt_k_axpy_seg", ptr(u), ptr(w["step"]), ptr(d), lenu, 1, st)
            if hist is not None:
                hist[i:i + 1].copy_(w["step"][0:1])

    # ------------------------------------------------------------------ cg_ptycho
    def cg_ptycho(self, data, init, h, lamd, rho, piter, model):
        """solver.py:206-242 on the chunk set by ``cl_ptycho.setobj`` (data
        already multiplied by coefdata, as the reference passes it)."""
        data = to_dev(data, f32)
        psi = to_dev(init, c64).clone()
        self._cg_ptycho_host(self.cl_ptycho, 1, data, psi, h, lamd, rho, piter, model, 1.0)
        return psi

    def cg_ptycho_batch(self, data, init, h, lamd, rho, piter, model):
        """solver.py:245-254: all angle chunks in one fused pass with
        per-chunk step lengths and Dai-Yuan coefficients."""
        d = self._dev_data(data)
        psi = to_dev(init, c64).clone()
        self._cg_ptycho_host(self._ptycho, self.nchunk, d, psi, h, lamd, rho, piter, model,
                             float(self.coefdata))
        return psi

    def _cg_ptycho_host(self, op, nseg, data, psi, h, lamd, rho, piter, model, coefdata):
        blk = self._scalar_block(rho, 0.5)
        hist = torch.zeros((max(piter, 1), nseg), dtype=f64, device=device())
        self._cg_ptycho_dev(op, nseg, data, psi, to_dev(h, c64), to_dev(lamd, c64), blk, piter,
                            model, coefdata, hist)
        g = hist[:piter].cpu().numpy()
        self._chunk_gammas = [[float(v) for v in g[:, s]] for s in range(nseg)]
        self._check_phase(blk)

    def _cg_ptycho_dev(self, op, nseg, data, psi, h, lamd, blk, piter, model, coefdata,
                       hist=None):
        """cg_ptycho on psi in place, nseg angle chunks with their own step and
        Dai-Yuan beta (solver.py:245-254); max|angle psi| goes to blk."""
        mdl = _lib.PT_MODEL[model]
        for req in self._cg_ptycho_gen(op, nseg, data, psi, h, lamd, blk, piter, coefdata, hist):
            run_ptycho_request(req, mdl, stream())

    def _cg_ptycho_gen(self, op, nseg, data, psi, h, lamd, blk, piter, coefdata, hist=None):
        """_cg_ptycho_dev as a generator: its two heavy launches -- the fused
        gradient and each line-search sweep -- are yielded as requests
        ("grad", GradArgs) and ("ls", LinesearchArgs, ngam, select) for the caller
        to make (run_ptycho_request, or one grouped call for many instances in
        lock-step); everything else is enqueued here on the current stream."""
        st = stream()
        L = psi.numel()
        w = self._work(("ptycho", id(op)), nseg, psi.shape)
        chunk = op.Ntheta // nseg
        cp, cd = float(self.coefptycho), float(coefdata)
        rho_dev = blk.data_ptr() + 8 * _RHO
        w["state"].copy_(w["state0"])             # gamma = 2 (solver.py:217)
        grad0 = None
        d = w["d"]
        for i in range(piter):
            grad = w["grad"][i % 2]
            yield ("grad", _lib.GradArgs(op._h, grad.data_ptr(), psi.data_ptr(), data.data_ptr(),
                                         h.data_ptr(), lamd.data_ptr(), 0.0, rho_dev, cp, cd))
            self._dai_yuan_dev(w, i, grad, grad0, L, nseg)
            grad0 = grad
            # minf = data term + rho*|h - psi + lamd/rho|^2 (solver.py:208-213): the
            # two terms in one pass over the overlap-add tiles
            for cand, ng, state, f1, f2, sel in self._line_search_gen(
                    w, nseg, _dp(blk, _ONE), _PSCHED_FIRST if i == 0 else _PSCHED_LATER):
                yield ("ls", _lib.LinesearchArgs(
                    op._h, f1.data_ptr(), f2.data_ptr(), psi.data_ptr(), d.data_ptr(),
                    data.data_ptr(), h.data_ptr(), lamd.data_ptr(), 0.0, rho_dev,
                    cand.data_ptr(), chunk, cp, cd, state.data_ptr()), ng, sel)
            _call("pt_k_axpy_seg", ptr(psi), ptr(w["step"]), ptr(d), L, nseg, st)
            if hist is not None:
                hist[i].copy_(w["step"][0::2])
        _call("pt_k_max_angle", _dp(blk, _MAXANG), ptr(psi), L, st)

    def _check_phase(self, blk):
        mx = float(blk[_MAXANG].item())
        if mx > 3.14:
            # the reference's warning (solver.py:238-240), on stderr: stdout
            # stays free for a caller's own output
            print('possible phase wrap, max computed angle', mx, file=sys.stderr)

    # ------------------------------------------------------------------ penalties / Lagrangian
    def update_penalty(self, psi, h, h0, phi, e, e0, rho, tau):
        """solver.py:267-282."""
        blk = self._scalar_block(rho, tau)
        psi, h, h0 = to_dev(psi, c64), to_dev(h, c64), to_dev(h0, c64)
        phi, e, e0 = to_dev(phi, c64), to_dev(e, c64), to_dev(e0, c64)
        self._penalty_dev(psi, h, h0, phi, e, e0, blk)
        v = blk[_RHO:_TAU + 1].cpu().numpy()
        return float(v[0]), float(v[1])

    def _penalty_dev(self, psi, h, h0, phi, e, e0, blk):
        st = stream()
        for k, (a, b) in enumerate(((psi, h), (h, h0), (phi, e), (e, e0))):
            _call("pt_k_norm2_lin", _dp(blk, _NORMS + k), ptr(a), ptr(b), 1.0, 0.0, -1.0, 0.0,
                  a.numel(), 1, st)
        _call("pt_k_penalty", _dp(blk, _RHO), _dp(blk, _NORMS), st)

    def take_lagr(self, psi, phi, data, h, e, lamd, mu, alpha, rho, tau, model):
        """solver.py:285-305 (lagr[6] = sum(lagr[0:5]) as in the reference)."""
        st = stream()
        dd = self._dev_data(data)
        psi, phi, h, e = to_dev(psi, c64), to_dev(phi, c64), to_dev(h, c64), to_dev(e, c64)
        lamd, mu = to_dev(lamd, c64), to_dev(mu, c64)
        lagr = np.zeros(7, dtype=np.float32)
        sums = torch.zeros(self.nchunk, dtype=f64, device=device())
        gz = torch.zeros(self.nchunk, dtype=f64, device=device())
        _call("pt_ptycho_minf", self._ptycho._h, ptr(sums), ptr(psi), None, ptr(dd), ptr(gz), 1,
              self.ptheta, float(self.coefptycho), float(self.coefdata), _lib.PT_MODEL[model],
              1, None, st)
        plane = self.nz * self.n * self.n
        _call("pt_k_tv_norm", ptr(self._sc[0:]), ptr(phi), plane, st)
        _call("pt_k_dot_diff", ptr(self._sc[1:]), ptr(lamd), ptr(h), ptr(psi), h.numel(), st)
        _call("pt_k_norm2_lin", ptr(self._sc[3:]), ptr(h), ptr(psi), 1.0, 0.0, -1.0, 0.0,
              h.numel(), 1, st)
        _call("pt_k_dot_diff", ptr(self._sc[4:]), ptr(mu), ptr(e), ptr(phi), e.numel(), st)
        _call("pt_k_norm2_lin", ptr(self._sc[6:]), ptr(e), ptr(phi), 1.0, 0.0, -1.0, 0.0,
              e.numel(), 1, st)
        v = self._scalars(7)
        lagr[0] = sums.sum().item()
        lagr[1] = alpha * v[0]
        lagr[2] = 2 * v[1]
        lagr[3] = rho * v[3]
        lagr[4] = 2 * v[4]
        lagr[5] = tau * v[6]
        lagr[6] = np.sum(lagr[0:5])
        return lagr

    # ------------------------------------------------------------------ ADMM
    def admm(self, data, h, e, psi, phi, lamd, mu, u, alpha, piter, titer, niter, model,
             lagr_every=10, verbose=True, rho=0.5, tau=0.5, m0=0, Ru=None, callback=None,
             graph=False):
        """solver.py:308-336.  Returns (u, psi) like the reference.

        Each iteration is enqueued on the device without host round trips:
        step lengths, Dai-Yuan coefficients, the takexi phase and the penalty
        update are computed by device kernels, and the state is updated in
        place in buffers owned by this call (the caller's arrays are not
        modified).  One synchronisation per iteration reads the steps and
        penalties into ``self.history``.  With ``graph=True`` the steady-state
        iteration (m >= 2, piter CG iterations) is captured once as a HIP
        graph and replayed.

        Beyond the reference: the full final state (h, e, psi, phi, lamd, mu,
        u, rho, tau, Ru) is kept in ``self.state``; ``rho``, ``tau``, ``m0``
        (index of the first iteration, which sets the piter+32 schedule of
        the first two iterations and the Lagrangian cadence) and ``Ru``
        (R u of the initial u) resume a run exactly where ``self.state`` left
        it.  ``callback(m, state)`` is called after every iteration with the
        live state buffers.
        """
        data = self._dev_data(data)
        ctx = self._admm_setup(h, e, psi, phi, lamd, mu, u, rho, tau, Ru, piter, titer)
        self.history = []
        graph_obj = None
        # graph capture uses a side stream; the whole run is enqueued on one
        # dedicated stream so that the library's per-stream workspaces are
        # sized by the eager iterations before the capture
        side = None
        scope = contextlib.nullcontext()
        if graph:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            scope = torch.cuda.stream(side)
        with scope:
            for m in range(m0, m0 + niter):
                if graph and m >= 2 and m > m0:
                    if graph_obj is None:
                        side.synchronize()
                        graph_obj = torch.cuda.CUDAGraph()
                        with torch.cuda.graph(graph_obj, stream=side):
                            self._admm_step(ctx, data, m, piter, titer, alpha, model)
                    graph_obj.replay()
                else:
                    self._admm_step(ctx, data, m, piter, titer, alpha, model)
                rec = self._admm_record(ctx, data, m, piter, titer, alpha, model, lagr_every,
                                        verbose, niter)
                if callback is not None:
                    S = ctx["S"]
                    callback(m, dict(h=S["h"], e=S["e"], psi=S["psi"], phi=S["phi"],
                                     lamd=S["lamd"], mu=S["mu"], u=S["u"], rho=rec["rho"],
                                     tau=rec["tau"], Ru=S["Ru"]))
        if side is not None:
            torch.cuda.current_stream().wait_stream(side)
        self._admm_finish(ctx, m0 + niter)
        return ctx["S"]["u"], ctx["S"]["psi"]

    # ------------------------------------------------------------------ ADMM pieces
    def _admm_setup(self, h, e, psi, phi, lamd, mu, u, rho, tau, Ru, piter, titer):
        """State buffers owned by one run (copies of the inputs), the device
        scalar block and the step history buffers."""
        S = {k: to_dev(v, c64).clone() for k, v in
             dict(h=h, e=e, psi=psi, phi=phi, lamd=lamd, mu=mu, u=u).items()}
        S["Ru"] = self.fwd_tomo_batch(S["u"]) if Ru is None else to_dev(Ru, c64).clone()
        S["xi0"], S["K"], S["xi1"] = empty(S["psi"].shape), empty(S["psi"].shape), \
            empty(S["phi"].shape)
        H = {"pg": torch.zeros((piter + 32, self.nchunk), dtype=f64, device=device()),
             "tg": torch.zeros(max(titer, 1), dtype=f64, device=device()),
             "rt": torch.zeros(2, dtype=f64, device=device())}
        return dict(S=S, blk=self._scalar_block(rho, tau), H=H)

    def _admm_step(self, ctx, data, m, piter, titer, alpha, model):
        pit = piter + (m < 2) * 32      # solver.py:315 (L6)
        self._admm_iter(ctx["S"], ctx["blk"], ctx["H"], data, pit, titer, alpha, model)

    def _admm_record(self, ctx, data, m, piter, titer, alpha, model, lagr_every, verbose,
                     niter):
        """Read one iteration's steps and penalties (one synchronisation), the
        Lagrangian every lagr_every iterations; appends to self.history."""
        S, blk, H = ctx["S"], ctx["blk"], ctx["H"]
        pit = piter + (m < 2) * 32
        v = torch.cat([H["rt"], blk[:_NSC], H["tg"], H["pg"][:pit].reshape(-1)]).cpu().numpy()
        rho_used, tau_used = float(v[0]), float(v[1])
        b = v[2:2 + _NSC]
        rho, tau = float(b[_RHO]), float(b[_TAU])
        tg = v[2 + _NSC:2 + _NSC + H["tg"].numel()][:titer]
        pg = v[2 + _NSC + H["tg"].numel():].reshape(pit, self.nchunk)
        if b[_MAXANG] > 3.14:
            print('possible phase wrap, max computed angle', float(b[_MAXANG]), file=sys.stderr)
        rec = {"m": m, "rho_used": rho_used, "tau_used": tau_used, "pshift": float(b[_PRM]),
               "ptycho_gammas": [[float(x) for x in pg[:, s]] for s in range(self.nchunk)],
               "tomo_gammas": [float(x) for x in tg], "rho": rho, "tau": tau,
               "max_angle": float(b[_MAXANG])}
        self._chunk_gammas, self._last_tomo_gammas = rec["ptycho_gammas"], rec["tomo_gammas"]
        if lagr_every and np.mod(m, lagr_every) == 0:
            lagr = self.take_lagr(S["psi"], S["phi"], data, S["h"], S["e"], S["lamd"], S["mu"],
                                  alpha, rho, tau, model)
            rec["lagr"] = [float(x) for x in lagr]
            if verbose:
                print("%d/%d) rho=%.2e, tau=%.2e, Lagrangian terms:  %.2e %.2e %.2e %.2e %.2e %.2e, Sum: %.2e" %
                      (m, niter, rho, tau, *lagr))
        self.history.append(rec)
        return rec

    def _admm_finish(self, ctx, m_next):
        S, blk = ctx["S"], ctx["blk"]
        rho, tau = (float(x) for x in blk[_RHO:_TAU + 1].cpu().numpy())
        self.state = dict(h=S["h"], e=S["e"], psi=S["psi"], phi=S["phi"], lamd=S["lamd"],
                          mu=S["mu"], u=S["u"], rho=rho, tau=tau, Ru=S["Ru"], m=m_next)

    def _admm_iter(self, S, blk, H, data, pit, titer, alpha, model):
        """One ADMM iteration (solver.py:312-330) on the state S in place, all
        scalars on the device (blk), steps recorded into H."""
        mdl = _lib.PT_MODEL[model]
        for req in self._admm_iter_gen(S, blk, H, data, pit, titer, alpha):
            run_ptycho_request(req, mdl, stream())

    def _admm_iter_gen(self, S, blk, H, data, pit, titer, alpha):
        """_admm_iter as a generator of the ptychography CG's heavy launch
        requests (see _cg_ptycho_gen), then ("end",) once the ptychography
        subproblem is enqueued."""
        st = stream()
        H["rt"].copy_(blk[_RHO:_TAU + 1])
        yield from self._cg_ptycho_gen(self._ptycho, self.nchunk, data, S["psi"], S["h"],
                                       S["lamd"], blk, pit, float(self.coefdata), H["pg"])
        yield ("end",)                  # the ptychography subproblem is enqueued
        st = stream()                   # the caller may continue on another stream
        self._takexi_dev(S["psi"], S["phi"], S["lamd"], S["mu"], blk, S["xi0"], S["K"], S["xi1"])
        self._cg_tomo_dev(S["xi0"], S["xi1"], S["K"], S["u"], S["Ru"], blk, titer, H["tg"])
        u = S["u"]
        # h = exptomo(fwd_tomo_batch(u)) * exp(i pshift) (solver.py:323): R u of
        # the new u is transformed afresh (the CG recursion's R u + g R d drifts
        # by FP32 rounding over many iterations) and carried into the next
        # iteration's cg_tomo
        self._tomo.fwd_scaled(S["Ru"].data_ptr(), u.data_ptr(), float(self.coeftomo))
        # phi, h, e, lamd += rho (h - psi), mu += tau (e - phi) and the residuals of
        # the penalty update (solver.py:320-330), each state read and written once
        c = self.voxelsize * self.wavenumber() / float(self.coeftomo)
        _call("pt_k_object_update", _dp(blk, _NORMS), ptr(S["h"]), ptr(S["lamd"]), ptr(S["psi"]),
              ptr(S["Ru"]), c, _dp(blk, _PRM), _dp(blk, _RHO), S["h"].numel(), st)
        _call("pt_k_split_update", _dp(blk, _NORMS + 2), ptr(S["phi"]), ptr(S["e"]), ptr(S["mu"]),
              ptr(u), _dp(blk, _TAU), float(alpha), *u.shape, st)
        _call("pt_k_penalty", _dp(blk, _RHO), _dp(blk, _NORMS), st)

    def admm_resume(self, data, alpha, piter, titer, niter, model, **kw):
        """Continue from ``self.state`` (checkpoint/resume of the full state)."""
        s = self.state
        return self.admm(data, s["h"], s["e"], s["psi"], s["phi"], s["lamd"], s["mu"], s["u"],
                         alpha, piter, titer, niter, model, rho=s["rho"], tau=s["tau"],
                         m0=s["m"], Ru=s["Ru"], **kw)


def run_ptycho_request(req, mdl, st):
    """Make one heavy launch request of _cg_ptycho_gen with the single-instance
    entry points."""
    if req[0] == "end":
        return
    a = req[1]
    if req[0] == "grad":
        _call("pt_ptycho_grad", a.h, a.grad, a.psi, a.data, a.hh, a.lamd, a.rho, a.rho_dev,
              a.coefptycho, a.coefdata, mdl, st)
    else:
        nxt, step, weights, ng_next, last = req[3]
        _call("pt_ptycho_linesearch_sweep", a, nxt, step, weights, req[2], ng_next, last, mdl, st)


def _dp(t, k=0):
    """device address of element k of a float64 tensor"""
    return ctypes.c_void_p(t.data_ptr() + 8 * k)
