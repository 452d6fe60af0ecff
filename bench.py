#!/usr/bin/env python
"""Benchmark: plain ADMM iterations per second for joint ptycho-tomography on
one MI355X (256^3 object, 384 angles, 16x16 probe, scan step 4, Poisson
data at 1e3 photons; piter = titer = 4).

A step is one ADMM outer iteration (cg_ptycho over all angle chunks,
takexi, cg_tomo, solve_reg, h/e/dual/penalty updates, Lagrangian every 10
iterations as in the reference), with all inputs resident in HBM.  W warm-up
iterations (including the two piter+32 iterations of the reference
schedule) precede K timed iterations.

Prints one JSON line (--full: the whole record to a file) with the headline number, the roofline of the dominant
kernel (HIP events around each of its launches inside the timed region), the
whole-volume operators' rates (tomography and ptychography forward/adjoint,
GB/s against HBM, and against the same operators on the host) and the CPU
baseline (the NumPy restatement of the reference operators on a bounded
sample, run on this host's cores).
"""
import argparse
import ctypes
import json
import math
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

HBM_PEAK_GBS = 8000.0
FP32_VECTOR_PEAK_GFLOPS = 157300.0
BF16_MFMA_PEAK_FLOPS = 2.5e15


def kernel_bytes(tag, slv):
    """Algorithmic HBM bytes of one launch of kernel `tag` (each input and
    output counted once)."""
    n, nz, nt = slv.n, slv.nz, slv.ntheta
    N = 3 * n // 2
    S, D = slv.nscan, slv.ndety
    vol_t = 8 * nt * nz * n            # psi-sized complex64 array
    # the samples' disc of the forward's 2N x 2N and the adjoint's 2n x 2n grid
    disc_f, disc_a = 8 * math.pi * N ** 2 * nz, 8 * math.pi * n ** 2 * nz
    samples = 8 * nt * N * nz          # polar samples
    if tag == "tomo_gather":            # grid in, polar samples out
        return disc_f + samples
    if tag == "tomo_line_idft":         # polar samples in, cropped projections out
        return samples + vol_t
    if tag == "tomo_adj_line":          # projections in, polar samples out
        return vol_t + samples
    if tag == "tomo_scatter":           # polar samples in, grid out
        return samples + disc_a
    if tag == "ptycho_grad_tile":       # psi in, data in, one psi-sized result out
        return vol_t + 4 * nt * S * D * D + vol_t
    if tag == "ptycho_minf":            # psi, d, h, lamd and data in (data and rho terms)
        return 4 * vol_t + 4 * nt * S * D * D
    if tag == "tomo_row_fwd":           # object in, N x 2N out
        return 8 * n * n * nz + 8 * N * 2 * N * nz
    if tag == "tomo_col_fwd":           # N x 2N in, grid out
        return 8 * N * 2 * N * nz + disc_f
    if tag == "tomo_col_adj":           # grid in, n x 2n out
        return disc_a + 8 * n * 2 * n * nz
    if tag == "tomo_row_adj":           # n x 2n in, object out
        return 8 * n * 2 * n * nz + 8 * n * n * nz
    return None


def minf_work(history, nchunk, piter):
    """Chunk evaluations done by the ptychography line-search kernel over
    `history` (one ADMM iteration per record).  A sweep evaluates every chunk
    whose search is still open (finished chunks exit at once), so the number
    of sweeps a chunk took follows from its accepted step: the search starts
    at 2 (then at the previous step) and tries the halvings of the solver's
    sweep schedule in order (the first CG step's schedule, then the later
    steps'); a step reaching 1e-12 ends at 0.  Also returns the number of
    Lagrangian evaluations (launched under their own tag)."""
    from ptychotomo_amd.solver import _PSCHED_FIRST, _PSCHED_LATER

    def nsweeps(k, sched):
        done = 0
        for s, n in enumerate(sched):
            done += n
            if k < done:
                return s + 1
        return len(sched)

    sweeps, lagr = 0, 0
    for rec in history:
        if rec.get("lagr"):
            lagr += 1
        for chunk_g in rec["ptycho_gammas"]:
            g0 = 2.0
            for i, g in enumerate(chunk_g):
                if g0 <= 1e-12:
                    k = 0
                elif g > 0:
                    k = int(round(math.log2(g0 / g)))
                else:
                    k = math.ceil(math.log2(g0 / 1e-12))
                sweeps += nsweeps(k, _PSCHED_FIRST if i == 0 else _PSCHED_LATER)
                g0 = g
    return sweeps, lagr


WARM_WEIGHTS = os.path.join(HERE, "ptychotomo_amd", "weights", "unet_warmstart_128.npz")

TAGS = ["tomo_row_fwd", "tomo_col_fwd", "tomo_gather", "tomo_line_idft", "tomo_adj_line",
        "tomo_scatter", "tomo_scatter_fix", "tomo_col_adj", "tomo_row_adj", "ptycho_grad_tile",
        "ptycho_fold", "ptycho_minf"]
GATHER_TAPS = 64        # 8 x 8 Kaiser-Bessel taps per polar sample and slice


def prof_run(lib, tag, fn):
    lib.pt_prof_start(tag.encode())
    fn()
    tot = ctypes.c_double()
    cnt = ctypes.c_long()
    lib.pt_prof_stop(ctypes.byref(tot), ctypes.byref(cnt))
    return tot.value, cnt.value


def cpu_baseline(w, budget_s=30.0):
    """NumPy/SciPy restatement of the reference operators (oracle) timed on a
    bounded sample of the workload and scaled to one reference ADMM
    iteration: 9 USFFT forward + 4 adjoint per iteration (cg_tomo with titer
    = 4 plus the h update), and per ptychography CG iteration 2 forward, 1
    adjoint and 3 far-field residual/functional passes (solver.py:206-242)."""
    import scipy.fft  # noqa: F401
    from oracle import ptycho as optycho
    from oracle import usfft as ousfft
    from ptychotomo_amd import synthetic
    cores = len(os.sched_getaffinity(0))
    theta, prb, scan, obj = synthetic.make_inputs(w)
    rng = np.random.default_rng(0)
    pz = 8
    t0 = time.perf_counter()
    ousfft.interp_matrix(theta, w.n)  # geometry set-up, not counted
    t_setup = time.perf_counter() - t0
    u = obj[:pz]
    t0 = time.perf_counter()
    g = ousfft.fwd(u, theta, workers=cores)
    t_tf = (time.perf_counter() - t0) * (w.nz / pz)
    t0 = time.perf_counter()
    ousfft.adj(g, theta, workers=cores)
    t_ta = (time.perf_counter() - t0) * (w.nz / pz)
    na = 32
    psi = np.exp(1j * 1e-2 * rng.standard_normal((na, w.nz, w.n))).astype(np.complex64)
    sc = scan[:, :na]
    t0 = time.perf_counter()
    far = optycho.fwd(psi, prb, sc, w.det, w.det)
    t_pf = (time.perf_counter() - t0) * (w.ntheta / na)
    t0 = time.perf_counter()
    optycho.adj(far, prb, sc, w.nz, w.n)
    t_pa = (time.perf_counter() - t0) * (w.ntheta / na)
    d = np.abs(far) ** 2
    t0 = time.perf_counter()
    r = far - d * far / (np.abs(far) ** 2 + 1e-32)
    f = np.sum(np.abs(far) ** 2 - 2 * d * np.log(np.maximum(np.abs(far), 1e-32)))
    del r, f
    t_pr = (time.perf_counter() - t0) * (w.ntheta / na)
    per_iter = cpu_iteration_seconds(
        {"usfft_fwd": t_tf, "usfft_adj": t_ta, "ptycho_fwd": t_pf, "ptycho_adj": t_pa,
         "ptycho_residual": t_pr}, w.piter)
    return {"value": 1.0 / per_iter, "unit": "ADMM iters/s", "cores": cores, "kind": "port",
            "sample": (f"oracle NumPy/SciPy FP32 restatement at {w.n}^3/{w.ntheta} angles: USFFT "
                       f"fwd+adj on {pz} slices (x{w.nz // pz}), ptychography fwd+adj+residual "
                       f"on {na} angles (x{w.ntheta // na}), composed to one reference ADMM "
                       f"iteration (9 USFFT fwd, 4 adj, piter x (2 fwd, 1 adj, 3 residual "
                       f"passes)); interpolation-matrix set-up {t_setup:.1f}s excluded"),
            "seconds_per_iter": per_iter,
            "op_seconds": {"usfft_fwd": t_tf, "usfft_adj": t_ta, "ptycho_fwd": t_pf,
                           "ptycho_adj": t_pa, "ptycho_residual": t_pr}}


def cpu_iteration_seconds(op, piter, titer=4):
    """One reference ADMM iteration composed from host operator times: cg_tomo
    with titer iterations (2 forward USFFTs and 1 adjoint each) plus the h
    update's forward, and per ptychography CG iteration 2 forward, 1 adjoint
    and 3 far-field residual/functional passes (solver.py:180-242, 323)."""
    return ((2 * titer + 1) * op["usfft_fwd"] + titer * op["usfft_adj"] +
            piter * (2 * op["ptycho_fwd"] + op["ptycho_adj"] + 3 * op["ptycho_residual"]))


def config0_rates(log):
    """The 64^3 / 96-angle workload's 32 ADMM iterations (the first two with
    piter + 32 CG steps) on the GPU, timed whole, against the same 32
    iterations on the host composed from the oracle's operator times on this
    host's cores (whole volume: the oracle runs it in seconds per operator)."""
    import torch
    from ptychotomo_amd import synthetic
    w = synthetic.CONFIGS["plain64"]
    slv, data, obj = synthetic.make_workload(w)
    st = synthetic.initial_state(w)
    run = dict(alpha=w.alpha, piter=w.piter, titer=w.titer, model=w.model, verbose=False)
    slv.admm(data, st["h"], st["e"], st["psi"], st["phi"], st["lamd"], st["mu"], st["u"],
             niter=2, lagr_every=10, **run)          # warm-up (library workspaces)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    slv.admm(data, st["h"], st["e"], st["psi"], st["phi"], st["lamd"], st["mu"], st["u"],
             niter=w.niter, lagr_every=10, **run)
    torch.cuda.synchronize()
    gpu_s = time.perf_counter() - t0
    cb = cpu_baseline(w)
    op = cb["op_seconds"]
    cpu_s = (2 * cpu_iteration_seconds(op, w.piter + 32) +
             (w.niter - 2) * cpu_iteration_seconds(op, w.piter))
    log(f"64^3: GPU {gpu_s:.3f}s, host {cpu_s:.1f}s for {w.niter} iterations")
    del slv, data
    torch.cuda.empty_cache()
    return {"workload": w.name, "iterations": w.niter, "gpu_s": gpu_s,
            "gpu_iters_per_s": w.niter / gpu_s, "cpu_s": cpu_s,
            "cpu_iters_per_s": w.niter / cpu_s, "cpu_cores": cb["cores"],
            "cpu_kind": "port (oracle FP32 restatement; operator times composed into the 32 "
                        "iterations' schedule)", "vs_cpu": cpu_s / gpu_s}


def kernel_rates(slv, breakdown):
    """Per-launch rates of the probed kernels: algorithmic GB/s against HBM
    and, for the USFFT gather (4 flops per complex x real tap, GATHER_TAPS per
    sample and slice), GFLOP/s against the FP32 vector peak.  The line-search
    kernel's rate is per full sweep (its launches include sweeps in which
    finished chunks exit at once)."""
    out = {}
    N = 3 * slv.n // 2
    for tag, b in breakdown.items():
        nb = kernel_bytes(tag, slv)
        if not nb or not b["launches"]:
            continue
        ms = b["ms_per_iter"] / b["launches"]
        r = {"avg_ms": ms, "algorithmic_bytes": nb, "GB_s": nb / (ms * 1e-3) / 1e9}
        if "full_sweeps" in b:
            # per full sweep (nb is a full sweep's bytes), not per launch
            ms = b["ms_per_iter"] / max(b["full_sweeps"], 1e-9)
            r = {"ms_per_full_sweep": ms, "full_sweeps": b["full_sweeps"], "launches": b["launches"],
                 "algorithmic_bytes": nb, "GB_s": nb / (ms * 1e-3) / 1e9}
        r["frac_hbm"] = r["GB_s"] / HBM_PEAK_GBS
        if tag == "tomo_gather":
            fl = 4.0 * GATHER_TAPS * slv.ntheta * N * slv.nz
            r["flops"] = fl
            r["GFLOP_s"] = fl / (ms * 1e-3) / 1e9
            r["frac_fp32_vector"] = r["GFLOP_s"] / FP32_VECTOR_PEAK_GFLOPS
        out[tag] = r
    return out


def unet_rates(n=128, reps=5):
    """The warm-start U-Net's convolutions at n^3 (the 2-channel input of the
    128^3 workload): per layer the forward launch time (median of `reps`,
    HIP events on the launch stream) and TFLOP/s at 2 * V * Cout * 27 * Cin
    flops against the 2.5 PFLOP/s dense bf16 MFMA peak, and one training step
    (forward, backward, Adam)."""
    import torch
    from ptychotomo_amd import unet
    net = unet.UNet3D(seed=0)
    x = torch.randn((n, n, n, 2), dtype=torch.float32, device="cuda") * 0.1
    net.forward(x)                       # buffers, activations
    torch.cuda.synchronize()
    d1 = (n, n, n)
    dims = {"e1a": d1, "e1b": d1, "e2a": tuple(v // 2 for v in d1),
            "e2b": tuple(v // 2 for v in d1), "bna": tuple(v // 4 for v in d1),
            "bnb": tuple(v // 4 for v in d1), "d2a": tuple(v // 2 for v in d1),
            "d2b": tuple(v // 2 for v in d1), "d1a": d1, "d1b": d1}
    inputs = {"e1a": "x", "e1b": "e1a", "e2a": "p1", "e2b": "e2a", "bna": "p2", "bnb": "bna",
              "d2a": "cat2", "d2b": "d2a", "d1a": "cat1", "d1b": "d1a"}
    layers = {}
    tot_fl, tot_ms = 0.0, 0.0
    for name in unet.CONVS:
        co, ci = net.shapes[name]
        xin = net._buf[inputs[name]]
        ms = []
        for _ in range(reps + 1):
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ev[0].record()
            net._conv(name, xin, dims[name], "bench_out")
            ev[1].record()
            ev[1].synchronize()
            ms.append(ev[0].elapsed_time(ev[1]))
        t = float(np.median(ms[1:]))
        V = dims[name][0] * dims[name][1] * dims[name][2]
        fl = 2.0 * V * co * 27 * ci
        tot_fl += fl
        tot_ms += t
        layers[name] = {"cin": ci, "cout": co, "ms": t, "TFLOP_s": fl / (t * 1e-3) / 1e12,
                        "frac_bf16_peak": fl / (t * 1e-3) / BF16_MFMA_PEAK_FLOPS}
    y = torch.randn_like(x) * 0.1
    net.train_step(x, y)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(3):
        net.train_step(x, y)
    torch.cuda.synchronize()
    step_ms = (time.perf_counter() - t0) / 3 * 1e3
    return {"n": n, "layers": layers, "forward_conv_ms": tot_ms,
            "forward_conv_TFLOP_s": tot_fl / (tot_ms * 1e-3) / 1e12,
            "forward_conv_frac_bf16_peak": tot_fl / (tot_ms * 1e-3) / BF16_MFMA_PEAK_FLOPS,
            "train_step_ms": step_ms}


def batch_rates(niter=6, log=None):
    """The batched workload: 16 reconstructions of n in {64, 96, 128, 192} (4
    each, ntheta = 1.5 n, 16 x 16 probe, step 4, seeds 100 + i), USFFT launch
    shapes from the autotuner (which leaves these sizes' register line FFT
    passes alone), advanced together by BatchSolver -- the
    ptychography CG's heavy launches grouped over all instances, the rest on
    per-instance streams; and without grouping, eagerly and as one graph per
    iteration -- against the same instances run one after the other.  All
    timed over `niter` iterations from the same state after a warm-up."""
    import tempfile
    import torch
    from ptychotomo_amd import synthetic
    from ptychotomo_amd.batch import BatchSolver
    sizes = [64, 96, 128, 192] * 4
    made = []
    for i, n in enumerate(sizes):
        w = synthetic.Workload(f"batch {n}", n, n, 3 * n // 2, 20, ptheta=16, seed=100 + i)
        made.append((w,) + synthetic.make_workload(w))
    w0 = made[0][0]
    kw = dict(alpha=w0.alpha, piter=w0.piter, titer=w0.titer, model=w0.model)
    t0 = time.perf_counter()
    with tempfile.TemporaryDirectory() as tmp:
        bs = BatchSolver([m[1] for m in made], tune=True, tune_cache=os.path.join(tmp, "t.json"))
    t_tune = time.perf_counter() - t0
    datas = [m[2] for m in made]
    # warm-up: the first iterations (piter + 32 CG steps)
    bs.admm(datas, [synthetic.initial_state(m[0]) for m in made], niter=3, lagr_every=0, **kw)
    states = [dict(s.state) for s in bs.solvers]

    def timed(fn):
        torch.cuda.synchronize()
        t = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        return time.perf_counter() - t

    modes = {}
    for name, opts in (("grouped", dict(grouped=True, graph=False)),
                       ("streams", dict(grouped=False, graph=False)),
                       ("streams_graph", dict(grouped=False, graph=True))):
        modes[name] = timed(lambda: bs.admm(datas, [dict(s) for s in states], niter=niter,
                                            lagr_every=0, m0=3, **opts, **kw))

    def singles():
        for s, st, d in zip(bs.solvers, states, datas):
            s.state = dict(st)
            s.admm_resume(d, niter=niter, lagr_every=0, **kw)
    t_single = timed(singles)
    if log:
        log(f"batch of {len(sizes)}: {modes}, one after the other {t_single:.3f}s")
    t_batch = modes["grouped"]
    return {"instances": len(sizes), "sizes": sorted(set(sizes)), "iterations": niter,
            "tuned_shapes": {str(n): list(sh) for n, sh in zip(sizes, bs.tuning)},
            "tune_s": t_tune, "batch_s": t_batch, "batch_iters_per_s": niter / t_batch,
            "modes_s": modes, "single_runs_s": t_single,
            "speedup_over_single_runs": t_single / t_batch}


def operator_rates(slv, reps=5):
    """The workload's whole-volume operators as the solver calls them
    (tomography forward and adjoint, ptychography forward to the far field
    and adjoint, scaled by coeftomo / coefptycho): median of `reps` calls
    after one untimed call, HIP events on the launch stream; algorithmic
    bytes = the input read and the output written once."""
    import torch
    n, nz, nt = slv.n, slv.nz, slv.ntheta
    S, D = slv.nscan, slv.ndety
    c64 = torch.complex64
    gen = torch.Generator(device="cuda").manual_seed(0)
    u = torch.randn((nz, n, n), dtype=c64, device="cuda", generator=gen)
    g = torch.randn((nt, nz, n), dtype=c64, device="cuda", generator=gen)
    u2, g2 = torch.empty_like(u), torch.empty_like(g)
    far = torch.empty((nt, S, D, D), dtype=c64, device="cuda")
    ct, cp = float(slv.coeftomo), float(slv.coefptycho)
    tomo_b = 8 * (nz * n * n + nt * nz * n)
    ptycho_b = 8 * nt * nz * n + 8 * nt * S * D * D
    ops = {
        "tomo_fwd": (lambda: slv._tomo.fwd_scaled(g2.data_ptr(), u.data_ptr(), ct), tomo_b),
        "tomo_adj": (lambda: slv._tomo.adj_scaled(u2.data_ptr(), g.data_ptr(), ct), tomo_b),
        "ptycho_fwd": (lambda: slv._ptycho.fwd_scaled(far.data_ptr(), g.data_ptr(), cp),
                       ptycho_b),
        "ptycho_adj": (lambda: slv._ptycho.adj_scaled(g2.data_ptr(), far.data_ptr(), cp),
                       ptycho_b),
    }
    out = {}
    for name, (fn, nbytes) in ops.items():
        fn()
        ms = []
        for _ in range(reps):
            ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ev[0].record()
            fn()
            ev[1].record()
            ev[1].synchronize()
            ms.append(ev[0].elapsed_time(ev[1]))
        t = float(np.median(ms))
        out[name] = {"ms": t, "algorithmic_bytes": nbytes, "GB_s": nbytes / (t * 1e-3) / 1e9,
                     "frac_hbm": nbytes / (t * 1e-3) / 1e9 / HBM_PEAK_GBS}
    del u, g, u2, g2, far
    torch.cuda.empty_cache()
    return out


def main():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="prod256")
    ap.add_argument("--full", default=None, metavar="FILE",
                    help="also write the whole record (traces, per-seed runs) as JSON")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--breakdown", action="store_true", help="per-kernel time per iteration")
    ap.add_argument("--no-breakdown-probe", action="store_true",
                    help="skip the per-kernel probe iteration (short runs under counter collection)")
    ap.add_argument("--copy-calib", type=int, default=0, metavar="MIB",
                    help="only run 5 device copies of MIB MiB (HBM counter calibration)")
    ap.add_argument("--tol-run", type=int, default=0,
                    help="also run N plain iterations for time-to-Lagrangian-tolerance")
    ap.add_argument("--warm-weights", default=WARM_WEIGHTS,
                    help="U-Net weights: time plain ADMM and the learned warm start on the "
                         "--tol-n^3 warm-start workload (--tol-iters iterations each)")
    ap.add_argument("--tol-n", type=int, default=128,
                    help="size of the plain-vs-warm comparison (plain ADMM does not converge "
                         "on the 256^3 workload)")
    ap.add_argument("--tol-iters", type=int, default=100)
    ap.add_argument("--tol-seeds", type=int, default=7, help="held-out phantoms compared")
    ap.add_argument("--no-warm", action="store_true", help="skip the plain-vs-warm comparison")
    ap.add_argument("--no-config0", action="store_true",
                    help="skip the 64^3 32-iteration GPU-vs-host row")
    ap.add_argument("--no-unet", action="store_true", help="skip the U-Net convolution rates")
    ap.add_argument("--no-batch", action="store_true",
                    help="skip the 16-instance batched workload row")
    ap.add_argument("--unet-only", type=int, default=0, metavar="N",
                    help="only measure the U-Net convolutions at N^3 (profiling)")
    ap.add_argument("--no-operators", action="store_true",
                    help="skip the whole-volume operator rates (profiled runs of the iteration)")
    ap.add_argument("--kernel", default=None,
                    help="roofline kernel tag (default: the largest of the breakdown probe; "
                         "ptycho_minf without the probe)")
    args = ap.parse_args()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus > 1 or world > 1:
        print(json.dumps({"error": "one GPU only: the ADMM path would shard over angle "
                                   "chunks (ptychography) and slice blocks (tomography), "
                                   "which is not built",
                          "n_gpus": max(args.gpus, world)}))
        sys.exit(2)

    import torch
    from ptychotomo_amd import _lib, synthetic

    if args.copy_calib:
        nbytes = args.copy_calib << 20
        a = torch.ones(nbytes // 4, dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        for _ in range(5):
            b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"copy_calib_bytes_read": nbytes, "copy_calib_bytes_written": nbytes,
                          "copies": 5}), flush=True)
        return

    if args.unet_only:
        print(json.dumps({"unet": unet_rates(args.unet_only)}), flush=True)
        return

    w = synthetic.CONFIGS[args.workload]
    log = lambda msg: print(f"[bench] {msg}", file=sys.stderr, flush=True)
    log(f"workload {args.workload}: generating data")
    t0 = time.perf_counter()
    slv, data, obj = synthetic.make_workload(w)
    torch.cuda.synchronize()
    t_gen = time.perf_counter() - t0
    st0 = synthetic.initial_state(w)
    run = dict(alpha=w.alpha, piter=w.piter, titer=w.titer, model=w.model, verbose=False)

    log(f"data ready in {t_gen:.1f}s; warm-up {args.warmup} iterations")
    # warm-up: includes the two piter+32 iterations of the reference schedule
    slv.admm(data, st0["h"], st0["e"], st0["psi"], st0["phi"], st0["lamd"], st0["mu"],
             st0["u"], niter=args.warmup, lagr_every=10, **run)
    torch.cuda.synchronize()

    # dominant kernel from a per-kernel breakdown over one (untimed) iteration
    lib = _lib.lib
    saved = dict(slv.state)
    breakdown = {}
    probe = TAGS if args.breakdown else ["tomo_gather", "tomo_scatter", "ptycho_grad_tile",
                                         "ptycho_minf"]
    for tag in ([] if args.no_breakdown_probe else probe):
        slv.state = dict(saved)
        ms, cnt = prof_run(lib, tag, lambda: slv.admm_resume(data, niter=1, lagr_every=10, **run))
        breakdown[tag] = {"ms_per_iter": ms, "launches": cnt}
        if tag == "ptycho_minf":
            # line-search sweeps: chunks whose search has ended exit at once
            breakdown[tag]["full_sweeps"] = minf_work(slv.history, slv.ntheta // slv.ptheta,
                                                      w.piter)[0] / (slv.ntheta // slv.ptheta)
    slv.state = dict(saved)
    dom = args.kernel or (max(breakdown, key=lambda k: breakdown[k]["ms_per_iter"])
                          if breakdown else "ptycho_minf")
    log(f"breakdown {breakdown}; timing {args.steps} iterations, roofline kernel {dom}")

    # timed region
    torch.cuda.synchronize()
    lib.pt_prof_start(dom.encode())
    t0 = time.perf_counter()
    slv.admm_resume(data, niter=args.steps, lagr_every=10, **run)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    tot = ctypes.c_double()
    cnt = ctypes.c_long()
    lib.pt_prof_stop(ctypes.byref(tot), ctypes.byref(cnt))
    avg_ms = tot.value / max(cnt.value, 1)
    nbytes = kernel_bytes(dom, slv)
    achieved = nbytes / (avg_ms * 1e-3) / 1e9 if nbytes else None
    work = None
    if dom == "ptycho_minf":
        # its launches are line-search sweeps; chunks whose search has ended
        # exit at once, so count the chunk evaluations actually done
        nchunk = slv.ntheta // slv.ptheta
        ev, nl = minf_work(slv.history, nchunk, w.piter)
        vol_t = 8 * slv.ntheta * slv.nz * slv.n
        dat = 4 * slv.ntheta * slv.nscan * slv.ndety * slv.ndety
        done = ev * (4 * vol_t + dat) / nchunk
        achieved = done / (tot.value * 1e-3) / 1e9
        work = {"chunk_evaluations": ev, "lagrangian_passes": nl, "nchunk": nchunk,
                "full_sweeps": ev / nchunk, "bytes_done": done,
                "bytes_per_launch": done / max(cnt.value, 1)}
        nbytes = done / max(cnt.value, 1)
    traffic = None
    tf = os.path.join(HERE, "profiles", f"{dom}_{args.workload}_traffic.txt")
    if os.path.exists(tf):
        with open(tf) as fh:
            for line in fh:
                if line.startswith("hbm_bytes_per_launch:") and dom != "ptycho_minf":
                    traffic = float(line.split(":", 1)[1])
                if line.startswith("hbm_bytes_per_full_sweep:") and work:
                    # per launch on the basis of this run's sweeps
                    traffic = float(line.split(":", 1)[1]) * work["full_sweeps"] / max(cnt.value, 1)
                if line.startswith("valu_wave_instructions_per_full_sweep:") and work:
                    # the kernel's actual bound: FP32 vector issue (4 cycles per wave
                    # instruction per SIMD, 1024 SIMDs at 2.4 GHz)
                    ins = float(line.split(":", 1)[1]) * work["full_sweeps"]
                    bound_ms = ins * 4 / (1024 * 2.4e9) * 1e3
                    work["valu_issue"] = {"wave_instructions": ins, "bound_ms": bound_ms,
                                          "frac": bound_ms / tot.value}

    out = {
        "metric": "ADMM iters/s + time-to-Lagrangian-tol, 256^3, plain vs warm-start, 1 MI355X",
        "value": args.steps / dt,
        "unit": "ADMM iters/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": dt / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "c64 (fp32 complex), fp64 reductions",
        "data": "synthetic (seeded ellipsoid phantom, Poisson counts)",
        "config": synthetic.CONFIGS[args.workload].describe() | {"parallelism": "single GPU"},
        "roofline": {"kernel": dom, "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": (achieved / HBM_PEAK_GBS) if achieved else None,
                     "traffic": traffic, "algorithmic_bytes": nbytes, "avg_launch_ms": avg_ms,
                     "launches": cnt.value, "kernel_ms_total": tot.value, "work": work},
        "breakdown_ms_per_iter": {k: round(v["ms_per_iter"], 3) for k, v in breakdown.items()},
        "kernels": kernel_rates(slv, breakdown),
        "datagen_s": round(t_gen, 2),
    }
    valu = (work or {}).get("valu_issue")
    if valu:
        # the line-search kernel's limiter is FP32 vector issue, not HBM: its
        # wave instructions (SQ_INSTS_VALU per full sweep) against the issue
        # rate, beside the HBM fraction above
        out["roofline"]["limiter"] = "valu"
        out["roofline"]["valu"] = {"frac": valu["frac"], "bound_ms": valu["bound_ms"],
                                   "measured_ms": tot.value,
                                   "peak": "1024 SIMDs x 2.4 GHz / 4 cycles per wave64 op"}
    lag = [r.get("lagr") for r in slv.history if r.get("lagr")]
    if lag:
        out["lagr_last"] = lag[-1]
    if not args.no_operators:
        log("operator rates")
        out["operators"] = operator_rates(slv)
    if args.tol_run:
        out["time_to_tol"] = time_to_tol(slv, data, w, run, args.tol_run)
    if args.warm_weights and not args.no_warm and os.path.exists(args.warm_weights):
        from ptychotomo_amd import warmstart
        del slv, data
        torch.cuda.empty_cache()
        net = warmstart.load(args.warm_weights)
        # the headline workload itself: plain ADMM and the warm start (the
        # 128^3-trained network applied at 256^3), both criteria, with the
        # plain run's per-iteration record
        log(f"warm start on the {args.workload} workload: {args.tol_iters} iterations each")
        r = warmstart.compare(net, w, n_ref=args.tol_iters, n_max=args.tol_iters, tol=1e-3,
                              trace=True)
        tt = {"workload": r["workload"], "iterations": args.tol_iters,
              "lagrangian": r["lagrangian"], "object_error": r["object_error"],
              "fallback_to_plain": r["fallback_to_plain"],
              "plain_trace": r["plain_trace"], "warm_trace": r["warm_trace"]}
        log(f"warm start: plain vs U-Net at {args.tol_n}^3, {args.tol_iters} iterations each")
        runs = []
        for k in range(args.tol_seeds):   # held-out seeds (training used 0 .. pairs-1)
            wt = warmstart.workload(args.tol_n, seed=10_000 + args.tol_n + k, photons=1e3)
            runs.append(warmstart.compare(net, wt, n_ref=args.tol_iters, n_max=args.tol_iters,
                                          tol=1e-3))
        sp = [r["object_error"]["speedup"] for r in runs]
        out["time_to_tol"] = tt
        out["time_to_tol_warm128"] = {
            "workload": runs[0]["workload"], "seeds": args.tol_seeds,
            "criterion": "object error at the plain run's converged level (median of its last "
                         "10 iterations); the Lagrangian criterion is not reached by plain ADMM",
            "speedup_per_seed": sp,
            "reached": sum(1 for r in runs if not r["fallback_to_plain"]),
            "speedup_median": float(np.median(sp)),
            "lagrangian_reached": [r["lagrangian"]["reached"] for r in runs],
            "runs": runs}
    if not args.no_unet:
        log("U-Net convolution rates")
        out["unet"] = unet_rates()
    if not args.no_batch:
        log("batched workload: 16 instances")
        out["batch"] = batch_rates(log=log)
    if not args.no_config0 and not args.no_cpu_baseline:
        log("64^3 workload: 32 iterations, GPU and host")
        out["config0"] = config0_rates(log)
    if not args.no_cpu_baseline:
        log("cpu baseline")
        out["cpu_baseline"] = cpu_baseline(w)
        # the same operators on the host (whole-volume times scaled from the
        # bounded sample)
        cs = out["cpu_baseline"]["op_seconds"]
        for name, key in (() if args.no_operators else
                          (("tomo_fwd", "usfft_fwd"), ("tomo_adj", "usfft_adj"),
                           ("ptycho_fwd", "ptycho_fwd"), ("ptycho_adj", "ptycho_adj"))):
            out["operators"][name]["cpu_ms"] = cs[key] * 1e3
            out["operators"][name]["vs_cpu"] = cs[key] * 1e3 / out["operators"][name]["ms"]
    if args.full:
        with open(args.full, "w") as fh:
            json.dump(out, fh)
    print(result_line(out), flush=True)


def result_line(out):
    """The JSON line of a record: strict JSON, five digits per number, and
    without the lists that only a closer look needs (the iterations' traces, the
    per-seed runs, the network's layers beyond their rates), so that it stays well
    under 8 KB; --full keeps everything."""
    def short(v):
        if isinstance(v, dict):
            return {k: short(x) for k, x in v.items() if k not in ("plain_trace", "warm_trace",
                                                                   "runs")}
        if isinstance(v, (list, tuple)):
            return [short(x) for x in v]
        if isinstance(v, float):
            return float(f"{v:.5g}") if math.isfinite(v) else None
        return v
    res = short(out)
    for k in ("value", "ms_per_step"):
        res[k] = out[k]
    if "unet" in res:
        res["unet"]["layers"] = {k: v["TFLOP_s"] for k, v in res["unet"]["layers"].items()}
    return json.dumps(res, allow_nan=False)


def time_to_tol(slv, data, w, run, niter, tol=1e-3):
    """Plain ADMM from the reference initial guess for `niter` iterations with
    the Lagrangian every iteration; time until lagr[6] stays within `tol`
    (relative) of its final value."""
    import torch
    from ptychotomo_amd import synthetic
    st = synthetic.initial_state(w)
    stamps = []

    def cb(m, s):
        torch.cuda.synchronize()
        stamps.append(time.perf_counter())

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    slv.admm(data, st["h"], st["e"], st["psi"], st["phi"], st["lamd"], st["mu"], st["u"],
             niter=niter, lagr_every=1, callback=cb, **run)
    lag = np.array([r["lagr"][6] for r in slv.history])
    final = lag[-1]
    ok = np.abs(lag - final) <= tol * abs(final)
    k = len(ok) - 1
    while k > 0 and ok[k - 1]:
        k -= 1
    return {"plain_s": stamps[k] - t0, "iterations": int(k + 1), "final_lagr": float(final),
            "niter": niter, "tol": tol, "warm_start_s": None}


if __name__ == "__main__":
    main()
