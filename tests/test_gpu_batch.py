"""Batched reconstructions of uneven sizes (one graph launch per iteration for
the whole batch) against each instance run alone, the per-instance FP64
direct-NUDFT error of the tomography operator, and the launch-shape
autotuner (shapes change the launch only: bit-identical results)."""
import numpy as np
import pytest

from oracle import usfft as ousfft
from ptychotomo_amd import objects

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SIZES = [32, 48, 64]


def _instance(n, seed):
    ntheta = 3 * n // 2
    theta = objects.make_theta(ntheta)
    prb = objects.gaussian_probe(8, 2.0)
    scan = objects.jittered_raster(ntheta, n, n, 8, 4, 1.0, np.random.default_rng(seed + 1))
    obj = objects.ellipsoid_phantom(n, n, 6, np.random.default_rng(seed), semi=(3, n / 5))
    args = (prb, scan, theta, [8, 8], 1e-6, 8.8, ntheta, n, n, ntheta // 4, n)
    return args, obj


def _init(slv):
    sh = (slv.ntheta, slv.nz, slv.n)
    sh3 = (3, slv.nz, slv.n, slv.n)
    z = lambda s: torch.zeros(s, dtype=torch.complex64, device="cuda")
    return dict(h=torch.ones(sh, dtype=torch.complex64, device="cuda"), e=z(sh3),
                psi=torch.ones(sh, dtype=torch.complex64, device="cuda"), phi=z(sh3),
                lamd=z(sh), mu=z(sh3), u=z((slv.nz, slv.n, slv.n)))


@pytest.mark.parametrize("grouped,graph,tiles", [
    (True, False, None), (True, False, 200), (False, True, None), (False, False, None),
    pytest.param(True, True, None, marks=pytest.mark.skip(
        reason="graph capture of the grouped iteration crashed the host process inside the "
               "HIP runtime's capture end, cause not found; BatchSolver refuses the "
               "combination"))])
def test_batch_matches_single_runs(grouped, graph, tiles):
    """tiles: the grouping threshold (200: the 32^3 instance grouped, the
    others on their own streams)"""
    from ptychotomo_amd.batch import BatchSolver
    from ptychotomo_amd.solver import Solver
    print("batch", SIZES, "grouped", grouped, "graph", graph, "tiles", tiles, flush=True)
    insts = [_instance(n, 100 + i) for i, n in enumerate(SIZES)]
    bs = BatchSolver.from_args([a for a, _ in insts])
    if tiles is not None:
        bs.GROUP_TILES = tiles
        assert [bs._small(i) for i in range(len(SIZES))] == [True, False, False]
    datas = []
    for slv, (_, obj) in zip(bs.solvers, insts):
        d = slv.fwd_ptycho_batch_dev(slv.exptomo(slv.fwd_tomo_batch(obj)))
        datas.append(torch.poisson(d * (1e2 / float(d.max()))))
    niter = 5
    res = bs.admm(datas, [_init(s) for s in bs.solvers], 3e-7, 4, 4, niter, "poisson",
                  lagr_every=1, grouped=grouped, graph=graph)
    for k, ((args, _), slv, d) in enumerate(zip(insts, bs.solvers, datas)):
        one = Solver(*args)
        st = _init(one)
        u, psi = one.admm(d, st["h"], st["e"], st["psi"], st["phi"], st["lamd"], st["mu"],
                          st["u"], 3e-7, 4, 4, niter, "poisson", lagr_every=1, verbose=False)
        assert len(slv.history) == niter
        for ra, rb in zip(slv.history, one.history):
            assert ra == rb, (SIZES[k], ra["m"])
        assert torch.equal(res[k][0], u) and torch.equal(res[k][1], psi), SIZES[k]


def test_nudft_error_per_instance():
    """Tomography operator of each batch size against the FP64 direct NUDFT
    (error stated per instance; the USFFT targets eps = 1e-6)."""
    from ptychotomo_amd.radonusfft import radonusfft
    for n in SIZES:
        ntheta = 3 * n // 2
        theta = objects.make_theta(ntheta)
        rng = np.random.default_rng(n)
        u = (rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))).astype(np.complex64)
        op = radonusfft(ntheta, 2, n)
        th = torch.from_numpy(theta).cuda()
        op.setobj(th.data_ptr())
        ud = torch.from_numpy(u).cuda()
        out = torch.zeros((ntheta, 2, n), dtype=torch.complex64, device="cuda")
        op.fwd(out.data_ptr(), ud.data_ptr())
        ref = ousfft.fwd_exact(u, theta)
        err = float(np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref))
        print(f"n={n}: USFFT vs FP64 direct NUDFT rel err {err:.2e}")
        assert err < 1e-5


def test_autotune_shapes_bit_identical(tmp_path):
    from ptychotomo_amd import _lib, autotune
    from ptychotomo_amd.radonusfft import radonusfft
    n, nz, ntheta = 64, 4, 96
    theta = objects.make_theta(ntheta)
    op = radonusfft(ntheta, nz, n)
    th = torch.from_numpy(theta).cuda()
    op.setobj(th.data_ptr())
    # n = 64 runs on the register line FFT by default: nothing to tune there
    assert autotune.register_lines(op)
    assert autotune.tune(op, nz, n, ntheta, cache=None)[1]["line_kernels"].startswith("register")
    _lib.call("pt_tomo_set_line_kernels", op._h, _lib.PT_LINES["generic"])
    assert not autotune.register_lines(op)
    rng = np.random.default_rng(1)
    u = torch.from_numpy((rng.standard_normal((nz, n, n)) + 1j).astype(np.complex64)).cuda()
    g = torch.from_numpy((rng.standard_normal((ntheta, nz, n)) + 1j).astype(np.complex64)).cuda()
    a0 = torch.empty((ntheta, nz, n), dtype=torch.complex64, device="cuda")
    b0 = torch.empty((nz, n, n), dtype=torch.complex64, device="cuda")
    op.fwd(a0.data_ptr(), u.data_ptr())
    op.adj(b0.data_ptr(), g.data_ptr())
    default = autotune.get(op)
    shape, entry = autotune.tune(op, nz, n, ntheta, cache=str(tmp_path / "t.json"))
    print("autotune", default, "->", shape, entry)
    assert autotune.get(op) == shape
    a1, b1 = torch.empty_like(a0), torch.empty_like(b0)
    for s in [shape, (1, 1, 1), default]:
        assert autotune._set(op, s)
        op.fwd(a1.data_ptr(), u.data_ptr())
        op.adj(b1.data_ptr(), g.data_ptr())
        assert torch.equal(a0, a1) and torch.equal(b0, b1), s
    assert not autotune._set(op, (1, 5, 1))       # columns: a power of two
    # cached: a second tune reads the file
    shape2, _ = autotune.tune(op, nz, n, ntheta, cache=str(tmp_path / "t.json"))
    assert shape2 == shape


def test_batch_resume_matches_single_resume():
    """A batch continued from each solver's saved state (first iteration index
    m0, the state's own rho, tau and R u) against each instance resumed alone."""
    from ptychotomo_amd.batch import BatchSolver
    from ptychotomo_amd.solver import Solver
    print("batch resume", SIZES, flush=True)
    insts = [_instance(n, 200 + i) for i, n in enumerate(SIZES)]
    bs = BatchSolver.from_args([a for a, _ in insts])
    datas = []
    for slv, (_, obj) in zip(bs.solvers, insts):
        d = slv.fwd_ptycho_batch_dev(slv.exptomo(slv.fwd_tomo_batch(obj)))
        datas.append(torch.poisson(d * (1e2 / float(d.max()))))
    n1, n2 = 3, 4
    bs.admm(datas, [_init(s) for s in bs.solvers], 3e-7, 4, 4, n1, "poisson")
    res = bs.admm(datas, [s.state for s in bs.solvers], 3e-7, 4, 4, n2, "poisson",
                  lagr_every=1, m0=n1)
    for k, ((args, _), slv, d) in enumerate(zip(insts, bs.solvers, datas)):
        one = Solver(*args)
        st = _init(one)
        one.admm(d, st["h"], st["e"], st["psi"], st["phi"], st["lamd"], st["mu"], st["u"],
                 3e-7, 4, 4, n1, "poisson", lagr_every=0, verbose=False)
        u, psi = one.admm_resume(d, 3e-7, 4, 4, n2, "poisson", lagr_every=1, verbose=False)
        assert [r["m"] for r in slv.history] == list(range(n1, n1 + n2))
        for ra, rb in zip(slv.history, one.history):
            assert ra == rb, (SIZES[k], ra["m"])
        assert slv.state["m"] == one.state["m"] == n1 + n2
        assert torch.equal(res[k][0], u) and torch.equal(res[k][1], psi), SIZES[k]


def test_group_entries_match_single_calls():
    """pt_ptycho_grad_group and pt_ptycho_linesearch_group on 9 instances of
    three sizes (more than one launch's worth) against the single-instance
    entry points: bit-identical outputs."""
    import ctypes
    from ptychotomo_amd import _lib
    from ptychotomo_amd.solver import Solver, _RHO
    sizes = [32, 48, 64] * 3
    g = torch.Generator(device="cuda").manual_seed(7)
    cplx = lambda sh: torch.complex(torch.randn(sh, device="cuda", generator=g),
                                    torch.randn(sh, device="cuda", generator=g)) * 0.1
    rows = []
    for k, n in enumerate(sizes):
        args, obj = _instance(n, 300 + k)
        slv = Solver(*args)
        op = slv._ptycho
        sh = (slv.ntheta, slv.nz, slv.n)
        psi = torch.exp(1j * cplx(sh).real).to(torch.complex64).contiguous()
        d = slv.fwd_ptycho_batch_dev(psi)
        data = torch.poisson(d * (1e2 / float(d.max()))).contiguous()
        blk = torch.tensor([1.0, 0.5 + 0.1 * k], dtype=torch.float64, device="cuda")
        nseg = slv.nchunk
        chunk = op.Ntheta // nseg
        ng = 3
        cand = torch.tensor([[0.0, 0.5, 0.25]] * nseg, dtype=torch.float64, device="cuda")
        skip = torch.zeros(2 * nseg, dtype=torch.float64, device="cuda")
        if nseg > 1:
            skip[3] = 1.0                      # second chunk finished: skipped
        rows.append(dict(slv=slv, op=op, psi=psi, dir=cplx(sh).contiguous(), h=cplx(sh) + 1,
                         lamd=cplx(sh), data=data, blk=blk, cand=cand, skip=skip, chunk=chunk,
                         nseg=nseg, ng=ng))
    mdl = _lib.PT_MODEL["poisson"]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rho_dev = lambda r: r["blk"].data_ptr() + 8 * _RHO
    # single calls
    for r in rows:
        cp, cd = float(r["slv"].coefptycho), float(r["slv"].coefdata)
        r["g1"] = torch.empty_like(r["psi"])
        _lib.call("pt_ptycho_grad", r["op"]._h, r["g1"].data_ptr(), r["psi"].data_ptr(),
                  r["data"].data_ptr(), r["h"].data_ptr(), r["lamd"].data_ptr(), 0.0,
                  rho_dev(r), cp, cd, mdl, st)
        r["f1"] = torch.full((r["nseg"] * r["ng"],), -1.0, dtype=torch.float64, device="cuda")
        r["f2"] = r["f1"].clone()
        _lib.call("pt_ptycho_linesearch", r["op"]._h, r["f1"].data_ptr(), r["f2"].data_ptr(),
                  r["psi"].data_ptr(), r["dir"].data_ptr(), r["data"].data_ptr(),
                  r["h"].data_ptr(), r["lamd"].data_ptr(), 0.0, rho_dev(r),
                  r["cand"].data_ptr(), r["ng"], r["chunk"], cp, cd, mdl, r["skip"].data_ptr(), st)
    # grouped calls
    ga, la = [], []
    for r in rows:
        cp, cd = float(r["slv"].coefptycho), float(r["slv"].coefdata)
        r["g2"] = torch.empty_like(r["psi"])
        r["F1"] = torch.full_like(r["f1"], -1.0)
        r["F2"] = r["F1"].clone()
        ga.append(_lib.GradArgs(r["op"]._h, r["g2"].data_ptr(), r["psi"].data_ptr(),
                                r["data"].data_ptr(), r["h"].data_ptr(), r["lamd"].data_ptr(),
                                0.0, rho_dev(r), cp, cd))
        la.append(_lib.LinesearchArgs(r["op"]._h, r["F1"].data_ptr(), r["F2"].data_ptr(),
                                      r["psi"].data_ptr(), r["dir"].data_ptr(),
                                      r["data"].data_ptr(), r["h"].data_ptr(),
                                      r["lamd"].data_ptr(), 0.0, rho_dev(r),
                                      r["cand"].data_ptr(), r["chunk"], cp, cd,
                                      r["skip"].data_ptr()))
    _lib.call("pt_ptycho_grad_group", (_lib.GradArgs * len(ga))(*ga), len(ga), mdl, st)
    _lib.call("pt_ptycho_linesearch_group", (_lib.LinesearchArgs * len(la))(*la), len(la), 3,
              mdl, st)
    torch.cuda.synchronize()
    for k, r in enumerate(rows):
        assert torch.equal(r["g1"], r["g2"]), (k, sizes[k])
        assert torch.equal(r["f1"], r["F1"]) and torch.equal(r["f2"], r["F2"]), (k, sizes[k])
        if r["nseg"] > 1:     # the skipped chunk's sums are left as they were
            assert float(r["F1"][r["ng"]]) == -1.0
        assert torch.isfinite(r["F1"][:r["ng"]]).all()
    print("grouped grad and line search match single calls on", sizes)
    # one handle twice in a group: refused before any launch
    with pytest.raises(_lib.PtError, match="twice"):
        _lib.call("pt_ptycho_grad_group", (_lib.GradArgs * 2)(ga[0], ga[0]), 2, mdl, st)


def test_group_sweep_decides_as_single_sweeps():
    """pt_ptycho_linesearch_sweep_group on instances on and off the tile path
    against pt_ptycho_linesearch_sweep at a near tie: the rho term's weight is
    walked in steps of one rounding through the value at which the two terms'
    changes cancel, so a sum that differs in its last bit decides otherwise.  The
    direction's entries span many powers of two, so that the order of an FP64 sum
    shows in its last bits.
    The same state, step and candidates at every weight, and both decisions met."""
    import ctypes
    from ptychotomo_amd import _lib
    from ptychotomo_amd.solver import Solver, _RHO
    print("grouped sweep at a near tie", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    cplx = lambda sh: torch.complex(torch.randn(sh, device="cuda", generator=g),
                                    torch.randn(sh, device="cuda", generator=g)) * 0.1
    f64 = lambda *v: torch.tensor(v, dtype=torch.float64, device="cuda")
    mdl, st = _lib.PT_MODEL["poisson"], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rows = []
    for k, (n, step) in enumerate([(64, 4), (48, 4), (128, 4), (64, 16)]):
        args, obj = _instance(n, 500 + k)
        if step != 4:        # sparse: off the tile path
            args = (args[0], objects.jittered_raster(args[6], n, n, 8, step, 1.0,
                                                     np.random.default_rng(k)), *args[2:])
        slv = Solver(*args)
        op = slv._ptycho
        sh = (slv.ntheta, slv.nz, slv.n)
        psi = torch.exp(1j * cplx(sh).real).to(torch.complex64).contiguous()
        d = slv.fwd_ptycho_batch_dev(psi)
        data = torch.poisson(d * (1e2 / float(d.max())), generator=g).contiguous()
        nseg, r = slv.nchunk, dict(slv=slv, keep=(psi, data))
        r.update(blk=f64(1.0, 0.5, 0.5), cand=f64(*[0.0, 0.5, 0.25] * nseg), nxt=f64(*[0.0] * 3 * nseg),
                 state=f64(*[0.5, 0.0] * nseg), step=f64(*[7.0] * 2 * nseg), w=f64(1.0, 1.0),
                 f=f64(*[0.0] * 3 * nseg), f2=f64(*[0.0] * 3 * nseg),
                 dir=cplx(sh) * torch.exp(4 * torch.randn(sh, device="cuda", generator=g)),
                 h=cplx(sh) + 1, lamd=cplx(sh))
        p = lambda key: r[key].data_ptr()
        r["args"] = _lib.LinesearchArgs(op._h, p("f"), p("f2"), psi.data_ptr(), p("dir"),
                                        data.data_ptr(), p("h"), p("lamd"), 0.0,
                                        p("blk") + 8 * _RHO, p("cand"), op.Ntheta // nseg,
                                        float(slv.coefptycho), float(slv.coefdata), p("state"))
        r["sweep"] = _lib.SweepArgs(p("nxt"), p("step"), p("w"))
        _lib.call("pt_ptycho_linesearch_group", r["args"], 1, 3, mdl, st)
        r["tie"] = -float(r["f"][1] / r["f2"][1])
        rows.append(r)
    out = ("state", "step", "nxt")
    arr = (_lib.LinesearchArgs * len(rows))(*[r["args"] for r in rows])
    sw = (_lib.SweepArgs * len(rows))(*[r["sweep"] for r in rows])
    seen = [set() for _ in rows]
    for e in range(-24, 25):
        got = []
        for grouped in (False, True):
            for r in rows:
                r["state"].copy_(f64(*[0.5, 0.0] * r["slv"].nchunk))
                r["step"].fill_(7.0)
                r["nxt"].fill_(-1.0)
                r["w"][1] = r["tie"] * (1.0 + e * 2.0 ** -52)
            if grouped:
                _lib.call("pt_ptycho_linesearch_sweep_group", arr, sw, len(rows), 3, 3, 0, mdl, st)
            else:
                for r in rows:
                    _lib.call("pt_ptycho_linesearch_sweep", r["args"], *(
                        r[k].data_ptr() for k in ("nxt", "step", "w")), 3, 3, 0, mdl, st)
            got.append([[r[k].tolist() for k in out] for r in rows])
        for k, (a, b) in enumerate(zip(*got)):
            assert a == b, (e, k, a, b)
            seen[k].add(a[0][0])
    print("steps met", seen)
    assert all(len(s) > 1 for s in seen)
    with pytest.raises(_lib.PtError, match="twice"):
        _lib.call("pt_ptycho_linesearch_sweep_group",
                  (_lib.LinesearchArgs * 2)(rows[0]["args"], rows[0]["args"]),
                  (_lib.SweepArgs * 2)(rows[0]["sweep"], rows[0]["sweep"]), 2, 3, 3, 0, mdl, st)
    with pytest.raises(_lib.PtError, match="null argument .instance 1"):
        _lib.call("pt_ptycho_linesearch_sweep_group", arr,
                  (_lib.SweepArgs * 2)(rows[0]["sweep"], _lib.SweepArgs()), 2, 3, 3, 0, mdl, st)


@pytest.mark.parametrize("n,count,small", [(48, 8, True), (96, 4, False)])
def test_default_grouping_is_the_faster_way(n, count, small):
    """Instances are grouped where that was measured faster than a stream each
    (up to 64^3, not from 80^3 on), and by default an iteration of either kind takes
    no longer than 1.15 times the faster of the two ways (48^3 on streams takes 1.3
    times)."""
    import time
    from ptychotomo_amd.batch import BatchSolver
    print(f"grouping {count} x {n}^3", flush=True)
    insts = [_instance(n, 700 + i) for i in range(count)]
    bs = BatchSolver.from_args([a for a, _ in insts])
    assert [bs._small(i) for i in range(count)] == [small] * count
    datas = []
    for slv, (_, obj) in zip(bs.solvers, insts):
        d = slv.fwd_ptycho_batch_dev(slv.exptomo(slv.fwd_tomo_batch(obj)))
        datas.append(torch.poisson(d * (1e2 / float(d.max()))))
    run = lambda st, niter, m0, grouped: bs.admm(datas, st, 3e-7, 4, 4, niter, "poisson",
                                                 m0=m0, grouped=grouped)
    run([_init(s) for s in bs.solvers], 3, 0, True)
    states = [dict(s.state) for s in bs.solvers]
    best = {}
    for _ in range(4):
        for name, tiles, grouped in (("default", None, True), ("all grouped", 1 << 40, True),
                                     ("streams", None, False)):
            bs.GROUP_TILES = BatchSolver.GROUP_TILES if tiles is None else tiles
            torch.cuda.synchronize()
            t = time.perf_counter()
            run([dict(s) for s in states], 4, 3, grouped)
            torch.cuda.synchronize()
            best[name] = min(best.get(name, np.inf), time.perf_counter() - t)
    print({k: f"{v * 250:.2f} ms/iteration" for k, v in best.items()})
    assert best["default"] < 1.15 * min(best.values())
