"""GPU parity of the native operators against the FP32 oracle restatement
(relative L2 <= 1e-5) and adjoint dot-product tests (<= 1e-5)."""
import numpy as np
import pytest

from oracle import ptycho as optycho
from oracle import usfft as ousfft

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def rel(a, b):
    a = np.asarray(a, np.complex128)
    b = np.asarray(b, np.complex128)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def crandn(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def make_scan(rng, pt, S, nz, n, P):
    scan = np.stack([rng.uniform(0, n - P, (pt, S)), rng.uniform(0, nz - P, (pt, S))]).astype(np.float32)
    return scan


@pytest.mark.parametrize("D,P,nz,n,S,pt", [(16, 16, 40, 48, 30, 3), (16, 12, 33, 41, 25, 2),
                                           (8, 5, 20, 24, 17, 2), (32, 32, 70, 64, 9, 2),
                                           (64, 16, 80, 80, 6, 1), (16, 16, 64, 256, 400, 2)])
def test_ptycho_fwd_adj(D, P, nz, n, S, pt):
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"ptycho D={D} P={P} nz={nz} n={n} S={S} pt={pt}", flush=True)
    rng = np.random.default_rng(D * 100 + P)
    psi = crandn(rng, (pt, nz, n))
    prb = crandn(rng, (P, P))  # asymmetric probe pins the transposed frame
    scan = make_scan(rng, pt, S, nz, n, P)
    scan[0, 0, 0] = -0.7  # skipped patch
    g = crandn(rng, (pt, S, D, D))
    op = ptychofft(pt, nz, n, pt, S, D, D, P)
    scand, prbd = dev(scan), dev(prb)  # keep alive across the call
    op.setobj(scand.data_ptr(), prbd.data_ptr())
    gd = torch.zeros((pt, S, D, D), dtype=torch.complex64, device="cuda")
    psid = dev(psi)
    op.fwd(gd.data_ptr(), psid.data_ptr())
    fd = torch.zeros((pt, nz, n), dtype=torch.complex64, device="cuda")
    gin = dev(g)
    op.adj(fd.data_ptr(), gin.data_ptr())
    torch.cuda.synchronize()
    ref_f = optycho.fwd(psi, prb, scan, D, D)
    ref_a = optycho.adj(g, prb, scan, nz, n)
    ef, ea = rel(gd.cpu().numpy(), ref_f), rel(fd.cpu().numpy(), ref_a)
    print(f"fwd rel {ef:.3e} adj rel {ea:.3e}")
    assert ef < 1e-5, ef
    assert ea < 1e-5, ea
    # adjointness of the device pair
    lhs = np.vdot(gd.cpu().numpy().astype(np.complex128), g.astype(np.complex128))
    rhs = np.vdot(psi.astype(np.complex128), fd.cpu().numpy().astype(np.complex128))
    ad = abs(lhs - rhs) / abs(lhs)
    print(f"adjoint {ad:.3e}")
    assert ad < 1e-5, ad


@pytest.mark.parametrize("n,pz,ntheta", [(16, 2, 12), (32, 3, 20), (64, 2, 24), (96, 1, 8),
                                         (128, 3, 10), (192, 2, 9), (256, 2, 16), (512, 1, 6)])
def test_tomo_fwd_adj(n, pz, ntheta):
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"tomo n={n} pz={pz} ntheta={ntheta}", flush=True)
    rng = np.random.default_rng(n)
    theta = np.linspace(0, np.pi, ntheta, endpoint=False).astype(np.float32)
    u = crandn(rng, (pz, n, n))
    g = crandn(rng, (ntheta, pz, n))
    op = radonusfft(ntheta, pz, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    out = torch.zeros((ntheta, pz, n), dtype=torch.complex64, device="cuda")
    ud = dev(u)
    op.fwd(out.data_ptr(), ud.data_ptr())
    back = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
    gd = dev(g)
    op.adj(back.data_ptr(), gd.data_ptr())
    torch.cuda.synchronize()
    ef = rel(out.cpu().numpy(), ousfft.fwd(u, theta))
    ea = rel(back.cpu().numpy(), ousfft.adj(g, theta))
    print(f"fwd rel {ef:.3e} adj rel {ea:.3e}")
    assert ef < 1e-5, ef
    assert ea < 1e-5, ea


@pytest.mark.parametrize("n,pz,ntheta", [(64, 3, 10), (96, 33, 6), (128, 5, 12), (192, 17, 7),
                                         (256, 17, 8), (512, 9, 4)])
def test_tomo_line_kernels_agree(n, pz, ntheta):
    """The register line FFT passes (the default for n = 64, 96, 128, 192, 256,
    512)
    against the generic LDS passes on the same handle: forward, adjoint and
    the ramp-filtered adjoint agree to FP32 rounding (the two sum in
    different orders).  pz above a workgroup's slice count exercises the
    partial slice blocks of the detector-line passes."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"tomo line kernels n={n} pz={pz} ntheta={ntheta}", flush=True)
    rng = np.random.default_rng(n + 7)
    theta = np.sort(rng.uniform(0, np.pi, ntheta)).astype(np.float32)
    ud, gd = dev(crandn(rng, (pz, n, n))), dev(crandn(rng, (ntheta, pz, n)))
    op = radonusfft(ntheta, pz, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    res = {}
    for kind in (_lib.PT_LINES["auto"], _lib.PT_LINES["generic"]):
        _lib.call("pt_tomo_set_line_kernels", op._h, kind)
        out = torch.zeros((ntheta, pz, n), dtype=torch.complex64, device="cuda")
        back = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
        fbp = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
        op.fwd(out.data_ptr(), ud.data_ptr())
        op.adj(back.data_ptr(), gd.data_ptr())
        op.setfilter("ramp")
        op.adj(fbp.data_ptr(), gd.data_ptr())
        op.setfilter("none")
        torch.cuda.synchronize()
        res[kind] = [x.cpu().numpy() for x in (out, back, fbp)]
    _lib.call("pt_tomo_set_line_kernels", op._h, _lib.PT_LINES["auto"])
    with pytest.raises(_lib.PtError):
        _lib.call("pt_tomo_set_line_kernels", op._h, 7)
    for name, a, b in zip(("fwd", "adj", "adj ramp"), res[0], res[1]):
        e = rel(a, b)
        print(f"{name}: register vs generic rel {e:.2e}")
        assert np.isfinite(a).all() and e < 2e-6, (name, e)


@pytest.mark.parametrize("n", [256, 384])
def test_tomo_large_vs_direct_nudft(n):
    """Production-size USFFT forward against the FP64 direct nonuniform DFT
    on four angles of one slice (the USFFT targets eps = 1e-6)."""
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"tomo direct NUDFT n={n}", flush=True)
    rng = np.random.default_rng(n + 1)
    theta = rng.uniform(0, np.pi, 4).astype(np.float32)
    u = crandn(rng, (1, n, n))
    op = radonusfft(4, 1, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    out = torch.zeros((4, 1, n), dtype=torch.complex64, device="cuda")
    ud = dev(u)
    op.fwd(out.data_ptr(), ud.data_ptr())
    ref = ousfft.fwd_exact(u, theta)
    err = rel(out.cpu().numpy(), ref)
    print(f"n={n}: USFFT vs FP64 direct NUDFT rel err {err:.2e}")
    assert err < 1e-5, err


@pytest.mark.parametrize("n,pz", [(4, 1), (8, 3), (20, 2), (36, 1), (60, 5), (64, 17), (100, 1),
                                  (128, 3)])
def test_tomo_fwd_vs_direct_sums(n, pz):
    """The forward against the FP64 direct nonuniform DFT, at sizes around the
    edges of the gridding kernel: a grid smaller than a tile and its halo,
    partial last tiles, odd slice counts, angles on the grid axes (integer
    sample positions).  Tolerance: the gridding kernel's 1e-7 plus a few ulp
    per FFT pass over three transforms, under 1e-6."""
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"tomo forward direct sums n={n} pz={pz}", flush=True)
    rng = np.random.default_rng(n + pz)
    theta = np.concatenate([[0, np.pi / 4, np.pi / 2, np.pi], rng.uniform(0, np.pi, 3)])
    theta = theta.astype(np.float32)
    u = crandn(rng, (pz, n, n))
    op = radonusfft(theta.size, pz, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    out = torch.zeros((theta.size, pz, n), dtype=torch.complex64, device="cuda")
    ud = dev(u)
    op.fwd(out.data_ptr(), ud.data_ptr())
    err = rel(out.cpu().numpy(), ousfft.fwd_exact(u, theta))
    print(f"rel {err:.2e}")
    assert err < 1e-6, err


@pytest.mark.parametrize("n,pz,nth", [(4, 1, 7), (8, 3, 7), (20, 2, 7), (36, 9, 7), (60, 5, 40),
                                      (64, 17, 96), (100, 1, 7), (96, 70, 7), (128, 3, 200)])
def test_tomo_adj_vs_direct_sums(n, pz, nth):
    """The adjoint against the FP64 direct adjoint, at sizes around the edges
    of the gridding: a footprint that wraps onto its own tile (n = 4), slice
    counts around the blocks of 8, dense centre tiles of several entry chunks,
    angles on the grid axes.  Tolerance: the gridding kernel's 1e-7 of all
    samples, of which the edge-replicating pad puts up to four times the
    output's norm outside the cropped object, plus a few ulp per FFT pass:
    under 2e-6."""
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"tomo adjoint direct sums n={n} pz={pz} nth={nth}", flush=True)
    rng = np.random.default_rng(n + pz)
    theta = np.concatenate([[0, np.pi / 4, np.pi / 2, np.pi], rng.uniform(0, np.pi, nth - 4)])
    theta = theta.astype(np.float32)
    g = crandn(rng, (nth, pz, n))
    op = radonusfft(nth, pz, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    back = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
    gd = dev(g)
    op.adj(back.data_ptr(), gd.data_ptr())
    z = sorted({0, pz // 2, pz - 1})   # the direct sums of some slices
    err = rel(back.cpu().numpy()[z], ousfft.adj_exact(g[:, z], theta))
    print(f"rel {err:.2e}")
    assert err < 2e-6, err


def test_tomo_adjoint_zero_border():
    """With a zero object border and zero detector edges the boundary pads
    vanish and the operator pair is exactly adjoint."""
    from ptychotomo_amd.radonusfft import radonusfft
    n, pz, ntheta = 32, 2, 16
    rng = np.random.default_rng(5)
    theta = np.linspace(0, np.pi, ntheta, endpoint=False).astype(np.float32)
    u = crandn(rng, (pz, n, n))
    u[:, 0, :] = u[:, -1, :] = u[:, :, 0] = u[:, :, -1] = 0
    g = crandn(rng, (ntheta, pz, n))
    g[:, :, 0] = g[:, :, -1] = 0
    op = radonusfft(ntheta, pz, n)
    th = dev(theta)
    op.setobj(th.data_ptr())
    out = torch.zeros((ntheta, pz, n), dtype=torch.complex64, device="cuda")
    back = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
    ud, gd = dev(u), dev(g)
    op.fwd(out.data_ptr(), ud.data_ptr())
    op.adj(back.data_ptr(), gd.data_ptr())
    torch.cuda.synchronize()
    lhs = np.vdot(out.cpu().numpy().astype(np.complex128), g.astype(np.complex128))
    rhs = np.vdot(u.astype(np.complex128), back.cpu().numpy().astype(np.complex128))
    assert abs(lhs - rhs) / abs(lhs) < 1e-5


def test_bitwise_reproducible():
    """Deterministic overlap-add and gridding: two runs are bit-identical."""
    from ptychotomo_amd.ptychofft import ptychofft
    from ptychotomo_amd.radonusfft import radonusfft
    rng = np.random.default_rng(9)
    pt, nz, n, S, D = 2, 48, 48, 60, 16
    psi = crandn(rng, (pt, nz, n))
    prb = crandn(rng, (D, D))
    scan = make_scan(rng, pt, S, nz, n, D)
    g = crandn(rng, (pt, S, D, D))
    op = ptychofft(pt, nz, n, pt, S, D, D, D)
    scand, prbd = dev(scan), dev(prb)
    op.setobj(scand.data_ptr(), prbd.data_ptr())
    gin = dev(g)
    outs = []
    for _ in range(2):
        f = torch.zeros((pt, nz, n), dtype=torch.complex64, device="cuda")
        op.adj(f.data_ptr(), gin.data_ptr())
        outs.append(f.cpu().numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    tomo = radonusfft(24, 2, 32)
    th = dev(np.linspace(0, np.pi, 24, endpoint=False).astype(np.float32))
    tomo.setobj(th.data_ptr())
    gg = dev(crandn(rng, (24, 2, 32)))
    outs = []
    for _ in range(2):
        f = torch.zeros((2, 32, 32), dtype=torch.complex64, device="cuda")
        tomo.adj(f.data_ptr(), gg.data_ptr())
        outs.append(f.cpu().numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


def test_tomo_ramp_filter_adj():
    """Filtered adjoint (applyfilter) against the restatement, then the filter
    switched off again restores the plain adjoint."""
    from ptychotomo_amd.radonusfft import radonusfft
    n, pz, ntheta = 32, 2, 20
    print(f"ramp filter n={n} pz={pz} ntheta={ntheta}", flush=True)
    rng = np.random.default_rng(11)
    theta = np.linspace(0, np.pi, ntheta, endpoint=False).astype(np.float32)
    g = crandn(rng, (ntheta, pz, n))
    op = radonusfft(ntheta, pz, n)
    th, gd = dev(theta), dev(g)
    op.setobj(th.data_ptr())
    back = torch.zeros((pz, n, n), dtype=torch.complex64, device="cuda")
    op.setfilter("ramp")
    op.adj(back.data_ptr(), gd.data_ptr())
    torch.cuda.synchronize()
    ef = rel(back.cpu().numpy(), ousfft.adj(g, theta, filt="ramp"))
    op.setfilter(None)
    op.adj(back.data_ptr(), gd.data_ptr())
    torch.cuda.synchronize()
    ea = rel(back.cpu().numpy(), ousfft.adj(g, theta))
    print(f"filtered adj rel {ef:.3e} plain adj rel {ea:.3e}")
    assert ef < 1e-5, ef
    assert ea < 1e-5, ea


def test_solver_fbp_inverts_radon():
    """Solver.fbp_tomo_batch(fwd_tomo_batch(u)) approximates u (inverse
    Radon transform; error of the reference's ramp filter itself ~9 %)."""
    from ptychotomo_amd import Solver, objects
    n, nz, ntheta = 64, 16, 96
    theta = np.linspace(0, np.pi, ntheta, endpoint=False).astype(np.float32)
    prb = objects.gaussian_probe(16, 4.0, 0.5)
    scan = np.zeros((2, ntheta, 4), np.float32)
    slv = Solver(prb, scan, theta, [16, 16], 1e-6, 8.8, ntheta, nz, n, ntheta, nz)
    y, x = np.mgrid[:n, :n] - n / 2 + 0.5
    u = np.exp(-(x ** 2 + y ** 2) / (2 * (n / 10) ** 2)).astype(np.complex64)
    u = np.repeat(u[None], nz, 0) * (1 + 0.1j)
    rec = slv.fbp_tomo_batch(slv.fwd_tomo_batch(u)).cpu().numpy()
    c = np.vdot(u, rec).real / np.vdot(u, u).real
    err = rel(rec / c, u)
    print(f"fbp scale {c:.4f} rel err {err:.3e}")
    assert abs(c - 1) < 0.05, c
    assert err < 0.12, err


@pytest.mark.parametrize("n,nz,det,step", [(72, 56, 16, 4), (32, 40, 8, 3), (64, 64, 32, 8)])
def test_ptycho_linesearch_fused_rho_term(n, nz, det, step):
    """pt_ptycho_linesearch: f1 identical to pt_ptycho_minf's data term; f2
    (the rho term summed over the pixels each overlap-add tile owns) equal to
    the separate element-wise pass pt_k_rho_minf up to FP64 summation order,
    on objects whose size is not a multiple of the tile size (the last tiles
    own the remainder), and on 32 x 32 frames (per-patch kernel, separate rho
    pass)."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"linesearch n={n} nz={nz} det={det} step={step}", flush=True)
    rng = np.random.default_rng(n + det)
    nt, chunk = 6, 3
    scan = objects.jittered_raster(nt, nz, n, det, step, 1.0, rng)
    op = ptychofft(nt, nz, n, nt, scan.shape[2], det, det, det)
    sc, pr = dev(scan), dev(objects.gaussian_probe(det, det / 4))
    op.setobj(sc.data_ptr(), pr.data_ptr())
    sh = (nt, nz, n)
    psi = dev(np.exp(1j * 0.3 * rng.standard_normal(sh)).astype(np.complex64))
    d = dev(crandn(rng, sh) * np.float32(0.05))
    h = dev(crandn(rng, sh))
    lamd = dev(crandn(rng, sh) * np.float32(0.1))
    data = dev(rng.poisson(4.0, (nt, scan.shape[2], det, det)).astype(np.float32))
    gam = np.array([0.0, 1.0, 0.5, 0.25, 0.125], np.float64)
    ng = len(gam)
    g = dev(np.tile(gam, nt // chunk))
    rho = torch.tensor([0.7], dtype=torch.float64, device="cuda")
    out = {k: torch.zeros(nt // chunk * ng, dtype=torch.float64, device="cuda")
           for k in ("f1", "f2", "m", "r")}
    for model in ("poisson", "gaussian"):
        mdl = _lib.PT_MODEL[model]
        _lib.call("pt_ptycho_linesearch", op._h, ptr(out["f1"]), ptr(out["f2"]), ptr(psi), ptr(d),
                  ptr(data), ptr(h), ptr(lamd), 0.0, ptr(rho), ptr(g), ng, chunk, 1.1, 0.9, mdl,
                  None, stream())
        _lib.call("pt_ptycho_minf", op._h, ptr(out["m"]), ptr(psi), ptr(d), ptr(data), ptr(g), ng,
                  chunk, 1.1, 0.9, mdl, 0, None, stream())
        _lib.call("pt_k_rho_minf", ptr(out["r"]), ptr(h), ptr(psi), ptr(lamd), ptr(d), 0.0,
                  ptr(rho), ptr(g), ng, psi.numel(), nt // chunk, None, stream())
        torch.cuda.synchronize()
        f1, f2, m, r = (out[k].cpu().numpy() for k in ("f1", "f2", "m", "r"))
        print(model, f2[:ng], r[:ng])
        np.testing.assert_array_equal(f1, m)
        assert np.all(f2[::ng] == 0) and np.all(r[::ng] == 0)      # gamma = 0
        np.testing.assert_allclose(f2, r, rtol=1e-12, atol=1e-12 * np.abs(r).max())


def test_ptycho_minf_candidate_cancelling_the_far_field():
    """A step candidate that nearly cancels the far field (psi + g*d = 1e-4
    psi at g = 0.25): the Poisson log ratio |ag|^2/|a|^2 ~ 1e-8 is taken
    from the ratio itself (1 + x loses it to rounding and can fall to <= 0,
    which made the sum NaN and the halving rule accept the step).  Every
    candidate's change is finite and matches the FP64 evaluation."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    from oracle import ptycho as optycho
    rng = np.random.default_rng(12)
    nt, nz, n, D = 4, 32, 32, 16
    scan = objects.jittered_raster(nt, nz, n, D, 4, 1.0, rng)
    prb = objects.gaussian_probe(D, D / 4)
    op = ptychofft(nt, nz, n, nt, scan.shape[2], D, D, D)
    sc, pr = dev(scan), dev(prb)
    op.setobj(sc.data_ptr(), pr.data_ptr())
    psi = np.exp(1j * 0.3 * rng.standard_normal((nt, nz, n))).astype(np.complex64)
    d = (-psi * np.float32((1 - 1e-4) / 0.25)).astype(np.complex64)
    far = optycho.fwd(psi.astype(np.complex128), prb, scan, D, D, np.complex128)
    data = rng.poisson(np.abs(far) ** 2 * 2.0).astype(np.float32)
    gam = np.array([0.0, 1.0, 0.5, 0.25, 0.125], np.float64)
    sums = torch.zeros(len(gam), dtype=torch.float64, device="cuda")
    cp, cd = 1.0, 1.0
    psid, dd, datad, gd = dev(psi), dev(d), dev(data), dev(gam)
    _lib.call("pt_ptycho_minf", op._h, ptr(sums), ptr(psid), ptr(dd), ptr(datad), ptr(gd),
              len(gam), nt, cp, cd, _lib.PT_MODEL["poisson"], 0, None, stream())
    s = sums.cpu().numpy()
    a = optycho.fwd(psi.astype(np.complex128), prb, scan, D, D, np.complex128)
    b = optycho.fwd(d.astype(np.complex128), prb, scan, D, D, np.complex128)
    d64 = data.astype(np.float64)

    def f(g):
        ag = (a.astype(np.complex64) + np.float32(g) * b.astype(np.complex64)).astype(np.complex128)
        return np.sum(np.abs(ag) ** 2 - 2 * d64 * np.log(np.maximum(np.abs(ag), 1e-32)))
    f0 = f(0.0)
    print(s, [f(g) - f0 for g in gam])
    assert np.all(np.isfinite(s))
    for j, g in enumerate(gam):
        ref = f(g) - f0
        assert abs(s[j] - ref) <= 1e-5 * abs(f0) + 1e-4 * abs(ref), (g, s[j], ref)


@pytest.mark.parametrize("det,P,n,nz,step", [(32, 32, 64, 64, 8), (32, 20, 70, 61, 5),
                                             (64, 16, 80, 72, 8), (64, 11, 71, 66, 7)])
@pytest.mark.parametrize("model", ["poisson", "gaussian"])
def test_ptycho_large_frames_vs_fp64(det, P, n, nz, step, model):
    """Fused gradient, line-search sums and adjoint of 32 x 32 and 64 x 64
    frames against FP64: probes that fill the frame, smaller ones (with an odd
    size, so an uneven offset), the largest that takes one wave per frame at 64
    (16); a skipped position in x and one in y, frames of an
    object that is zero there (|a| = 0).  Tolerances: the FP64 forward's final
    rounding and an FP32 inverse transform (1e-7 each, 12 passes) in the
    gradient, FP32 terms summed in FP64 in the functional: under 1e-5."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"large frames det={det} P={P} n={n} nz={nz} {model}", flush=True)
    rng = np.random.default_rng(det + P)
    nt, chunk, cp, cd, rho = 4, 2, 1.1, 0.9, 0.7
    scan = objects.jittered_raster(nt, nz, n, P, step, 1.0, rng)
    scan[0, 0, 1], scan[1, 1, 2] = -0.8, -0.9
    prb = crandn(rng, (P, P))
    op = ptychofft(nt, nz, n, nt, scan.shape[2], det, det, P)
    sc, pr = dev(scan), dev(prb)
    op.setobj(sc.data_ptr(), pr.data_ptr())
    sh = (nt, nz, n)
    psi = np.exp(1j * 0.3 * rng.standard_normal(sh)).astype(np.complex64)
    psi[2] = 0
    d = crandn(rng, sh) * np.float32(0.05)
    h, lamd = crandn(rng, sh), crandn(rng, sh) * np.float32(0.1)
    data = rng.poisson(4.0, (nt, scan.shape[2], det, det)).astype(np.float32)
    far = lambda x: cp * optycho.fwd(x, prb, scan, det, det, np.complex128)  # noqa: E731
    a, b, q = far(psi), far(d), np.float64(np.float32(cd)) * data
    if model == "poisson":
        r = a - q * a / (np.abs(a) ** 2 + 1e-32)
    else:
        r = a - np.sqrt(q) * np.exp(1j * np.angle(np.where(a == 0, 0, a)))  # angle(0) = 0
    ref = cp * optycho.adj(r, prb, scan, nz, n, np.complex128) - rho * (h - psi + lamd / rho)
    mdl = _lib.PT_MODEL[model]
    t = {k: dev(v) for k, v in dict(psi=psi, d=d, h=h, lamd=lamd, data=data).items()}
    out = torch.zeros(sh, dtype=torch.complex64, device="cuda")
    _lib.call("pt_ptycho_grad", op._h, ptr(out), ptr(t["psi"]), ptr(t["data"]), ptr(t["h"]),
              ptr(t["lamd"]), rho, None, cp, cd, mdl, stream())
    eg = rel(out.cpu().numpy(), ref)
    gam = np.array([0.0, 1.0, 0.25, 2.0 ** -9], np.float64)
    g = dev(np.tile(gam, nt // chunk))
    f1 = torch.zeros(nt // chunk * 4, dtype=torch.float64, device="cuda")
    _lib.call("pt_ptycho_minf", op._h, ptr(f1), ptr(t["psi"]), ptr(t["d"]), ptr(t["data"]),
              ptr(g), 4, chunk, cp, cd, mdl, 0, None, stream())
    mlog = lambda x: np.log(np.maximum(x, 1e-32))  # noqa: E731
    m0, es = np.abs(a), []
    for c in range(nt // chunk):
        s = slice(c * chunk, (c + 1) * chunk)
        for j, gj in enumerate(gam):
            m = np.abs(a + gj * b)
            e = m ** 2 - m0 ** 2 - 2 * q * (mlog(m) - mlog(m0)) if model == "poisson" else \
                (m - np.sqrt(q)) ** 2 - (m0 - np.sqrt(q)) ** 2
            es.append(abs(float(f1[c * 4 + j]) - e[s].sum()) / max(np.abs(e[s]).sum(), 1e-30))
    gin = crandn(rng, data.shape)
    gd = dev(gin)
    op.adj(out.data_ptr(), gd.data_ptr())
    ea = rel(out.cpu().numpy(), optycho.adj(gin, prb, scan, nz, n, np.complex128))
    print(f"grad {eg:.2e} sums {max(es):.2e} adj {ea:.2e}")
    assert eg < 1e-5 and max(es) < 1e-5 and ea < 1e-5, (eg, es, ea)


@pytest.mark.parametrize("det,P", [(8, 5), (16, 16), (16, 11), (32, 32), (32, 17), (64, 16),
                                   (64, 7), (64, 17)])
def test_ptycho_intensity(det, P):
    """Far-field intensities without the far field, one wave per frame or rows
    per lane, with a skipped position, against FP64; tolerance an FP32
    transform's (1e-7 per pass, 12 passes, squared): under 5e-6."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"intensity det={det} P={P}", flush=True)
    rng = np.random.default_rng(det + P)
    nt, nz, n = 3, 70, 75
    scan = objects.jittered_raster(nt, nz, n, P, 9, 1.0, rng)
    scan[1, 0, 3] = -0.7
    prb, psi = crandn(rng, (P, P)), crandn(rng, (nt, nz, n))
    op = ptychofft(nt, nz, n, nt, scan.shape[2], det, det, P)
    sc, pr, pd = dev(scan), dev(prb), dev(psi)
    op.setobj(sc.data_ptr(), pr.data_ptr())
    out = torch.full((nt, scan.shape[2], det, det), 7.0, device="cuda")
    _lib.call("pt_ptycho_intensity", op._h, ptr(out), ptr(pd), 1.3, 0.4, stream())
    ref = 0.4 * np.abs(1.3 * optycho.fwd(psi, prb, scan, det, det, np.complex128)) ** 2
    err = rel(out.cpu().numpy(), ref)
    print(f"rel {err:.2e}")
    assert err < 5e-6, err


@pytest.mark.parametrize("nt,nz,n", [(1, 1, 4), (3, 5, 12), (24, 24, 36)])
@pytest.mark.parametrize("fit", [1.0, 2.0 ** -7, 2.0 ** -8, 2.0 ** -23, -1.0])
def test_tomo_linesearch_follows_the_sweeps(nt, nz, n, fit):
    """pt_k_tomo_linesearch against the same search from its parts (sweeps of 7
    candidates): accepted in the first group, in its last slot, in the next
    groups, and never (an ascent direction: step 0).  The residual is the
    direction's image times `fit`, so steps below 2 fit decrease the functional;
    whole halvings, so the steps are equal."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd._dev import ptr, stream
    print(f"tomo line search nt={nt} nz={nz} n={n} fit={fit}", flush=True)
    rng = np.random.default_rng(n)
    K, Rd, Ru = (crandn(rng, (nt, nz, n)) for _ in range(3))
    u, d = crandn(rng, (nz, n, n)), crandn(rng, (nz, n, n))
    J = lambda v: np.stack([  # noqa: E731
        np.pad(np.diff(v, axis=2), ((0, 0), (0, 0), (0, 1))),
        np.pad(np.diff(v, axis=1), ((0, 0), (0, 1), (0, 0))),
        np.pad(np.diff(v, axis=0), ((0, 1), (0, 0), (0, 0)))]) * (2 / np.sqrt(3))
    # just below the crossing, away from ties
    xi0 = K * (Ru + 0.9 * fit * Rd)
    xi1 = J(u + 0.9 * fit * d)
    t = {k: dev(np.ascontiguousarray(v, dtype=np.complex64)) for k, v in
         dict(K=K, Ru=Ru, Rd=Rd, xi0=xi0, u=u, d=d, xi1=xi1).items()}
    z = lambda *v: torch.tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    w, st = z(0.5, 0.25), stream()
    state, step = z(2.0, 0.0), z(7.0, 7.0)
    _lib.call("pt_k_tomo_linesearch", ptr(state), ptr(step), ptr(t["K"]), ptr(t["Ru"]),
              ptr(t["Rd"]), ptr(t["xi0"]), ptr(t["u"]), ptr(t["d"]), ptr(t["xi1"]), ptr(w),
              K.size, nz, n, n, st)
    s2, p2, c, f1, f2 = z(2.0, 0.0), z(7.0, 7.0), z(*[0.0] * 8), z(*[0.0] * 8), z(*[0.0] * 8)
    _lib.call("pt_k_ls_begin", ptr(s2), ptr(c), 1, 8, st)
    for sw in range(6):
        _lib.call("pt_k_tomo_minf", ptr(f1), ptr(t["K"]), ptr(t["Ru"]), ptr(t["Rd"]),
                  ptr(t["xi0"]), ptr(c), 8, K.size, ptr(s2), st)
        _lib.call("pt_k_reg_minf", ptr(f2), ptr(t["u"]), ptr(t["d"]), ptr(t["xi1"]), ptr(c), 8,
                  nz, n, n, ptr(s2), st)
        _lib.call("pt_k_ls_select", ptr(s2), ptr(c), ptr(c), ptr(p2), ptr(f1), ptr(f2), ptr(w),
                  1, 8, 8, int(sw == 5), st)
    got, ref = step.cpu().numpy(), p2.cpu().numpy()
    print(got, ref)
    assert np.array_equal(got, ref) and np.array_equal(state.cpu().numpy(), s2.cpu().numpy())
    if fit > 2.0 ** -20:
        assert 0.45 * fit < got[0] <= 1.8 * fit


def _product_far(psi, prb, scan, det, rounded):
    """FP64 transforms of the frames probe x object, the products in FP32 with
    one fused multiply-add per part (rounded) or exact."""
    pos = (np.sign(scan) * np.floor(np.abs(scan) + 0.5)).astype(int)
    P, o = len(prb), (det - len(prb)) // 2
    fr = np.zeros((*scan.shape[1:], det, det), np.complex128)
    r = (lambda x: x.astype(np.float32).astype(np.float64)) if rounded else (lambda x: x)
    pr, pi = prb.real.astype(np.float64), prb.imag.astype(np.float64)
    for t, s in np.ndindex(*scan.shape[1:]):
        x, y = pos[:, t, s]
        if min(x, y) < 0:
            continue
        v = psi[t, y:y + P, x:x + P].T.astype(np.complex128)
        re, im = r(pr * v.real - r(pi * v.imag)), r(pr * v.imag + r(pi * v.real))
        fr[t, s, o:o + P, o:o + P] = re + 1j * im
    return np.fft.fft2(fr)


@pytest.mark.parametrize("det,P,n,nz,step", [(8, 8, 40, 33, 3), (8, 5, 33, 40, 2),
                                             (16, 16, 64, 49, 4), (16, 11, 50, 61, 3)])
@pytest.mark.parametrize("model", ["poisson", "gaussian"])
def test_ptycho_grad_small_frames_vs_fp64(det, P, n, nz, step, model):
    """Fused gradient of 8 x 8 and 16 x 16 frames, probes that fill the frame and
    smaller odd ones, against FP64; a skipped position, frames of an object that
    is zero there, a last group of patches that does not fill a wave, and the
    grouped call of the same.  Tolerance: the FP64 forward's final rounding and
    an FP32 inverse transform (1e-7 each, 8 passes): under 1e-5."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"small frames det={det} P={P} n={n} nz={nz} {model}", flush=True)
    rng = np.random.default_rng(det + P)
    nt, cp, cd, rho = 3, 1.1, 0.9, 0.7
    scan = objects.jittered_raster(nt, nz, n, P, step, 1.0, rng)
    scan[0, 0, 1] = -0.8
    prb = crandn(rng, (P, P))
    op = ptychofft(nt, nz, n, nt, scan.shape[2], det, det, P)
    sc, pr = dev(scan), dev(prb)
    op.setobj(sc.data_ptr(), pr.data_ptr())
    sh = (nt, nz, n)
    psi = np.exp(1j * 0.3 * rng.standard_normal(sh)).astype(np.complex64)
    psi[2] = 0
    h, lamd = crandn(rng, sh), crandn(rng, sh) * np.float32(0.1)
    data = rng.poisson(4.0, (nt, scan.shape[2], det, det)).astype(np.float32)
    a = cp * optycho.fwd(psi, prb, scan, det, det, np.complex128)
    # the residual d a/|a|^2 magnifies the rounding of the FP32 products probe x
    # object without bound at small |a|: the reference transforms those products
    f32, f64 = _product_far(psi, prb, scan, det, True), _product_far(psi, prb, scan, det, False)
    assert np.allclose(np.abs(a), cp / det * np.abs(f64), rtol=0, atol=1e-9)
    a = a * np.divide(f32, f64, out=np.ones_like(f64), where=f64 != 0)
    q = np.float64(np.float32(cd)) * data
    if model == "poisson":
        r = a - q * a / (np.abs(a) ** 2 + 1e-32)
    else:
        r = a - np.sqrt(q) * np.exp(1j * np.angle(np.where(a == 0, 0, a)))  # angle(0) = 0
    ref = cp * optycho.adj(r, prb, scan, nz, n, np.complex128) - rho * (h - psi + lamd / rho)
    mdl = _lib.PT_MODEL[model]
    t = {k: dev(v) for k, v in dict(psi=psi, h=h, lamd=lamd, data=data).items()}
    out, out2 = (torch.zeros(sh, dtype=torch.complex64, device="cuda") for _ in range(2))
    _lib.call("pt_ptycho_grad", op._h, ptr(out), ptr(t["psi"]), ptr(t["data"]), ptr(t["h"]),
              ptr(t["lamd"]), rho, None, cp, cd, mdl, stream())
    arr = (_lib.GradArgs * 1)(_lib.GradArgs(op._h, out2.data_ptr(), t["psi"].data_ptr(),
                                            t["data"].data_ptr(), t["h"].data_ptr(),
                                            t["lamd"].data_ptr(), rho, None, cp, cd))
    _lib.call("pt_ptycho_grad_group", arr, 1, mdl, stream())
    e = rel(out.cpu().numpy(), ref)
    print(f"grad {e:.2e}")
    assert e < 1e-5, e
    assert torch.equal(torch.view_as_real(out), torch.view_as_real(out2))


@pytest.mark.parametrize("n,pz,ntheta", [(20, 3, 11), (64, 3, 20), (36, 9, 14)])
def test_tomo_grid_corners_are_not_read(n, pz, ntheta):
    """The grid's corners beyond the samples' disc are neither written nor read:
    after a pass over NaN in each direction the results equal a fresh handle's
    (generic and register line passes, an odd slice count)."""
    from ptychotomo_amd.radonusfft import radonusfft
    print(f"grid corners n={n} pz={pz} ntheta={ntheta}", flush=True)
    rng = np.random.default_rng(n)
    th = dev(np.linspace(0, np.pi, ntheta, endpoint=False).astype(np.float32))
    u, g = dev(crandn(rng, (pz, n, n))), dev(crandn(rng, (ntheta, pz, n)))
    un, gn = torch.full_like(u, float("nan")), torch.full_like(g, float("nan"))
    res = []
    for stale in (False, True):
        op = radonusfft(ntheta, pz, n)
        op.setobj(th.data_ptr())
        f, b = torch.zeros_like(g), torch.zeros_like(u)
        if stale:
            op.fwd(f.data_ptr(), un.data_ptr())
            op.adj(b.data_ptr(), gn.data_ptr())
            op.fwd(f.data_ptr(), un.data_ptr())
        op.adj(b.data_ptr(), g.data_ptr())
        if stale:
            op.adj(un.data_ptr(), gn.data_ptr())
        op.fwd(f.data_ptr(), u.data_ptr())
        torch.cuda.synchronize()
        res.append((f.cpu().numpy(), b.cpu().numpy()))
    np.testing.assert_array_equal(res[0][0], res[1][0])
    np.testing.assert_array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("det,P,n,nz,step", [(16, 16, 72, 56, 4), (8, 8, 40, 40, 8),
                                             (32, 32, 64, 64, 8), (64, 20, 90, 80, 9)])
@pytest.mark.parametrize("model", ["poisson", "gaussian"])
def test_ptycho_linesearch_sweep_is_its_parts(det, P, n, nz, step, model):
    """pt_ptycho_linesearch_sweep against pt_ptycho_linesearch and
    pt_k_ls_select over a whole search: the same state, step and candidates
    after every sweep (the sums differ in FP64 order only), for frames on the
    overlap-add tiles, sparse ones, 32 x 32 ones and 64 x 64 ones with a large
    probe; directions along and against the gradient and a long one."""
    import ctypes
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"sweep det={det} P={P} {model}", flush=True)
    rng = np.random.default_rng(n + det)
    nt, chunk, cp, cd = 6, 2, 1.1, 0.9
    nc, mdl = nt // chunk, _lib.PT_MODEL[model]
    scan = objects.jittered_raster(nt, nz, n, P, step, 1.0, rng)
    op = ptychofft(nt, nz, n, nt, scan.shape[2], det, det, P)
    sc, pr = dev(scan), dev(objects.gaussian_probe(P, P / 4) * np.float32(3))
    op.setobj(sc.data_ptr(), pr.data_ptr())
    sh = (nt, nz, n)
    t = dict(psi=np.exp(1j * 0.3 * rng.standard_normal(sh)), h=crandn(rng, sh),
             lamd=crandn(rng, sh) * 0.1,
             data=rng.poisson(4.0, (nt, scan.shape[2], det, det)).astype(np.float32))
    t = {k: dev(v if k == "data" else v.astype(np.complex64)) for k, v in t.items()}
    d = torch.zeros(sh, dtype=torch.complex64, device="cuda")
    _lib.call("pt_ptycho_grad", op._h, ptr(d), ptr(t["psi"]), ptr(t["data"]), ptr(t["h"]),
              ptr(t["lamd"]), 0.7, None, cp, cd, mdl, stream())
    d *= -0.2
    d[chunk:2 * chunk] *= 30.0
    d[2 * chunk:] *= -1.0
    w = torch.tensor([1.0, 0.7], dtype=torch.float64, device="cuda")
    z = lambda k: torch.zeros(k, dtype=torch.float64, device="cuda")  # noqa: E731
    sched = (2, 5) + (7,) * 5 + (3,)
    runs = []
    for fused in (False, True):
        state, stp, f1, f2 = z(2 * nc), z(2 * nc), z(8 * nc), z(8 * nc)
        bufs = [z(8 * nc), z(8 * nc)]
        state[0::2] = 2.0
        _lib.call("pt_k_ls_begin", ptr(state), ptr(bufs[0]), nc, sched[0] + 1, stream())
        trace = []
        for s, k in enumerate(sched):
            last = int(s == len(sched) - 1)
            ng, nx = k + 1, (sched[s] if last else sched[s + 1]) + 1
            cur, nxt = bufs[s % 2], bufs[(s + 1) % 2]
            a = _lib.LinesearchArgs(op._h, f1.data_ptr(), f2.data_ptr(), t["psi"].data_ptr(),
                                    d.data_ptr(), t["data"].data_ptr(), t["h"].data_ptr(),
                                    t["lamd"].data_ptr(), 0.7, None, cur.data_ptr(), chunk, cp, cd,
                                    state.data_ptr())
            if fused:
                _lib.call("pt_ptycho_linesearch_sweep", ctypes.byref(a), ptr(nxt), ptr(stp), ptr(w),
                          ng, nx, last, mdl, stream())
            else:
                _lib.call("pt_ptycho_linesearch", op._h, ptr(f1), ptr(f2), ptr(t["psi"]), ptr(d),
                          ptr(t["data"]), ptr(t["h"]), ptr(t["lamd"]), 0.7, None, ptr(cur), ng,
                          chunk, cp, cd, mdl, ptr(state), stream())
                _lib.call("pt_k_ls_select", ptr(state), ptr(cur), ptr(nxt), ptr(stp), ptr(f1),
                          ptr(f2), ptr(w), nc, ng, nx, last, stream())
            trace.append([x.cpu().numpy().copy() for x in (state, stp, nxt)])
        runs.append(trace)
    print("steps", runs[1][-1][1][0::2])
    for a, b in zip(*runs):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
    assert np.all(runs[1][-1][0][1::2] == 1.0)


@pytest.mark.parametrize("nz,ny,nx,nt", [(1, 5, 7, 3), (9, 33, 16, 11)])
def test_admm_tail_passes_vs_fp64(nz, ny, nx, nt):
    """pt_k_split_update and pt_k_object_update against FP64: updated states and
    the residual sums; a part of the soft threshold's arguments below it.  The
    arithmetic is a few FP32 operations per element: relative 1e-6."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd._dev import ptr, stream
    print(f"admm tail {nz}x{ny}x{nx} {nt}", flush=True)
    rng = np.random.default_rng(nx)
    u, e0 = crandn(rng, (nz, ny, nx)), crandn(rng, (3, nz, ny, nx))
    mu = crandn(rng, (3, nz, ny, nx))
    tau, alpha, rho, c, ps = 0.5, 3.0, 2.0, 0.3, 0.7
    blk = torch.tensor([tau, rho, ps, np.cos(ps), np.sin(ps), 0, 0, 0, 0], dtype=torch.float64,
                       device="cuda")
    at = lambda k: blk.data_ptr() + 8 * k  # noqa: E731
    t = {k: dev(v) for k, v in dict(u=u, e=e0, mu=mu, phi=np.zeros_like(mu)).items()}
    _lib.call("pt_k_split_update", at(5), ptr(t["phi"]), ptr(t["e"]), ptr(t["mu"]), ptr(t["u"]),
              at(0), alpha, nz, ny, nx, stream())
    U = u.astype(np.complex128)
    g = np.zeros((3, nz, ny, nx), np.complex128)
    g[0, :, :, :-1], g[1, :, :-1], g[2, :-1] = np.diff(U, axis=2), np.diff(U, axis=1), np.diff(U, axis=0)
    g *= 2 / np.sqrt(3)
    q = g + mu / tau
    za = np.sqrt((np.abs(q) ** 2).sum(0))
    assert 0 < (za <= alpha / tau).sum() < za.size
    phi = np.where(za <= alpha / tau, 0, q - alpha / tau * q / za)
    sh = (nt, nz, nx)
    h, lamd, psi, Ru = (crandn(rng, sh) for _ in range(4))
    o = {k: dev(v) for k, v in dict(h=h, lamd=lamd, psi=psi, Ru=Ru).items()}
    _lib.call("pt_k_object_update", at(7), ptr(o["h"]), ptr(o["lamd"]), ptr(o["psi"]), ptr(o["Ru"]),
              c, at(2), at(1), h.size, stream())
    hn = np.exp(1j * np.float32(c) * Ru.astype(np.complex128)) * np.exp(1j * ps)
    ref = dict(phi=phi, e=g, mu=mu + tau * (g - phi), h=hn, lamd=lamd + rho * (hn - psi))
    for k, v in ref.items():
        d = rel({**t, **o}[k].cpu().numpy(), v)
        print(k, f"{d:.2e}")
        assert d < 1e-6, (k, d)
    n = blk.cpu().numpy()[5:]
    sq = lambda x: (np.abs(x) ** 2).sum()  # noqa: E731
    np.testing.assert_allclose(n, [sq(phi - g), sq(g - e0), sq(psi - hn), sq(hn - h)], rtol=2e-6)


def _device_us(f, reps=20, rounds=7):
    """device time of one call among `reps` back to back: the least of `rounds`"""
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    f()
    best = np.inf
    for _ in range(rounds):
        a.record()
        for _ in range(reps):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / reps)
    return best


@pytest.mark.parametrize("det,P,n,step", [(32, 32, 128, 16), (64, 16, 128, 16), (64, 9, 90, 10)])
def test_ptycho_fwd_patches_per_wave(det, P, n, step):
    """Large frames' far fields with one to four patches per wave (the counts
    around the rule's steps, 4096 patches per step): each angle's as the
    operator of a few angles gives it, bit for bit.  And a few hundred patches,
    which fit the device at once, take no longer than 1.8 times what four take
    (four patches in a row on a quarter of the waves took 2.3 to 3.3 times)."""
    from ptychotomo_amd import objects
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"fwd patches per wave det={det} P={P}", flush=True)
    S = objects.jittered_raster(1, n, n, P, step, 1.0, np.random.default_rng(0)).shape[2]
    nt = 4 * 4096 // S + 2
    rng = np.random.default_rng(det + P)
    scan = objects.jittered_raster(nt, n, n, P, step, 1.0, rng)
    psi = dev(np.exp(1j * 0.3 * rng.standard_normal((nt, n, n))).astype(np.complex64))
    pr = dev(objects.gaussian_probe(P, P / 4))

    def op_of(nta, nscan):
        op = ptychofft(nta, n, n, nta, nscan, det, det, P)
        sc = dev(np.ascontiguousarray(scan[:, :nta, :nscan]))
        op.setobj(sc.data_ptr(), pr.data_ptr())
        return op, torch.empty((nta, nscan, det, det), dtype=torch.complex64, device="cuda")
    one, ref = op_of(1, S)
    one.fwd(ref.data_ptr(), psi.data_ptr())
    for k in range(1, 5):
        for nta in (k * 4096 // S, k * 4096 // S + 1):
            op, far = op_of(nta, S)
            op.fwd(far.data_ptr(), psi.data_ptr())
            assert torch.equal(far[0], ref[0]), (k, nta)
            few, last = op_of(1, S)
            sc = dev(np.ascontiguousarray(scan[:, nta - 1:nta]))
            few.setobj(sc.data_ptr(), pr.data_ptr())
            few.fwd(last.data_ptr(), psi[nta - 1].data_ptr())
            assert torch.equal(far[-1], last[0]), (k, nta)
    four, f4 = op_of(1, 4)
    many, fm = op_of(max(1, 256 // S), S)
    t4 = _device_us(lambda: four.fwd(f4.data_ptr(), psi.data_ptr()))
    tm = _device_us(lambda: many.fwd(fm.data_ptr(), psi.data_ptr()))
    print(f"4 patches {t4:.1f} us, {fm.shape[0] * S} patches {tm:.1f} us")
    assert tm < 1.8 * t4, (t4, tm)


@pytest.mark.parametrize("nt,nz,n", [(8, 32, 180), (130, 64, 128), (16, 208, 204)])
def test_tomo_linesearch_groups_of_halvings(nt, nz, n):
    """pt_k_tomo_linesearch where all later groups of halvings share a sweep,
    where the first two have their own and where every group has: the steps of
    the search made from its parts, accepted in each group and never.  And a step
    accepted at the tenth halving (second group) of a problem that memory bounds
    takes no longer than 2.8 times one accepted at the second (reading everything
    once more is 1.6 times; evaluating all later groups for it took 3.5)."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd._dev import ptr, stream
    print(f"tomo line search groups nt={nt} nz={nz} n={n}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    cr = lambda *sh: torch.view_as_complex(  # noqa: E731
        torch.randn((*sh, 2), generator=gen, device="cuda"))

    def J(v):
        o = torch.zeros((3, *v.shape), dtype=v.dtype, device="cuda")
        o[0, :, :, :-1], o[1, :, :-1], o[2, :-1] = (v.diff(dim=k) for k in (2, 1, 0))
        return o * (2 / 3 ** 0.5)

    z = lambda *v: torch.tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    w = z(0.5, 0.25)

    def search(nt, nz, n, fits):
        K, Ru, Rd = (cr(nt, nz, n) for _ in range(3))
        u, d = cr(nz, n, n), cr(nz, n, n)
        for fit in fits:
            xi0, xi1 = K * (Ru + 0.9 * fit * Rd), J(u + 0.9 * fit * d)
            state, step = z(2.0, 0.0), z(7.0, 7.0)

            def run():
                state[0] = 2.0
                _lib.call("pt_k_tomo_linesearch", ptr(state), ptr(step), ptr(K), ptr(Ru), ptr(Rd),
                          ptr(xi0), ptr(u), ptr(d), ptr(xi1), ptr(w), K.numel(), nz, n, n,
                          stream())

            def parts():
                s2, p2 = z(2.0, 0.0), z(7.0, 7.0)
                c, f1, f2 = (torch.zeros(8, dtype=torch.float64, device="cuda") for _ in range(3))
                _lib.call("pt_k_ls_begin", ptr(s2), ptr(c), 1, 8, stream())
                for sw in range(6):
                    _lib.call("pt_k_tomo_minf", ptr(f1), ptr(K), ptr(Ru), ptr(Rd), ptr(xi0), ptr(c),
                              8, K.numel(), ptr(s2), stream())
                    _lib.call("pt_k_reg_minf", ptr(f2), ptr(u), ptr(d), ptr(xi1), ptr(c), 8, nz, n,
                              n, ptr(s2), stream())
                    _lib.call("pt_k_ls_select", ptr(s2), ptr(c), ptr(c), ptr(p2), ptr(f1), ptr(f2),
                              ptr(w), 1, 8, 8, int(sw == 5), stream())
                return s2, p2
            run()
            yield fit, run, step, state, parts

    for fit, _, step, state, parts in search(nt, nz, n, [1.0, 2.0 ** -8, 2.0 ** -15, 2.0 ** -22, -1.0]):
        s2, p2 = parts()
        print(fit, step.tolist(), p2.tolist())
        assert torch.equal(step, p2) and torch.equal(state, s2), fit
        if fit > 0:
            assert 0.45 * fit < step[0].item() <= 1.8 * fit
    if nt == 130:
        us = [_device_us(run, 5) for _, run, *_ in search(192, 128, 128, [1.0, 2.0 ** -9])]
        print("accepted in the first, second group:", us)
        assert us[1] < 2.8 * us[0], us


@pytest.mark.parametrize("det,P,n,nz,step", [(8, 8, 40, 33, 3), (8, 8, 33, 40, 2), (8, 5, 33, 40, 2),
                                             (16, 16, 64, 49, 4), (16, 11, 50, 61, 3),
                                             (32, 32, 64, 64, 8), (64, 16, 64, 64, 6),
                                             (64, 20, 90, 80, 9)])
@pytest.mark.parametrize("model", ["poisson", "gaussian"])
def test_ptycho_grad_rounds_its_products_alike(det, P, n, nz, step, model):
    """The gradient's FP64 transforms take the products probe x object rounded
    one way (a multiply-add whose second product is rounded first), whatever the
    frame size and probe form: against FP64 from products rounded so, what is left
    is the rounding of residual, FP32 inverse and sums, a few ulp.  With the
    other product rounded first the Poisson residual differs by 3e-7 to 3e-6."""
    from ptychotomo_amd import _lib, objects
    from ptychotomo_amd._dev import ptr, stream
    from ptychotomo_amd.ptychofft import ptychofft
    print(f"grad products det={det} P={P} {model}", flush=True)
    nt, cp, cd, rho = 3, np.float32(1.1), np.float32(0.9), 0.7
    for seed in range(2):
        rng = np.random.default_rng(1000 * det + 10 * P + seed)
        scan = objects.jittered_raster(nt, nz, n, P, step, 1.0, rng)
        S = scan.shape[2]
        prb = objects.gaussian_probe(P, P / 4) * np.exp(1j * rng.standard_normal((P, P)))
        prb = prb.astype(np.complex64)
        op = ptychofft(nt, nz, n, nt, S, det, det, P)
        sc, pr = dev(scan), dev(prb)
        op.setobj(sc.data_ptr(), pr.data_ptr())
        psi, h, lamd = (crandn(rng, (nt, nz, n)) for _ in range(3))
        data = rng.poisson(4.0, (nt, S, det, det)).astype(np.float32)
        a = [dev(v) for v in (psi, data, h, lamd)]
        out = torch.zeros((nt, nz, n), dtype=torch.complex64, device="cuda")
        _lib.call("pt_ptycho_grad", op._h, ptr(out), *(ptr(v) for v in a), rho, None, float(cp),
                  float(cd), _lib.PT_MODEL[model], stream())
        far = _product_far(psi, prb, scan, det, True) / det * np.float64(cp)
        d, m = data * np.float64(cd), np.abs(far)
        res = far - (d / (m ** 2 + 1e-32) if model == "poisson" else np.sqrt(d) / m) * far
        res = np.fft.ifft2(res) * det * np.float64(cp)
        ref = -rho * (h - psi.astype(np.complex128) + lamd / rho)
        pos, o = np.floor(scan + 0.5).astype(int), (det - P) // 2
        for t, s in np.ndindex(nt, S):
            x, y = pos[:, t, s]
            ref[t, y:y + P, x:x + P] += (res[t, s, o:o + P, o:o + P] * prb.conj()).T
        e = rel(out.cpu().numpy(), ref)
        print(f"rel {e:.2e}")
        assert e < 2.5e-7, e


@pytest.mark.parametrize("nt,nz,ny,nx", [(3, 1, 5, 7), (5, 9, 33, 16), (2, 4, 1, 300)])
def test_cg_step_passes(nt, nz, ny, nx):
    """The element-wise passes of a cg_tomo step: pt_k_cg_resid (with and without
    the previous step's update of Ru) and pt_k_cg_reg_grad, and their parts
    pt_k_axpy_seg, pt_k_tomo_resid and pt_k_reg_grad with their sums, against
    FP64.  A few FP32 operations per element: relative 1e-6."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd._dev import ptr, stream
    print(f"cg step passes {nt} {nz}x{ny}x{nx}", flush=True)
    rng = np.random.default_rng(nx)
    K, Ru, Rd, xi0 = (crandn(rng, (nt, nz, nx)) for _ in range(4))
    u, grad, xi1 = crandn(rng, (nz, ny, nx)), crandn(rng, (nz, ny, nx)), crandn(rng, (3, nz, ny, nx))
    z = lambda *v: torch.tensor(v, dtype=torch.float64, device="cuda")  # noqa: E731
    step, rho, tau, sums = z(0.3, 0.0), z(0.7), z(1.9), z(-1.0, -1.0)
    Kd, Rdd, xd, st = dev(K), dev(Rd), dev(xi0), stream()
    for upd in (False, True):
        r, r2, a, b = dev(np.zeros_like(Ru)), dev(np.zeros_like(Ru)), dev(Ru), dev(Ru)
        _lib.call("pt_k_cg_resid", ptr(r), ptr(a), ptr(Rdd) if upd else None, ptr(step), ptr(Kd),
                  ptr(xd), ptr(rho), Ru.size, st)
        if upd:
            _lib.call("pt_k_axpy_seg", ptr(b), ptr(step), ptr(Rdd), Ru.size, 1, st)
        _lib.call("pt_k_tomo_resid", ptr(r2), ptr(sums), ptr(Kd), ptr(b), ptr(xd), 0.0, ptr(rho),
                  Ru.size, st)
        new = Ru.astype(np.complex128) + 0.3 * upd * Rd
        e = K.astype(np.complex128) * new - xi0
        ref = 0.7 * K.conj() * e
        errs = [rel(a.cpu().numpy(), new), rel(r.cpu().numpy(), ref), rel(r2.cpu().numpy(), ref)]
        print("Ru, r, r of the parts", errs)
        assert max(errs) < 1e-6
        assert rel(a.cpu().numpy(), b.cpu().numpy()) < 1e-7
        assert rel(r.cpu().numpy(), r2.cpu().numpy()) < 5e-7
        np.testing.assert_allclose(sums[0].item(), (np.abs(e) ** 2).sum(), rtol=1e-6)
    ud, x1, g1, g2 = dev(u), dev(xi1), dev(grad), dev(grad)
    _lib.call("pt_k_cg_reg_grad", ptr(g1), ptr(ud), ptr(x1), ptr(tau), nz, ny, nx, st)
    _lib.call("pt_k_reg_grad", ptr(g2), ptr(sums), ptr(ud), ptr(x1), 0.0, ptr(tau), nz, ny, nx, st)
    c, w = 2 / np.sqrt(3), np.zeros((3, nz, ny, nx), np.complex128)
    U = u.astype(np.complex128)
    w[0, :, :, :-1], w[1, :, :-1], w[2, :-1] = (np.diff(U, axis=k) * c for k in (2, 1, 0))
    w -= xi1
    d = w.sum(0)
    d[:, :, 1:] -= w[0, :, :, :-1]
    d[:, 1:] -= w[1, :, :-1]
    d[1:] -= w[2, :-1]
    ref = grad - 1.9 * c * d
    errs = [rel(g1.cpu().numpy(), ref), rel(g2.cpu().numpy(), ref)]
    print("grad, grad of the reducing pass", errs)
    assert max(errs) < 1e-6
    np.testing.assert_allclose(sums[0].item(), (np.abs(w) ** 2).sum(), rtol=1e-6)


def test_intensity_of_a_far_field():
    """pt_k_intensity (out = scale |x|^2) against numpy, with a length that is no
    multiple of a wave."""
    from ptychotomo_amd import _lib
    from ptychotomo_amd._dev import ptr, stream
    x = crandn(np.random.default_rng(3), (1037,))
    out = torch.zeros(x.size, dtype=torch.float32, device="cuda")
    xd = dev(x)
    _lib.call("pt_k_intensity", ptr(out), ptr(xd), 0.4, x.size, stream())
    ref = np.float64(np.float32(0.4)) * np.abs(x.astype(np.complex128)) ** 2
    assert rel(out.cpu().numpy(), ref) < 3e-7
