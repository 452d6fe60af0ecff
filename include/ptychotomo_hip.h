/*
 * ptychotomo_hip.h -- C ABI of the MI355X (gfx950) ptycho-tomography library.
 *
 * Plain C: opaque handles, raw device pointers, sizes, int status codes.
 * Complex arrays are interleaved complex64 (re, im float pairs), C order.
 * Every pointer argument named as a buffer is a device pointer; the library
 * never reads host memory through them.  `stream` is a hipStream_t (NULL =
 * the null stream).  Calls only enqueue work, except the set-up calls
 * (*_create, pt_tomo_set_theta, pt_ptycho_set_scan_probe), which block.
 * A handle owns scratch memory and must not be used by two streams at once.
 *
 * Status codes: PT_OK (0) or a negative PT_ERR_*; pt_last_error() returns a
 * thread-local message for the last failure.
 *
 * Reference interfaces replaced (paths relative to the reference tree):
 *   class radonusfft   src/include/radonusfft.cuh:3-37, src/cuda/radonusfft.i:15-46
 *   class ptychofft    src/include/ptychofft.cuh:3-36,  src/cuda/ptychofft.i:14-48
 *   CuPy chains of     src/ptychotomo/solver.py (solver kernels, pt_k_*)
 */
#ifndef PTYCHOTOMO_HIP_H
#define PTYCHOTOMO_HIP_H

#ifdef __cplusplus
extern "C" {
#endif

#define PT_OK 0
#define PT_ERR_ARG (-1)   /* null handle / pointer, bad enum */
#define PT_ERR_SIZE (-2)  /* size precondition violated (n%4, radix, ...) */
#define PT_ERR_HIP (-3)   /* HIP runtime error */
#define PT_ERR_STATE (-4) /* e.g. operator called before set_theta */

#define PT_MODEL_GAUSSIAN 0
#define PT_MODEL_POISSON 1

/* Detector-frequency filters of the tomography adjoint. */
#define PT_FILTER_NONE 0
#define PT_FILTER_RAMP 1

/* Line-pass kernels of the tomography operators (pt_tomo_set_line_kernels). */
#define PT_LINES_AUTO 0
#define PT_LINES_GENERIC 1

typedef struct pt_tomo pt_tomo;
typedef struct pt_ptycho pt_ptycho;
typedef void* pt_stream; /* hipStream_t */

/* Thread-local text of the last error (never NULL). */
const char* pt_last_error(void);
/* Library ABI version (increments on incompatible change). */
int pt_abi_version(void);
/* First 16 hex digits of the SHA-256 of this header's text at build time.
 * A binding compares it with the header it was written against and refuses
 * a library built from another one: calling a function whose parameter list
 * differs from the caller's (a stale build) passes arguments in the wrong
 * registers -- e.g. an integer where the stream handle is expected -- and
 * crashes inside the HIP runtime instead of failing cleanly. */
const char* pt_header_digest(void);

/* Launch profiler (no reference counterpart; measurement only).  After
 * pt_prof_start(tag), every launch of the kernel named `tag` (e.g.
 * "tomo_gather", "tomo_scatter", "ptycho_grad_tile") is bracketed by HIP
 * events on its launch stream; pt_prof_stop synchronises on them and returns
 * the summed kernel time and the launch count. */
int pt_prof_start(const char* tag);
int pt_prof_stop(double* total_ms, long* launches);

/* ------------------------------------------------------------------ tomo
 * USFFT Radon transform on a slab of pnz slices of an n x n object.
 * f: [pnz, n, n] complex64, g: [ntheta, pnz, n] complex64.
 */

/* radonusfft::radonusfft(Ntheta, Nz, N)  radonusfft.cu:5-39.
 * Requires n % 4 == 0 and 3n/2 factorable into radices {2,3,4,5,8}. */
int pt_tomo_create(int ntheta, int pnz, int n, pt_tomo** out);
/* radonusfft::~radonusfft  radonusfft.cu:41-52 */
int pt_tomo_destroy(pt_tomo* h);
/* radonusfft::setobj(theta)  radonusfft.cu:141-144.  theta: [ntheta] float32
 * device array.  Also builds the sample-position tables and the tile bins of
 * the deterministic adjoint gridding (blocking). */
int pt_tomo_set_theta(pt_tomo* h, const float* theta, pt_stream stream);
/* radonusfft::fwd(g, f)  radonusfft.cu:54-92 (unnormalised). */
int pt_tomo_fwd(pt_tomo* h, void* g, const void* f, pt_stream stream);
/* radonusfft::adj(f, g)  radonusfft.cu:94-139 (unnormalised, with the
 * reference's edge-replicating detector pad). */
int pt_tomo_adj(pt_tomo* h, void* f, const void* g, pt_stream stream);
/* Same operators with the output multiplied by `scale` (solver.py:71,79
 * multiply by coeftomo after the native call). */
int pt_tomo_fwd_scaled(pt_tomo* h, void* g, const void* f, float scale, pt_stream stream);
int pt_tomo_adj_scaled(pt_tomo* h, void* f, const void* g, float scale, pt_stream stream);
/* Filter applied by every later adjoint between its detector DFT and the
 * gridding: PT_FILTER_RAMP is applyfilter (kernels.cuh:174-187, the
 * commented-out step at radonusfft.cu:121), i.e. filtered backprojection;
 * PT_FILTER_NONE (the default) restores radonusfft::adj.  Blocking. */
int pt_tomo_set_filter(pt_tomo* h, int kind);
/* Launch shapes of the USFFT passes (no counterpart in the reference; set by
 * the autotuner): FFT lines per workgroup of the row pass (rows, two
 * N-point FFTs each), grid columns per workgroup of the column passes (cols,
 * a power of two whose N x cols tile fits the per-thread registers) and
 * (angle, slice) lines per workgroup of the detector-line passes, forward
 * inverse DFT and adjoint DFT (adj_lines <= 8).  Rejected if a shape does
 * not fit 64 KB of LDS; results do not depend on them. */
int pt_tomo_get_tuning(pt_tomo* h, int* rows, int* cols, int* adj_lines);
int pt_tomo_set_tuning(pt_tomo* h, int rows, int cols, int adj_lines);
/* Which kernels run the USFFT's row, column and detector-line passes (no
 * counterpart in the reference): PT_LINES_AUTO (the default) uses the
 * register line FFT (fixed launch shapes; the tuning above is then unused)
 * for n = 64, 96, 128, 192, 256, 512 and the generic LDS FFT (tuned shapes)
 * for other n; PT_LINES_GENERIC always uses the generic one.  Both compute the
 * same transform; FP32 sums run in a different order. */
int pt_tomo_set_line_kernels(pt_tomo* h, int kind);
/* *reg = 1 if this handle's line passes run on the register line FFT
 * (PT_LINES_AUTO and a supported n), else 0, when the launch shapes of
 * pt_tomo_set_tuning apply (no counterpart in the reference). */
int pt_tomo_get_line_kernels(pt_tomo* h, int* reg);

/* ---------------------------------------------------------------- ptycho
 * Probe x object patch, D x D far field per scan position.
 * f: [ptheta, nz, n] complex64, g: [ptheta, nscan, detx, dety] complex64.
 */

/* ptychofft::ptychofft(Ntheta, Nz, N, Ntheta0, Nscan, detx, dety, Nprb)
 * ptychofft.cu:5-33 (Ntheta0 is unused there and here).
 * Requires detx == dety in {8,16,32,64} and nprb <= detx.
 * 64 x 64 frames with nprb > 16 run a lane per frame row: a line-search sweep of 6
 * candidates takes about 0.8 ms per 1000 frames, with nprb <= 16 (one wave per frame)
 * 0.025 ms; gradients and adjoints 2 to 7 times as long as with nprb <= 16. */
int pt_ptycho_create(int ptheta, int nz, int n, int ntheta0, int nscan, int detx, int dety,
                     int nprb, pt_ptycho** out);
/* ptychofft::~ptychofft  ptychofft.cu:35-46 */
int pt_ptycho_destroy(pt_ptycho* h);
/* ptychofft::setobj(scan, prb)  ptychofft.cu:48-56.  scan: [2, ptheta, nscan]
 * float32 (x plane first), prb: [nprb, nprb] complex64, device arrays.
 * Rounds positions, builds the shift factors and the tile bins of the
 * deterministic overlap-add (blocking).  Positions whose rounded value
 * places the probe outside the object are rejected (PT_ERR_ARG); negative
 * rounded positions are skipped, as in the reference. */
int pt_ptycho_set_scan_probe(pt_ptycho* h, const float* scan, const void* prb, pt_stream stream);
/* ptychofft::fwd(g, f)  ptychofft.cu:58-76 (unnormalised). */
int pt_ptycho_fwd(pt_ptycho* h, void* g, const void* f, pt_stream stream);
/* ptychofft::adj(f, g)  ptychofft.cu:78-93 (unnormalised). */
int pt_ptycho_adj(pt_ptycho* h, void* f, const void* g, pt_stream stream);
/* Same with the output multiplied by `scale` (coefptycho, solver.py:104,124). */
int pt_ptycho_fwd_scaled(pt_ptycho* h, void* g, const void* f, float scale, pt_stream stream);
int pt_ptycho_adj_scaled(pt_ptycho* h, void* f, const void* g, float scale, pt_stream stream);
/* Far-field intensities (solver.py:115) without the far field: out =
 * iscale * |scale * F f|^2, out: [ptheta, nscan, detx, dety] float32. */
int pt_ptycho_intensity(pt_ptycho* h, float* out, const void* f, float scale, float iscale,
                        pt_stream stream);

/* Fused ptychography gradient of cg_ptycho (solver.py:219-225):
 *   fpsi = coefptycho * F(psi)
 *   r    = fpsi - d*fpsi/(|fpsi|^2+1e-32)          (poisson)
 *        = fpsi - sqrt(d)*exp(i*angle(fpsi))        (gaussian)
 *   grad = coefptycho * F*(r) - rho*(h - psi + lamd/rho)
 * with d = coefdata*data, data: [ptheta, nscan, detx, dety] float32.
 * The far field is never written to memory.  rho_dev, if not NULL, is a
 * device FP64 scalar used instead of rho. */
int pt_ptycho_grad(pt_ptycho* h, void* grad, const void* psi, const float* data, const void* hh,
                   const void* lamd, double rho, const double* rho_dev, float coefptycho,
                   float coefdata, int model, pt_stream stream);

/* One instance of pt_ptycho_grad_group: the arguments of pt_ptycho_grad. */
typedef struct pt_ptycho_grad_args {
  pt_ptycho* h;
  void* grad;
  const void* psi;
  const float* data;
  const void* hh;
  const void* lamd;
  double rho;
  const double* rho_dev;
  float coefptycho;
  float coefdata;
} pt_ptycho_grad_args;

/* pt_ptycho_grad for n independent reconstructions at once (no counterpart in
 * the reference: the batched solver's multi-instance launch).  Instances with
 * the same detector size share one overlap-add tile launch and one fold
 * launch (up to 8 per launch, every instance's tiles in one grid).  Results
 * are identical to n separate pt_ptycho_grad calls. */
int pt_ptycho_grad_group(const pt_ptycho_grad_args* a, int n, int model, pt_stream stream);
/* Data term of the cg_ptycho functional (solver.py:208-212) at ngam step
 * candidates psi + gamma*d, segmented by angle chunks of `chunk` angles, as
 * its change from gamma = 0 (the quantity the halving rule decides on):
 *   sums[c*ngam + j] = sum_{chunk c} t(a_j) - t(a_0),
 *   t(a) = |a|^2 - 2 d mlog|a|  (poisson),  (|a| - sqrt(d))^2  (gaussian),
 *   a_j = coefptycho*F(psi) + gammas[c*ngam+j]*coefptycho*F(dir) formed in FP32,
 * evaluated per element (difference of squares as a product, log ratio as
 * log1p) and summed in FP64.
 * sums, gammas: device FP64 arrays.  dir may be NULL (then only gamma = 0
 * is meaningful).  With lagr != 0 the poisson sum also subtracts
 * d - 2 d mlog(sqrt d), giving lagr[0] of take_lagr (solver.py:294-296).
 * skip, if not NULL, is a line-search state (pt_k_ls_begin): chunks whose
 * search has finished are not evaluated. */
int pt_ptycho_minf(pt_ptycho* h, double* sums, const void* psi, const void* dir, const float* data,
                   const double* gammas, int ngam, int chunk, float coefptycho, float coefdata,
                   int model, int lagr, const double* skip, pt_stream stream);

/* The whole line-search evaluation of cg_ptycho (solver.py:208-213) at ngam
 * step candidates per angle chunk, in one pass over the overlap-add tiles:
 * f1 = the data term's change as pt_ptycho_minf (lagr = 0), and
 *   f2[c*ngam + j] = sum_{chunk c} |h - (psi + g_j*dir) + lamd/rho|^2
 *                                - |h - psi + lamd/rho|^2,
 * psi + g_j*dir formed in FP32 per element, summed in FP64 (the halving rule
 * takes f1 + rho*f2).  Each tile sums the rho term over the pixels it owns
 * (the tiles of an angle partition the object).  Frames or scans that do not
 * take the tile kernel compute f2 with pt_k_rho_minf.  rho_dev, if not NULL,
 * is a device FP64 scalar used instead of rho. */
int pt_ptycho_linesearch(pt_ptycho* h, double* f1, double* f2, const void* psi, const void* dir,
                         const float* data, const void* hh, const void* lamd, double rho,
                         const double* rho_dev, const double* gammas, int ngam, int chunk,
                         float coefptycho, float coefdata, int model, const double* skip,
                         pt_stream stream);

/* One instance of pt_ptycho_linesearch_group: the arguments of
 * pt_ptycho_linesearch that differ between instances. */
typedef struct pt_ptycho_linesearch_args {
  pt_ptycho* h;
  double* f1;
  double* f2;
  const void* psi;
  const void* dir;
  const float* data;
  const void* hh;
  const void* lamd;
  double rho;
  const double* rho_dev;
  const double* gammas;
  int chunk;
  float coefptycho;
  float coefdata;
  const double* skip;
} pt_ptycho_linesearch_args;

/* One sweep of cg_ptycho's line search: pt_ptycho_linesearch at the ngam
 * candidates a->gammas of the chunks that the search state a->skip leaves
 * open (updated in place), then pt_k_ls_select with the weights w; a->f1 and
 * a->f2 are not used. */
int pt_ptycho_linesearch_sweep(const pt_ptycho_linesearch_args* a, double* cand_next, double* step,
                               const double* w, int ngam, int ngam_next, int last, int model,
                               pt_stream stream);

/* pt_ptycho_linesearch for n independent reconstructions at once (no
 * counterpart in the reference, which reconstructs one object per run: the
 * batched solver's multi-instance launch).  Instances that take the
 * overlap-add tile kernel with the same detector size and probe form share
 * one launch (up to 8 per launch: every instance's tiles in one grid, its
 * arguments passed by value) and two grouped reductions; the others run as
 * pt_ptycho_linesearch.  Results are identical to n separate calls (each
 * tile's partial sums have their own slot, summed in a fixed order).  All
 * instances use ngam candidates and the given model. */
int pt_ptycho_linesearch_group(const pt_ptycho_linesearch_args* a, int n, int ngam, int model,
                               pt_stream stream);
/* One sweep of the line search of n independent reconstructions (the arguments
 * of pt_ptycho_linesearch_sweep that differ between them in s): grouped as
 * pt_ptycho_linesearch_group, with the decisions of a group in one launch.
 * Sums, their order and decisions are those of n calls of
 * pt_ptycho_linesearch_sweep, bit for bit. */
typedef struct pt_ptycho_sweep_args {
  double* cand_next;
  double* step;
  const double* w;
} pt_ptycho_sweep_args;
int pt_ptycho_linesearch_sweep_group(const pt_ptycho_linesearch_args* a,
                                     const pt_ptycho_sweep_args* s, int n, int ngam, int ngam_next,
                                     int last, int model, pt_stream stream);

/* pt_ptycho_minf for callers that cannot allocate device memory (code under
 * HIP graph capture, serving loops, harnesses that forbid hipMalloc).  No
 * counterpart in the reference.  Same arguments and results as
 * pt_ptycho_minf (the same kernels); its per-launch partial sums live in a
 * fixed per-device array of PT_MINF_NOALLOC_PARTIALS doubles (16 MiB, held
 * until the process ends) instead of the handle's buffer, and the call
 * allocates nothing.  A launch of more partial sums than that fails with
 * PT_ERR_SIZE; on overlap-add tiles they are counted as two per tile and
 * candidate (the limit is ~1 M tiles x candidates; the 256^3, 384-angle workload
 * with 8 candidates counts 1.6 M), though the kernel writes fewer.  Calls that
 * overlap on one device share the array and race: serialise them (one
 * stream, or events). */
#define PT_MINF_NOALLOC_PARTIALS (2 * 1024 * 1024)
int pt_ptycho_minf_noalloc(pt_ptycho* h, double* sums, const void* psi, const void* dir,
                           const float* data, const double* gammas, int ngam, int chunk,
                           float coefptycho, float coefdata, int model, int lagr,
                           const double* skip, pt_stream stream);

/* ------------------------------------------------------- solver kernels
 * Complex64 vectors of length `len`, optionally split into `nseg` equal
 * contiguous segments (per-chunk scalars).  Reductions accumulate in FP64
 * and write their results to device memory.  Scalar arrays named *_dev are
 * device FP64 arrays indexed by segment (complex scalars as re,im pairs).
 * A real scalar argument x with a companion `const double* x_dev` is read
 * from device memory when x_dev is not NULL (the device-driven solver keeps
 * rho, tau and the takexi phase there).
 */
/* out[2*s..] = sum_seg conj(x)*y */
int pt_k_dot(double* out, const void* x, const void* y, long len, int nseg, pt_stream stream);
/* out[s] = sum_seg |x|^2 */
int pt_k_norm2(double* out, const void* x, long len, int nseg, pt_stream stream);
/* out[s] = sum_seg |a*x + b*y|^2 with complex host scalars a, b */
int pt_k_norm2_lin(double* out, const void* x, const void* y, double ar, double ai, double br,
                   double bi, long len, int nseg, pt_stream stream);
/* z = a[s]*x + b[s]*y with complex device scalars (per segment); y may be NULL */
int pt_k_lincomb(void* z, const double* a_dev, const void* x, const double* b_dev, const void* y,
                 long len, int nseg, pt_stream stream);
/* Dai-Yuan direction update (solver.py:195-196, 230-231) per segment:
 *   d = -grad + beta[s]*d,  beta = ||grad||^2 / sum(conj(d)*(grad-grad0)),
 * beta given as complex device scalars; first != 0 gives d = -grad. */
int pt_k_dy_update(void* d, const void* grad, const double* beta_dev, int first, long len,
                   int nseg, pt_stream stream);
/* Dai-Yuan reductions per segment: out[3*s+0] = ||grad||^2,
 * out[3*s+1], out[3*s+2] = re, im of sum conj(d)*(grad-grad0). */
int pt_k_dy_reduce(double* out, const void* grad, const void* grad0, const void* d, long len,
                   int nseg, pt_stream stream);

/* fwd_reg (solver.py:128-134): out [3,nz,ny,nx] = J u, forward differences
 * times 2/sqrt(3), last plane 0. */
int pt_k_reg_fwd(void* out, const void* u, int nz, int ny, int nx, pt_stream stream);
/* adj_reg (solver.py:137-146): out [nz,ny,nx] = J* g (times -2/sqrt(3)). */
int pt_k_reg_adj(void* out, const void* g, int nz, int ny, int nx, pt_stream stream);
/* solve_reg (solver.py:257-264): z = J u + mu/tau, isotropic soft threshold at
 * alpha/tau over the 3 components. */
int pt_k_reg_solve(void* out, const void* u, const void* mu, double tau, const double* tau_dev,
                   double alpha, int nz, int ny, int nx, pt_stream stream);

/* exptomo (solver.py:59-60) with an optional extra phase (solver.py:322):
 * out = exp(i*c*psi) * exp(i*phase).  phase_dev, if not NULL, points to
 * {phase, cos phase, sin phase} (the prm of pt_k_takexi_dev). */
int pt_k_exptomo(void* out, const void* psi, double c, double phase, const double* phase_dev,
                 long len, pt_stream stream);
/* mlog (solver.py:48-52): log(x) with |x| < 1e-32 replaced by 1e-32. */
int pt_k_mlog(void* out, const void* x, long len, pt_stream stream);

/* takexi statistics (solver.py:151-156,164): out[0] = sum angle(psi[:,:,r:2r]),
 * out[1] = sum angle(psi[:,:,n-2r:n-r]), out[2] = max |psi - lamd/rho|. */
int pt_k_takexi_stats(double* out, const void* psi, const void* lamd, double rho,
                      const double* rho_dev, int ntheta, int nz, int n, int r, pt_stream stream);
/* takexi body (solver.py:158-167): given pshift and kscale = c/max|K_raw|:
 *   t = (psi - lamd/rho) e^{-i pshift}; K = i*kc*t*kscale;
 *   xi0 = K * (-i mlog(t) / c1) * coeftomo. */
int pt_k_takexi(void* xi0, void* K, const void* psi, const void* lamd, double rho, double pshift,
                double kc, double kscale, double c1, double coeftomo, long len, pt_stream stream);
/* takexi with its scalars formed on the device from pt_k_takexi_stats' out
 * (stats) as solver.py:149-168 forms them: pshift = float32 mean of the two
 * band means (cnt samples each), kscale = 1/(kc*max|t|) (0 if max|t| = 0);
 * prm receives {pshift, cos pshift, sin pshift, kc*kscale}. */
int pt_k_takexi_dev(void* xi0, void* K, double* prm, const void* psi, const void* lamd,
                    const double* rho_dev, const double* stats, double cnt, double kc, double c1,
                    double coeftomo, long len, pt_stream stream);

/* cg_tomo pieces (solver.py:180-203), single segment:
 * r = scale*conj(K)*(K*Ru - xi0), out[0] = ||K*Ru - xi0||^2 */
int pt_k_tomo_resid(void* r, double* out, const void* K, const void* Ru, const void* xi0,
                    double scale, const double* scale_dev, long len, pt_stream stream);
/* grad += tau * J*(J u - xi1) (adj_reg of fwd_reg residual, solver.py:188-190),
 * out[0] = ||J u - xi1||^2.  u: [nz,ny,nx], xi1: [3,nz,ny,nx]. */
int pt_k_reg_grad(void* grad, double* out, const void* u, const void* xi1, double tau,
                  const double* tau_dev, int nz, int ny, int nx, pt_stream stream);
/* Line-search candidates (solver.py:171-177), formed as the reference forms
 * them: the stepped quantity x + gamma*dx element-wise in FP32, so a step
 * below FP32 resolution reproduces the gamma = 0 value exactly.  Each sum is
 * the change from gamma = 0, |r_g|^2 - |r_0|^2 = (r_g - r_0).(r_g + r_0) per
 * element, summed in FP64.  gammas: device FP64, ngam (<= 8) candidates per
 * segment.  cg_ptycho rho term (solver.py:213), per angle-chunk segment:
 *   out[s*ngam+j] = ||h - (psi + g_j d) + lamd/rho||^2 - (g_j = 0 value) */
int pt_k_rho_minf(double* out, const void* h, const void* psi, const void* lamd, const void* d,
                  double rho, const double* rho_dev, const double* gammas, int ngam, long len,
                  int nseg, const double* skip, pt_stream stream);
/* cg_tomo (solver.py:182-183): out[j] = change of ||K*Ru + g_j*(K*Rd) - xi0||^2 */
int pt_k_tomo_minf(double* out, const void* K, const void* Ru, const void* Rd, const void* xi0,
                   const double* gammas, int ngam, long len, const double* skip,
                   pt_stream stream);
/* cg_tomo: out[j] = change of ||J u + g_j*J d - xi1||^2 */
int pt_k_reg_minf(double* out, const void* u, const void* d, const void* xi1,
                  const double* gammas, int ngam, int nz, int ny, int nx, const double* skip,
                  pt_stream stream);
/* (skip of the three: as in pt_ptycho_minf, segments whose line search has
 * finished are not evaluated.) */
/* out = sum conj(a)*(b - c) (complex, re/im) -- take_lagr terms 2 and 4 */
int pt_k_dot_diff(double* out, const void* a, const void* b, const void* c, long len,
                  pt_stream stream);
/* out[0] = sum_i sqrt(sum_k |phi_k(i)|^2), phi: [3, plane] -- take_lagr term 1 */
int pt_k_tv_norm(double* out, const void* phi, long plane, pt_stream stream);
/* z = a*x + b*y + c*w with complex host scalars (y, w may be NULL) */
int pt_k_lincomb3(void* z, double ar, double ai, const void* x, double br, double bi, const void* y,
                  double cr, double ci, const void* w, long len, pt_stream stream);
/* y += a[s]*x per segment, complex device scalars */
int pt_k_axpy_seg(void* y, const double* a_dev, const void* x, long len, int nseg,
                  pt_stream stream);
/* out = |g|^2 * scale (float32), fwd_ptycho_batch intensities (solver.py:115) */
int pt_k_intensity(float* out, const void* g, float scale, long len, pt_stream stream);
/* out[0] = max |angle(x)| (phase-wrap check of solver.py:238-240) */
int pt_k_max_angle(double* out, const void* x, long len, pt_stream stream);
/* ADMM dual update (solver.py:326-327): out = lam + k*(a - b) with k = c,
 * or k = 1/c if inv != 0; a may be NULL (0), giving xi1 = phi - mu/tau of
 * takexi (solver.py:168).  out may alias lam. */
int pt_k_dual(void* out, const void* lam, const void* a, const void* b, double c,
              const double* c_dev, int inv, long len, pt_stream stream);

/* ------------------------------------------------------- device-side decisions
 * The scalar rules of the CG and ADMM loops evaluated on the device (FP64),
 * so that an ADMM iteration enqueues without host round trips. */
/* Dai-Yuan beta (solver.py:195-196, 230-231) from pt_k_dy_reduce's red
 * [nseg][3]: beta[s] = ||g||^2 / conj-dot (re, im); 0 if the denominator is
 * 0 or not finite (after a zero step, where the reference divides 0 by 0). */
int pt_k_dai_yuan(double* beta, const double* red, int nseg, pt_stream stream);
/* Halving line search (solver.py:171-177) per segment as sweeps of ngam
 * candidates (slot 0 is gamma = 0; sweeps may differ in width).  state
 * [nseg][2] = {current step, done}: begin writes cand[s][0] = 0,
 * cand[s][j] = cur*2^-(j-1) (ngam slots per segment) and clears done.  After
 * the functional f = w[0]*f1 + w[1]*f2 (f2 may be NULL; w: 2 device FP64) is
 * evaluated at cand, select accepts per segment the first candidate that is
 * not a strict ascent or is <= 1e-12 (then 0), writing step[s] = {gamma, 0}
 * and state = {gamma, 1}; unfinished segments get the next sweep's ngam_next
 * candidates in cand_next (a second buffer when ngam_next != ngam and
 * nseg > 1); with last != 0 they end at 0. */
int pt_k_ls_begin(double* state, double* cand, int nseg, int ngam, pt_stream stream);
int pt_k_ls_select(double* state, double* cand, double* cand_next, double* step, const double* f1,
                   const double* f2, const double* w, int nseg, int ngam, int ngam_next, int last,
                   pt_stream stream);
/* cg_tomo's whole line search (solver.py:171-183): the halving rule on
 * w[0]*||K*(Ru + g Rd) - xi0||^2 + w[1]*||J(u + g d) - xi1||^2 from state[0]
 * down to 1e-12, as pt_k_ls_begin and sweeps of pt_k_tomo_minf, pt_k_reg_minf
 * and pt_k_ls_select give it; writes step = {gamma, 0}, state = {gamma, 1}.
 * K, Ru, Rd, xi0 have len elements, u and d [nz,ny,nx], xi1 [3,nz,ny,nx]. */
int pt_k_tomo_linesearch(double* state, double* step, const void* K, const void* Ru,
                         const void* Rd, const void* xi0, const void* u, const void* d,
                         const void* xi1, const double* w, long len, int nz, int ny, int nx,
                         pt_stream stream);
/* A CG step of cg_tomo (solver.py:186-191): Ru += step[0] Rd (Rd NULL: as it
 * is), r = scale * conj(K) (K Ru - xi0), and grad += tau * J*(J u - xi1); as
 * pt_k_axpy_seg, pt_k_tomo_resid and pt_k_reg_grad without the sums.  step,
 * scale and tau: device FP64. */
int pt_k_cg_resid(void* r, void* Ru, const void* Rd, const double* step, const void* K,
                  const void* xi0, const double* scale, long len, pt_stream stream);
int pt_k_cg_reg_grad(void* grad, const void* u, const void* xi1, const double* tau, int nz, int ny,
                     int nx, pt_stream stream);
/* The end of an ADMM iteration (solver.py:322-330), in place, with device FP64
 * scalars.  split: e_new = J u, phi = soft threshold of e_new + mu/tau at
 * alpha/tau, mu += tau (e_new - phi); norms = {||phi - e_new||^2,
 * ||e_new - e||^2}; e = e_new.  object: h_new = exp(i c Ru) exp(i pshift)
 * (pshift = {phase, cos, sin} as pt_k_takexi_dev leaves it), lamd += rho
 * (h_new - psi); norms = {||psi - h_new||^2, ||h_new - h||^2}; h = h_new. */
int pt_k_split_update(double* norms, void* phi, void* e, void* mu, const void* u,
                      const double* tau, double alpha, int nz, int ny, int nx, pt_stream stream);
int pt_k_object_update(double* norms, void* h, void* lamd, const void* psi, const void* Ru,
                       double c, const double* pshift, const double* rho, long len,
                       pt_stream stream);
/* Residual balancing (solver.py:267-282): rho_tau = {rho, tau} updated in
 * place from norms = {||psi-h||^2, ||h-h0||^2, ||phi-e||^2, ||e-e0||^2}. */
int pt_k_penalty(double* rho_tau, const double* norms, pt_stream stream);

/* ------------------------------------------------------- warm-start 3D U-Net
 * No counterpart in the reference: a learned initial guess for ADMM.
 * Activations are bf16 channels-last [D][H][W][C] (raw 16-bit storage);
 * conv weights bf16 [Cout][Kp] with k = tap*Cin + ci, tap = 9 dz + 3 dy + dx
 * for offsets (dz-1, dy-1, dx-1), zero-padded to Kp = ceil16(27 Cin);
 * master weights FP32 [Cout][27][Cin].  Convolutions run on the matrix
 * cores (bf16 in, FP32 accumulate); reductions are deterministic. */
/* y = [relu](bias + conv3x3x3(x, w)), zero padding; Cout in {16, 32, 64};
 * bias may be NULL. */
int pt_nn_conv3d(void* y, const void* x, const void* w, const float* bias, int D, int H, int W,
                 int Cin, int Cout, int relu, pt_stream stream);
/* weights of the input gradient: wt[ci][t*Cout + co] = w[co][(26-t)*Cin + ci]
 * (dx = pt_nn_conv3d(dy, wt) with Cin, Cout swapped, no bias). */
int pt_nn_conv3d_wflip(void* wt, const void* w, int Cin, int Cout, pt_stream stream);
/* weight and bias gradients of pt_nn_conv3d for the pre-activation gradient
 * dy: dw [Cout][27][Cin] FP32, dbias [Cout] (may be NULL); part (FP32,
 * part_cap floats) and bpart (256*Cout doubles) are workspaces. */
int pt_nn_conv3d_wgrad(float* dw, float* dbias, float* part, long part_cap, double* bpart,
                       const void* dy, const void* x, int D, int H, int W, int Cin, int Cout,
                       pt_stream stream);
/* dpre = y > 0 ? dy : 0 (bf16, n elements) */
int pt_nn_relu_bwd(void* dpre, const void* dy, const void* y, long n, pt_stream stream);
/* 2x average pooling of [D][H][W][C] and its gradient (dx = dy(parent)/8,
 * plus `add` if not NULL). */
int pt_nn_pool(void* y, const void* x, int D, int H, int W, int C, pt_stream stream);
int pt_nn_pool_bwd(void* dx, const void* dy, const void* add, int D, int H, int W, int C,
                   pt_stream stream);
/* nearest 2x upsampling of [d][h][w][C] into channels [c0, c0+C) of a
 * Ct-channel [2d][2h][2w] tensor, and its gradient (sum of the 8 children). */
int pt_nn_up(void* y, const void* x, int d, int h, int w, int C, int Ct, int c0, pt_stream stream);
int pt_nn_up_bwd(void* dx, const void* dy, int d, int h, int w, int C, int Ct, int c0,
                 pt_stream stream);
/* dst[v][d0 + c] = src[v][s0 + c], c < C (concatenation) */
int pt_nn_chan_copy(void* dst, int Cd, int d0, const void* src, int Cs, int s0, int C, long V,
                    pt_stream stream);
/* residual 1x1x1 head (FP32 out): out[v][k] = inp[v][k] + b[k] + sum_c w[k][c] x[v][c] */
int pt_nn_head(float* out, const void* x, const float* w, const float* b, const float* inp,
               long V, int C, int K, pt_stream stream);
/* head gradient: dx (bf16) and dwb[k][c] (c < C: weights, c = C: bias),
 * part: part_cap doubles of workspace.  Built for C = 16, K = 2. */
int pt_nn_head_bwd(void* dx, float* dwb, double* part, long part_cap, const float* dout,
                   const void* x, const float* w, long V, int C, int K, pt_stream stream);
/* MSE: part[b] = block partial of sum (pred-target)^2 (FP64, nblk blocks);
 * grad = 2 (pred - target)/n if not NULL. */
int pt_nn_mse(double* part, int nblk, float* grad, const float* pred, const float* target,
              long n, pt_stream stream);
/* Adam step t (bias-corrected) on FP32 master weights; wb, if not NULL,
 * receives the bf16 conv copy (master index co*K + k -> co*Kp + k). */
int pt_nn_adam(float* wm, void* wb, const float* g, float* m, float* v, long n, int K, int Kp,
               float lr, float b1, float b2, float eps, int t, pt_stream stream);
/* bf16 conv weights from FP32 masters */
int pt_nn_pack_w(void* wb, const float* wm, int Cout, int Cin, pt_stream stream);
/* FP32 <-> bf16 (round to nearest even) */
int pt_nn_to_bf16(void* y, const float* x, long n, pt_stream stream);
int pt_nn_to_f32(float* y, const void* x, long n, pt_stream stream);
/* c (16x16 FP32, row-major) = a * b for bf16 16x16 row-major a, b: one
 * matrix-core instruction (operand-layout check). */
int pt_nn_mfma_tile(float* c, const void* a, const void* b, pt_stream stream);
/* c (16x16 FP32, row-major) = a * b for bf16 a [16][32] and b [32][16],
 * row-major: one 16x16x32 matrix-core instruction (the operand layout of the
 * convolutions with 16k input channels). */
int pt_nn_mfma32_tile(float* c, const void* a, const void* b, pt_stream stream);

#ifdef __cplusplus
}
#endif
#endif /* PTYCHOTOMO_HIP_H */
