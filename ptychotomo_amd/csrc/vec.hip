// Solver kernels for gfx950: the element-wise and reduction chains of
// src/ptychotomo/solver.py (cg_tomo, cg_ptycho, solve_reg, takexi,
// update_penalty, take_lagr), each as one fused pass.  Reductions accumulate
// in FP64 with a fixed grid and a fixed-order second pass (deterministic).
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"

namespace pt {

static thread_local std::string g_last_error = "no error";
void set_error(const std::string& msg) { g_last_error = msg; }

// ------------------------------------------------------------------ launch profiler
namespace {
struct Profiler {
  std::mutex mu;
  bool on = false;
  std::string tag;
  std::vector<hipEvent_t> ev;  // pairs (start, stop)
  size_t used = 0;
} g_prof;
}  // namespace

ProfScope::ProfScope(const char* tag, hipStream_t stream) : active(false), slot(-1), st(stream) {
  std::lock_guard<std::mutex> lk(g_prof.mu);
  if (!g_prof.on || g_prof.tag != tag) return;
  if (g_prof.used + 2 > g_prof.ev.size()) {
    for (int i = 0; i < 64; ++i) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return;
      g_prof.ev.push_back(e);
    }
  }
  slot = (int)g_prof.used;
  g_prof.used += 2;
  if (hipEventRecord(g_prof.ev[slot], st) != hipSuccess) return;
  active = true;
}

ProfScope::~ProfScope() {
  if (!active) return;
  std::lock_guard<std::mutex> lk(g_prof.mu);
  (void)hipEventRecord(g_prof.ev[slot + 1], st);
}

namespace {

constexpr int RB = 256;          // threads per reduction block
constexpr int RMAXBLK = 8192;    // blocks per segment cap
constexpr int RMAXTOT = 4096;    // blocks per segmented reduction cap (all segments)

// scratch for partial sums, one per stream (grown on demand): reductions
// enqueued on different streams may run concurrently
struct Partial { double* ptr = nullptr; size_t cap = 0; };
struct Partials {
  std::mutex mu;
  std::map<hipStream_t, Partial> per_stream;
} g_part;

int partial_buf(size_t n, double** out, hipStream_t st) {
  std::lock_guard<std::mutex> lk(g_part.mu);
  Partial& p = g_part.per_stream[st];
  if (n > p.cap) {
    // a buffer in use by queued work on this stream must outlive it
    if (p.ptr) PT_HIP(hipStreamSynchronize(st));
    if (p.ptr) PT_HIP(hipFree(p.ptr));
    p.ptr = nullptr;
    PT_HIP(hipMalloc(&p.ptr, n * sizeof(double)));
    p.cap = n;
  }
  *out = p.ptr;
  return PT_OK;
}

template <int NV, typename F>
__global__ __launch_bounds__(RB) void k_seg_reduce(double* __restrict__ partial, long seglen, F f,
                                                   const double* __restrict__ skip) {
  __shared__ double sm[NV * 16];
  const int seg = blockIdx.y;
  // segments whose line search has finished (skip[2*seg+1] != 0) are not evaluated
  if (skip && skip[2 * seg + 1] != 0.0) return;
  const long base = (long)seg * seglen;
  double v[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < seglen;
       i += (long)gridDim.x * blockDim.x)
    f(base + i, v);
  block_sum<NV>(v, sm);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) partial[((long)seg * gridDim.x + blockIdx.x) * NV + k] = v[k];
  }
}

// second pass: one workgroup per (segment, accumulator): thread-strided sums
// in block order, then the fixed-shape workgroup tree (deterministic)
__global__ __launch_bounds__(RB) void k_finish_n(double* __restrict__ out,
                                                 const double* __restrict__ partial, int nblk,
                                                 int nv, int nout,
                                                 const double* __restrict__ skip) {
  __shared__ double sm[16];
  const int seg = blockIdx.x, k = blockIdx.y;
  if (skip && skip[2 * seg + 1] != 0.0) return;
  double s[1] = {0.0};
  for (int b = threadIdx.x; b < nblk; b += blockDim.x) s[0] += partial[((long)seg * nblk + b) * nv + k];
  block_sum<1>(s, sm);
  if (threadIdx.x == 0) out[seg * nout + k] = s[0];
}

template <int NV, typename F>
int seg_reduce(double* out, long len, int nseg, F f, hipStream_t st) {
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "reduction: nseg must divide len");
  const long seglen = len / nseg;
  int nblk = (int)std::min<long>(RMAXBLK, std::max<long>(1, (seglen + RB * 4 - 1) / (RB * 4)));
  nblk = std::max(1, std::min(nblk, std::max(1, (nseg == 1 ? RMAXBLK : RMAXTOT) / nseg)));
  double* part;
  int rc = partial_buf((size_t)nseg * nblk * NV, &part, st);
  if (rc) return rc;
  hipLaunchKernelGGL((k_seg_reduce<NV, F>), dim3(nblk, nseg), dim3(RB), 0, st, part, seglen, f,
                     (const double*)nullptr);
  PT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_finish_n, dim3(nseg, NV), dim3(RB), 0, st, out, part, nblk, NV, NV,
                     (const double*)nullptr);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// as seg_reduce with NV = PT_MAX_CAND accumulators, of which the first
// `nout` are written per segment
template <typename F>
int seg_partials_n(double** part, int* nblk, long len, int nseg, F f, hipStream_t st,
                   const double* skip) {
  constexpr int NV = 8;
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "reduction: nseg must divide len");
  const long seglen = len / nseg;
  *nblk = (int)std::min<long>(RMAXBLK, std::max<long>(1, (seglen + RB * 4 - 1) / (RB * 4)));
  *nblk = std::max(1, std::min(*nblk, std::max(1, (nseg == 1 ? RMAXBLK : RMAXTOT) / nseg)));
  int rc = partial_buf((size_t)nseg * *nblk * NV, part, st);
  if (rc) return rc;
  hipLaunchKernelGGL((k_seg_reduce<NV, F>), dim3(*nblk, nseg), dim3(RB), 0, st, *part, seglen, f,
                     skip);
  PT_LAUNCH_CHECK();
  return PT_OK;
}
template <typename F>
int seg_reduce_n(double* out, long len, int nseg, int nout, F f, hipStream_t st,
                 const double* skip = nullptr) {
  double* part;
  int nblk, rc = seg_partials_n(&part, &nblk, len, nseg, f, st, skip);
  if (rc) return rc;
  hipLaunchKernelGGL(k_finish_n, dim3(nseg, nout), dim3(RB), 0, st, out, part, nblk, 8, nout,
                     skip);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

template <typename F>
__global__ void k_map(long len, F f) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < len;
       i += (long)gridDim.x * blockDim.x)
    f(i);
}

template <typename F>
int map(long len, F f, hipStream_t st) {
  long nb = (len + 255) / 256;
  if (nb > 65536) nb = 65536;
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL((k_map<F>), dim3((unsigned)nb), dim3(256), 0, st, len, f);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// A scalar kernel argument given either by value or by a device address (the
// device-driven solver keeps rho, tau and the takexi phase in device memory).
struct SV {
  double v; const double* p;
  __device__ double get() const { return p ? p[0] : v; }
};

// ------------------------------------------------------------------ functors
struct FDot {
  const float2* x; const float2* y;
  __device__ void operator()(long i, double (&v)[2]) const {
    const float2 a = x[i], b = y[i];
    v[0] += (double)a.x * b.x + (double)a.y * b.y;
    v[1] += (double)a.x * b.y - (double)a.y * b.x;
  }
};
struct FNorm2 {
  const float2* x;
  __device__ void operator()(long i, double (&v)[1]) const {
    const float2 a = x[i];
    v[0] += (double)a.x * a.x + (double)a.y * a.y;
  }
};
struct FNorm2Lin {
  const float2* x; const float2* y; float ar, ai, br, bi;
  __device__ void operator()(long i, double (&v)[1]) const {
    const float2 a = x[i];
    const float2 b = y ? y[i] : make_float2(0.f, 0.f);
    const float re = ar * a.x - ai * a.y + br * b.x - bi * b.y;
    const float im = ar * a.y + ai * a.x + br * b.y + bi * b.x;
    v[0] += (double)re * re + (double)im * im;
  }
};
struct FDyReduce {
  const float2* g; const float2* g0; const float2* d;
  __device__ void operator()(long i, double (&v)[3]) const {
    const float2 a = g[i], b = g0[i], c = d[i];
    const float dx = a.x - b.x, dy = a.y - b.y;
    v[0] += (double)a.x * a.x + (double)a.y * a.y;
    v[1] += (double)c.x * dx + (double)c.y * dy;
    v[2] += (double)c.x * dy - (double)c.y * dx;
  }
};

struct FLincomb {
  float2* z; const double* a; const float2* x; const double* b; const float2* y; long seglen;
  __device__ void operator()(long i) const {
    const long s = i / seglen;
    const float2 av = make_float2((float)a[2 * s], (float)a[2 * s + 1]);
    float2 r = cmul(av, x[i]);
    if (y) {
      const float2 bv = make_float2((float)b[2 * s], (float)b[2 * s + 1]);
      r = cadd(r, cmul(bv, y[i]));
    }
    z[i] = r;
  }
};
struct FDyUpdate {
  float2* d; const float2* g; const double* beta; int first; long seglen;
  __device__ void operator()(long i) const {
    const float2 gv = g[i];
    if (first) {
      d[i] = make_float2(-gv.x, -gv.y);
    } else {
      const long s = i / seglen;
      const float2 bv = make_float2((float)beta[2 * s], (float)beta[2 * s + 1]);
      const float2 t = cmul(bv, d[i]);
      d[i] = make_float2(t.x - gv.x, t.y - gv.y);
    }
  }
};

// fwd_reg: res[0] x-diff, res[1] y-diff, res[2] z-diff, times 2/sqrt(3)
struct FRegFwd {
  float2* out; const float2* u; int nz, ny, nx;
  __device__ void operator()(long i) const {
    const long plane = (long)nz * ny * nx;
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    const float c = 1.15470053837925152902f;  // 2/sqrt(3)
    const float2 v = u[i];
    float2 a = make_float2(0.f, 0.f), b = a, e = a;
    if (x < nx - 1) { float2 w = u[i + 1]; a = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    if (y < ny - 1) { float2 w = u[i + nx]; b = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    if (z < nz - 1) { float2 w = u[i + (long)ny * nx]; e = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    out[i] = a;
    out[plane + i] = b;
    out[2 * plane + i] = e;
  }
};
// adj_reg (solver.py:137-146)
struct FRegAdj {
  float2* out; const float2* g; int nz, ny, nx;
  __device__ void operator()(long i) const {
    const long plane = (long)nz * ny * nx;
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    const float c = -1.15470053837925152902f;
    const float2* g0 = g;
    const float2* g1 = g + plane;
    const float2* g2 = g + 2 * plane;
    float2 s = g0[i];
    if (x > 0) s = csub(s, g0[i - 1]);
    float2 t = g1[i];
    if (y > 0) t = csub(t, g1[i - nx]);
    s = cadd(s, t);
    float2 w = g2[i];
    if (z > 0) w = csub(w, g2[i - (long)ny * nx]);
    s = cadd(s, w);
    out[i] = make_float2(s.x * c, s.y * c);
  }
};
// solve_reg (solver.py:257-264)
struct FRegSolve {
  float2* out; const float2* u; const float2* mu; SV tau; double alpha; int nz, ny, nx;
  __device__ void operator()(long i) const {
    const double t = tau.get();
    const float itau = (float)(1.0 / t), thr = (float)(alpha / t);
    const long plane = (long)nz * ny * nx;
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    const float c = 1.15470053837925152902f;
    const float2 v = u[i];
    float2 g[3] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
    if (x < nx - 1) { float2 w = u[i + 1]; g[0] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    if (y < ny - 1) { float2 w = u[i + nx]; g[1] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    if (z < nz - 1) { float2 w = u[i + (long)ny * nx]; g[2] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float2 m = mu[k * plane + i];
      g[k] = make_float2(g[k].x + m.x * itau, g[k].y + m.y * itau);
      ss += g[k].x * g[k].x + g[k].y * g[k].y;
    }
    const float za = sqrtf(ss);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      float2 o;
      if (za <= thr) o = make_float2(0.f, 0.f);
      else {
        const float q = thr / za;
        o = make_float2(g[k].x - q * g[k].x, g[k].y - q * g[k].y);
      }
      out[k * plane + i] = o;
    }
  }
};

struct FExpTomo {
  float2* out; const float2* psi; float c; float2 ph; const double* ph_dev;
  __device__ void operator()(long i) const {
    // device phase: ph_dev = {pshift, cos(pshift), sin(pshift)}
    const float2 phv = ph_dev ? make_float2((float)ph_dev[1], (float)ph_dev[2]) : ph;
    // exp(i*c*psi) = exp(-c*Im psi) * (cos(c*Re psi) + i sin(c*Re psi))
    const float2 p = psi[i];
    const float a = expf(-c * p.y);
    float sn, cs;
    sincosf(c * p.x, &sn, &cs);
    out[i] = cmul(make_float2(a * cs, a * sn), phv);
  }
};

// The end of an ADMM iteration as two passes over its states (solver.py:257-264,
// 322-330).  Element-wise the formulas of FRegSolve, FRegFwd, FExpTomo, FDual and
// FNorm2Lin; v[0], v[1] = the primal and dual residual sums of the penalty update.
// Bound: memory.  As separate kernels with copies of the new h and e they moved 13
// and 12 arrays' worth where these read and write 6 and 5 (e, phi, mu: 403 MB each
// at 256^3; h, lamd, psi, Ru: 201 MB at 384 angles): 1.5 -> 0.64 ms there.
struct FSplitTail {  // phi, mu and e from u: v = |phi - e|^2, |e - e_old|^2
  float2* phi; float2* e; float2* mu; const float2* u; SV tau; double alpha; int nz, ny, nx;
  __device__ void operator()(long i, double (&v)[2]) const {
    const double t = tau.get();
    const float itau = (float)(1.0 / t), thr = (float)(alpha / t), tf = (float)t;
    const long plane = (long)nz * ny * nx;
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    const float c = 1.15470053837925152902f;  // 2/sqrt(3)
    const float2 w = u[i];
    float2 g[3] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f), make_float2(0.f, 0.f)}, q[3], m[3];
    if (x < nx - 1) { float2 s = u[i + 1]; g[0] = make_float2((s.x - w.x) * c, (s.y - w.y) * c); }
    if (y < ny - 1) { float2 s = u[i + nx]; g[1] = make_float2((s.x - w.x) * c, (s.y - w.y) * c); }
    if (z < nz - 1) { float2 s = u[i + (long)ny * nx]; g[2] = make_float2((s.x - w.x) * c, (s.y - w.y) * c); }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      m[k] = mu[k * plane + i];
      q[k] = make_float2(g[k].x + m[k].x * itau, g[k].y + m[k].y * itau);
      ss += q[k].x * q[k].x + q[k].y * q[k].y;
    }
    const float za = sqrtf(ss), sh = thr / za;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const long j = k * plane + i;
      const float2 p = za <= thr ? make_float2(0.f, 0.f)
                                 : make_float2(q[k].x - sh * q[k].x, q[k].y - sh * q[k].y);
      const float2 d = csub(g[k], p), o = csub(g[k], e[j]);
      phi[j] = p;
      mu[j] = make_float2(m[k].x + tf * d.x, m[k].y + tf * d.y);
      e[j] = g[k];
      v[0] += (double)d.x * d.x + (double)d.y * d.y;
      v[1] += (double)o.x * o.x + (double)o.y * o.y;
    }
  }
};
struct FObjectTail {  // h and lamd from Ru: v = |psi - h|^2, |h - h_old|^2
  float2* h; float2* lamd; const float2* psi; const float2* Ru; float c; const double* ph; SV rho;
  __device__ void operator()(long i, double (&v)[2]) const {
    const float2 p = Ru[i];
    const float a = expf(-c * p.y), rf = (float)rho.get();
    float sn, cs;
    sincosf(c * p.x, &sn, &cs);
    const float2 hn = cmul(make_float2(a * cs, a * sn), make_float2((float)ph[1], (float)ph[2]));
    const float2 l = lamd[i], d = csub(hn, psi[i]), o = csub(hn, h[i]);
    lamd[i] = make_float2(l.x + rf * d.x, l.y + rf * d.y);
    h[i] = hn;
    v[0] += (double)d.x * d.x + (double)d.y * d.y;
    v[1] += (double)o.x * o.x + (double)o.y * o.y;
  }
};

__device__ __forceinline__ float2 mlog_c(float2 x) {
  const float m = hypotf(x.x, x.y);
  if (m < 1e-32f) return make_float2(logf(1e-32f), 0.f);
  return make_float2(logf(m), atan2f(x.y, x.x));
}

struct FMlog {
  float2* out; const float2* x;
  __device__ void operator()(long i) const { out[i] = mlog_c(x[i]); }
};

struct FTakexiStats {
  const float2* psi; const float2* lamd; SV rho; int nz, n, r;
  __device__ void operator()(long i, double (&v)[3]) const {
    const float irho = (float)(1.0 / rho.get());
    const int x = (int)(i % n);
    const float2 p = psi[i];
    if (x >= r && x < 2 * r) v[0] += (double)atan2f(p.y, p.x);
    if (x >= n - 2 * r && x < n - r) v[1] += (double)atan2f(p.y, p.x);
    const float2 l = lamd[i];
    const float tx = p.x - l.x * irho, ty = p.y - l.y * irho;
    const double m = (double)hypotf(tx, ty);
    if (m > v[2]) v[2] = m;
  }
};

struct FTakexi {
  float2* xi0; float2* K; const float2* psi; const float2* lamd; SV rhov; float2 ephv;
  float kfacv; float xfac; const double* prm;
  __device__ void operator()(long i) const {
    // device parameters: prm = {pshift, cos(pshift), sin(pshift), kfac}
    const float rho = (float)rhov.get();
    const float2 eph = prm ? make_float2((float)prm[1], -(float)prm[2]) : ephv;
    const float kfac = prm ? (float)prm[3] : kfacv;
    const float2 p = psi[i], l = lamd[i];
    float2 t = make_float2(p.x - l.x / rho, p.y - l.y / rho);
    t = cmul(t, eph);
    const float2 lt = mlog_c(t);
    // K = i*kfac*t
    const float2 k = make_float2(-kfac * t.y, kfac * t.x);
    K[i] = k;
    // xi0 = K * (-i * logt) * xfac
    const float2 m = make_float2(lt.y * xfac, -lt.x * xfac);
    xi0[i] = cmul(k, m);
  }
};


// cg_tomo residual: r = conj(K)*(K*Ru - xi0); v[0] += |K*Ru - xi0|^2
struct FTomoResid {
  float2* r; const float2* K; const float2* Ru; const float2* xi0; SV scale;
  __device__ void operator()(long i, double (&v)[1]) const {
    const float2 k = K[i];
    const float2 e = csub(cmul(k, Ru[i]), xi0[i]);
    r[i] = cscale(cmul(cconj(k), e), (float)scale.get());
    v[0] += (double)e.x * e.x + (double)e.y * e.y;
  }
};

__device__ __forceinline__ void grad3(const float2* __restrict__ u, long i, int x, int y, int z,
                                      int nz, int ny, int nx, float2 (&g)[3]) {
  const float c = 1.15470053837925152902f;
  const float2 v = u[i];
  g[0] = g[1] = g[2] = make_float2(0.f, 0.f);
  if (x < nx - 1) { float2 w = u[i + 1]; g[0] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
  if (y < ny - 1) { float2 w = u[i + nx]; g[1] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
  if (z < nz - 1) { float2 w = u[i + (long)ny * nx]; g[2] = make_float2((w.x - v.x) * c, (w.y - v.y) * c); }
}

// grad = rho_part + tau * J*(J u - xi1);  v[0] += |J u - xi1|^2
struct FRegGrad {
  float2* grad; const float2* u; const float2* xi1; SV tau; int nz, ny, nx;
  __device__ void operator()(long i, double (&v)[1]) const {
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    at(i, x, y, z, v);
  }
  __device__ __forceinline__ void at(long i, int x, int y, int z, double (&v)[1]) const {
    const long plane = (long)nz * ny * nx;
    float2 g[3];
    grad3(u, i, x, y, z, nz, ny, nx, g);
    float2 w[3];
    for (int k = 0; k < 3; ++k) {
      w[k] = csub(g[k], xi1[k * plane + i]);
      v[0] += (double)w[k].x * w[k].x + (double)w[k].y * w[k].y;
    }
    // adj_reg of w (solver.py:137-146): sum_k w_k(i) - w_k(i - e_k) (if i_k > 0)
    float2 s = make_float2(w[0].x + w[1].x + w[2].x, w[0].y + w[1].y + w[2].y);
    float2 gn[3];
    if (x > 0) {
      grad3(u, i - 1, x - 1, y, z, nz, ny, nx, gn);
      s = csub(s, csub(gn[0], xi1[i - 1]));
    }
    if (y > 0) {
      grad3(u, i - nx, x, y - 1, z, nz, ny, nx, gn);
      s = csub(s, csub(gn[1], xi1[plane + i - nx]));
    }
    if (z > 0) {
      const long off = (long)ny * nx;
      grad3(u, i - off, x, y, z - 1, nz, ny, nx, gn);
      s = csub(s, csub(gn[2], xi1[2 * plane + i - off]));
    }
    const float c = -1.15470053837925152902f * (float)tau.get();
    const float2 gv = grad[i];
    grad[i] = make_float2(gv.x + c * s.x, gv.y + c * s.y);
  }
};
// A CG step's two element-wise passes of cg_tomo (FTomoResid and FRegGrad without
// their sums, which the solver does not use: no second pass).  The residual pass
// first makes the previous step's Ru += step Rd, whose result only it reads: K, xi0,
// Rd, Ru read, Ru, r written once (5.8 TB/s at 256^3, 384 angles, the copy's rate):
// 271 -> 208 us there, 18 -> 8 us at 64^3, 96 angles, against pt_k_axpy_seg and
// pt_k_tomo_resid.  The gradient pass runs over planes (blockIdx.y = z), one 32-bit
// division per voxel instead of 64-bit ones: 237 -> 216 us at 256^3, 11.4 -> 7.5 us at
// 64^3, bound by the neighbours' rows read again from the caches.
struct FCgResid {
  float2* r; float2* Ru; const float2* Rd; const double* step; const float2* K; const float2* xi0;
  SV scale;
  __device__ void operator()(long i) const {
    float2 ru = Ru[i];
    if (Rd) {
      ru = cadd(ru, cmul(make_float2((float)step[0], (float)step[1]), Rd[i]));
      Ru[i] = ru;
    }
    const float2 k = K[i];
    const float2 e = csub(cmul(k, ru), xi0[i]);
    r[i] = cscale(cmul(cconj(k), e), (float)scale.get());
  }
};
__global__ __launch_bounds__(256) void k_cg_reg_grad(FRegGrad f) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= f.ny * f.nx) return;
  const int y = (int)((unsigned)p / (unsigned)f.nx), x = p - y * f.nx;
  for (int z = blockIdx.y; z < f.nz; z += gridDim.y) {
    double v[1];
    f.at((long)z * f.ny * f.nx + p, x, y, z, v);
  }
}

// Line-search candidates, formed as the reference forms them: the stepped
// quantity x + gamma*dx element-wise in FP32 (a step below FP32 resolution
// gives exactly the gamma = 0 value).  What is summed (in FP64) is the change
// of the squared residual from gamma = 0, per element, |r_g|^2 - |r_0|^2 =
// (r_g - r_0).(r_g + r_0): the halving rule decides on f(gamma) - f(0), and
// this form does not lose it to the rounding of two large sums.
#define PT_MAX_CAND 8
// cg_ptycho rho term (solver.py:213): change of |h - (psi + g*d) + lamd/rho|^2
struct FRhoMinf {
  const float2* h; const float2* psi; const float2* lamd; const float2* d; SV rhov;
  const double* gam; int ngam; long seglen;
  __device__ void operator()(long i, double (&v)[PT_MAX_CAND]) const {
    const long s = i / seglen;
    const float rho = (float)rhov.get();
    const float2 a = h[i], p = psi[i], l = lamd[i], dd = d[i];
    const float lx = l.x / rho, ly = l.y / rho;
    const float r0x = a.x - p.x + lx, r0y = a.y - p.y + ly;
#pragma unroll
    for (int j = 0; j < PT_MAX_CAND; ++j) {
      if (j < ngam) {
        const float g = (float)gam[s * ngam + j];
        const float tx = p.x + g * dd.x, ty = p.y + g * dd.y;
        const float rx = a.x - tx + lx, ry = a.y - ty + ly;
        v[j] += (double)((rx - r0x) * (rx + r0x) + (ry - r0y) * (ry + r0y));
      }
    }
  }
};
// cg_tomo data term (solver.py:182-183): change of |K*Ru + g*(K*Rd) - xi0|^2
struct FTomoMinf {
  const float2* K; const float2* Ru; const float2* Rd; const float2* xi0; const double* gam;
  int ngam;
  __device__ void operator()(long i, double (&v)[PT_MAX_CAND]) const {
    const float2 k = K[i];
    const float2 a = cmul(k, Ru[i]), b = cmul(k, Rd[i]), x = xi0[i];
    const float r0x = a.x - x.x, r0y = a.y - x.y;
#pragma unroll
    for (int j = 0; j < PT_MAX_CAND; ++j) {
      if (j < ngam) {
        const float g = (float)gam[j];
        const float rx = (a.x + g * b.x) - x.x, ry = (a.y + g * b.y) - x.y;
        v[j] += (double)((rx - r0x) * (rx + r0x) + (ry - r0y) * (ry + r0y));
      }
    }
  }
};
// cg_tomo regulariser term: change of |J u + g*J d - xi1|^2 over the 3 components
struct FRegMinf {
  const float2* u; const float2* d; const float2* xi1; const double* gam; int ngam;
  int nz, ny, nx;
  __device__ void operator()(long i, double (&v)[PT_MAX_CAND]) const {
    const long plane = (long)nz * ny * nx;
    const int x = (int)(i % nx);
    const long r = i / nx;
    const int y = (int)(r % ny);
    const int z = (int)(r / ny);
    float2 gu[3], gd[3], xi[3];
    grad3(u, i, x, y, z, nz, ny, nx, gu);
    grad3(d, i, x, y, z, nz, ny, nx, gd);
    for (int k = 0; k < 3; ++k) xi[k] = xi1[k * plane + i];
#pragma unroll
    for (int j = 0; j < PT_MAX_CAND; ++j) {
      if (j < ngam) {
        const float g = (float)gam[j];
        double dacc = 0.0;
        for (int k = 0; k < 3; ++k) {
          const float rx = (gu[k].x + g * gd[k].x) - xi[k].x;
          const float ry = (gu[k].y + g * gd[k].y) - xi[k].y;
          const float r0x = gu[k].x - xi[k].x, r0y = gu[k].y - xi[k].y;
          dacc += (double)((rx - r0x) * (rx + r0x) + (ry - r0y) * (ry + r0y));
        }
        v[j] += dacc;
      }
    }
  }
};
// sum conj(a)*(b - c)
struct FDotDiff {
  const float2* a; const float2* b; const float2* c;
  __device__ void operator()(long i, double (&v)[2]) const {
    const float2 x = a[i], y = csub(b[i], c[i]);
    v[0] += (double)x.x * y.x + (double)x.y * y.y;
    v[1] += (double)x.x * y.y - (double)x.y * y.x;
  }
};
// sum_i sqrt(sum_k |phi_k(i)|^2)
struct FTvNorm {
  const float2* phi; long plane;
  __device__ void operator()(long i, double (&v)[1]) const {
    float s = 0.f;
    for (int k = 0; k < 3; ++k) {
      const float2 a = phi[k * plane + i];
      s += a.x * a.x + a.y * a.y;
    }
    v[0] += (double)sqrtf(s);
  }
};
struct FLincomb3 {
  float2* z; float2 a; const float2* x; float2 b; const float2* y; float2 c; const float2* w;
  __device__ void operator()(long i) const {
    float2 r = cmul(a, x[i]);
    if (y) r = cadd(r, cmul(b, y[i]));
    if (w) r = cadd(r, cmul(c, w[i]));
    z[i] = r;
  }
};
// ADMM dual update (solver.py:326-327): out = lam + k*(a - b), k = c or 1/c;
// a may be null (0), which gives xi1 = phi - mu/tau (solver.py:168)
struct FDual {
  float2* out; const float2* lam; const float2* a; const float2* b; SV c; int inv;
  __device__ void operator()(long i) const {
    const double cv = c.get();
    const float cf = (float)(inv ? 1.0 / cv : cv);
    const float2 av = a ? a[i] : make_float2(0.f, 0.f);
    const float2 l = lam[i], t = csub(av, b[i]);
    out[i] = make_float2(l.x + cf * t.x, l.y + cf * t.y);
  }
};
struct FAxpySeg {
  float2* y; const double* a; const float2* x; long seglen;
  __device__ void operator()(long i) const {
    const long s = i / seglen;
    const float2 av = make_float2((float)a[2 * s], (float)a[2 * s + 1]);
    y[i] = cadd(y[i], cmul(av, x[i]));
  }
};
}  // namespace
}  // namespace pt

using namespace pt;

extern "C" const char* pt_last_error(void) { return g_last_error.c_str(); }
extern "C" int pt_abi_version(void) { return 1; }

#ifndef PT_HEADER_DIGEST
#define PT_HEADER_DIGEST "unknown"
#endif
extern "C" const char* pt_header_digest(void) { return PT_HEADER_DIGEST; }

extern "C" int pt_k_dot(double* out, const void* x, const void* y, long len, int nseg,
                        pt_stream stream) {
  PT_REQUIRE(out && x && y, PT_ERR_ARG, "pt_k_dot: null argument");
  return seg_reduce<2>(out, len, nseg, FDot{(const float2*)x, (const float2*)y}, (hipStream_t)stream);
}
extern "C" int pt_k_norm2(double* out, const void* x, long len, int nseg, pt_stream stream) {
  PT_REQUIRE(out && x, PT_ERR_ARG, "pt_k_norm2: null argument");
  return seg_reduce<1>(out, len, nseg, FNorm2{(const float2*)x}, (hipStream_t)stream);
}
extern "C" int pt_k_norm2_lin(double* out, const void* x, const void* y, double ar, double ai,
                              double br, double bi, long len, int nseg, pt_stream stream) {
  PT_REQUIRE(out && x, PT_ERR_ARG, "pt_k_norm2_lin: null argument");
  return seg_reduce<1>(out, len, nseg,
                       FNorm2Lin{(const float2*)x, (const float2*)y, (float)ar, (float)ai,
                                 (float)br, (float)bi},
                       (hipStream_t)stream);
}
extern "C" int pt_k_lincomb(void* z, const double* a_dev, const void* x, const double* b_dev,
                            const void* y, long len, int nseg, pt_stream stream) {
  PT_REQUIRE(z && a_dev && x && (!y || b_dev), PT_ERR_ARG, "pt_k_lincomb: null argument");
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "pt_k_lincomb: nseg must divide len");
  return map(len, FLincomb{(float2*)z, a_dev, (const float2*)x, b_dev, (const float2*)y, len / nseg},
             (hipStream_t)stream);
}
extern "C" int pt_k_dy_update(void* d, const void* grad, const double* beta_dev, int first,
                              long len, int nseg, pt_stream stream) {
  PT_REQUIRE(d && grad && (first || beta_dev), PT_ERR_ARG, "pt_k_dy_update: null argument");
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "pt_k_dy_update: nseg must divide len");
  return map(len, FDyUpdate{(float2*)d, (const float2*)grad, beta_dev, first, len / nseg},
             (hipStream_t)stream);
}
extern "C" int pt_k_dy_reduce(double* out, const void* grad, const void* grad0, const void* d,
                              long len, int nseg, pt_stream stream) {
  PT_REQUIRE(out && grad && grad0 && d, PT_ERR_ARG, "pt_k_dy_reduce: null argument");
  return seg_reduce<3>(out, len, nseg,
                       FDyReduce{(const float2*)grad, (const float2*)grad0, (const float2*)d},
                       (hipStream_t)stream);
}

extern "C" int pt_k_reg_fwd(void* out, const void* u, int nz, int ny, int nx, pt_stream stream) {
  PT_REQUIRE(out && u, PT_ERR_ARG, "pt_k_reg_fwd: null argument");
  return map((long)nz * ny * nx, FRegFwd{(float2*)out, (const float2*)u, nz, ny, nx},
             (hipStream_t)stream);
}
extern "C" int pt_k_reg_adj(void* out, const void* g, int nz, int ny, int nx, pt_stream stream) {
  PT_REQUIRE(out && g, PT_ERR_ARG, "pt_k_reg_adj: null argument");
  return map((long)nz * ny * nx, FRegAdj{(float2*)out, (const float2*)g, nz, ny, nx},
             (hipStream_t)stream);
}
extern "C" int pt_k_reg_solve(void* out, const void* u, const void* mu, double tau,
                              const double* tau_dev, double alpha, int nz, int ny, int nx,
                              pt_stream stream) {
  PT_REQUIRE(out && u && mu, PT_ERR_ARG, "pt_k_reg_solve: null argument");
  PT_REQUIRE(tau_dev || tau > 0, PT_ERR_ARG, "pt_k_reg_solve: tau must be positive");
  return map((long)nz * ny * nx,
             FRegSolve{(float2*)out, (const float2*)u, (const float2*)mu, SV{tau, tau_dev}, alpha,
                       nz, ny, nx},
             (hipStream_t)stream);
}
extern "C" int pt_k_exptomo(void* out, const void* psi, double c, double phase,
                            const double* phase_dev, long len, pt_stream stream) {
  PT_REQUIRE(out && psi, PT_ERR_ARG, "pt_k_exptomo: null argument");
  const float2 ph = make_float2((float)std::cos(phase), (float)std::sin(phase));
  return map(len, FExpTomo{(float2*)out, (const float2*)psi, (float)c, ph, phase_dev},
             (hipStream_t)stream);
}
extern "C" int pt_k_mlog(void* out, const void* x, long len, pt_stream stream) {
  PT_REQUIRE(out && x, PT_ERR_ARG, "pt_k_mlog: null argument");
  return map(len, FMlog{(float2*)out, (const float2*)x}, (hipStream_t)stream);
}

// max-reduction variant: the stats functor keeps a running max in v[2]; the
// block sum would add maxima, so use a dedicated kernel.
namespace pt {
namespace {
__global__ __launch_bounds__(RB) void k_takexi_stats(double* __restrict__ partial,
                                                     FTakexiStats f, long len) {
  __shared__ double sm[3 * 16];
  double v[3] = {0.0, 0.0, 0.0};
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < len;
       i += (long)gridDim.x * blockDim.x)
    f(i, v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  v[0] = wave_sum(v[0]);
  v[1] = wave_sum(v[1]);
  for (int off = 32; off > 0; off >>= 1) v[2] = fmax(v[2], __shfl_xor(v[2], off, 64));
  if (lane == 0) { sm[wid] = v[0]; sm[16 + wid] = v[1]; sm[32 + wid] = v[2]; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = 0, b = 0, m = 0;
    for (int w = 0; w < nw; ++w) { a += sm[w]; b += sm[16 + w]; m = fmax(m, sm[32 + w]); }
    partial[blockIdx.x * 3 + 0] = a;
    partial[blockIdx.x * 3 + 1] = b;
    partial[blockIdx.x * 3 + 2] = m;
  }
}
__global__ void k_takexi_finish(double* out, const double* partial, int nblk) {
  if (threadIdx.x) return;
  double a = 0, b = 0, m = 0;
  for (int i = 0; i < nblk; ++i) {
    a += partial[i * 3];
    b += partial[i * 3 + 1];
    m = fmax(m, partial[i * 3 + 2]);
  }
  out[0] = a; out[1] = b; out[2] = m;
}
}  // namespace
}  // namespace pt

extern "C" int pt_k_takexi_stats(double* out, const void* psi, const void* lamd, double rho,
                                 const double* rho_dev, int ntheta, int nz, int n, int r,
                                 pt_stream stream) {
  PT_REQUIRE(out && psi && lamd, PT_ERR_ARG, "pt_k_takexi_stats: null argument");
  PT_REQUIRE((rho_dev || rho > 0) && r >= 0 && 2 * r <= n, PT_ERR_ARG,
             "pt_k_takexi_stats: bad rho or r");
  hipStream_t st = (hipStream_t)stream;
  const long len = (long)ntheta * nz * n;
  const int nblk = (int)std::min<long>(1024, std::max<long>(1, (len + RB * 8 - 1) / (RB * 8)));
  double* part;
  int rc = partial_buf((size_t)nblk * 3, &part, st);
  if (rc) return rc;
  FTakexiStats f{(const float2*)psi, (const float2*)lamd, SV{rho, rho_dev}, nz, n, r};
  hipLaunchKernelGGL(k_takexi_stats, dim3(nblk), dim3(RB), 0, st, part, f, len);
  PT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_takexi_finish, dim3(1), dim3(64), 0, st, out, part, nblk);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

extern "C" int pt_k_takexi(void* xi0, void* K, const void* psi, const void* lamd, double rho,
                           double pshift, double kc, double kscale, double c1, double coeftomo,
                           long len, pt_stream stream) {
  PT_REQUIRE(xi0 && K && psi && lamd, PT_ERR_ARG, "pt_k_takexi: null argument");
  PT_REQUIRE(rho > 0, PT_ERR_ARG, "pt_k_takexi: rho must be positive");
  const float2 eph = make_float2((float)std::cos(-pshift), (float)std::sin(-pshift));
  // K = i*kc*t*kscale ; xi0 = K*(-i*logt/c1)*coeftomo
  return map(len,
             FTakexi{(float2*)xi0, (float2*)K, (const float2*)psi, (const float2*)lamd,
                     SV{rho, nullptr}, eph, (float)(kc * kscale), (float)(coeftomo / c1),
                     nullptr},
             (hipStream_t)stream);
}

namespace pt {
namespace {
// takexi scalars from the statistics pass, as solver.py:149-168 forms them:
// pshift = float32 mean of the two column-band angle means, kscale =
// 1/(kc*max|t|) (0 if max|t| = 0).  prm = {pshift, cos, sin, kc*kscale}.
__global__ void k_takexi_params(double* prm, const double* stats, double cnt, double kc) {
  if (threadIdx.x) return;
  const float m1 = (float)(stats[0] / cnt), m2 = (float)(stats[1] / cnt);
  const double pshift = (double)((m1 + m2) / 2.0f);
  const double tmax = stats[2];
  const double kscale = tmax > 0 ? 1.0 / (kc * tmax) : 0.0;
  prm[0] = pshift;
  prm[1] = cos(pshift);
  prm[2] = sin(pshift);
  prm[3] = kc * kscale;
}
}  // namespace
}  // namespace pt

extern "C" int pt_k_takexi_dev(void* xi0, void* K, double* prm, const void* psi,
                               const void* lamd, const double* rho_dev, const double* stats,
                               double cnt, double kc, double c1, double coeftomo, long len,
                               pt_stream stream) {
  PT_REQUIRE(xi0 && K && prm && psi && lamd && rho_dev && stats, PT_ERR_ARG,
             "pt_k_takexi_dev: null argument");
  PT_REQUIRE(cnt > 0, PT_ERR_ARG, "pt_k_takexi_dev: cnt must be positive");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_takexi_params, dim3(1), dim3(64), 0, st, prm, stats, cnt, kc);
  PT_LAUNCH_CHECK();
  return map(len,
             FTakexi{(float2*)xi0, (float2*)K, (const float2*)psi, (const float2*)lamd,
                     SV{0.0, rho_dev}, make_float2(0.f, 0.f), 0.f, (float)(coeftomo / c1), prm},
             st);
}

namespace pt {
namespace {
__global__ __launch_bounds__(RB) void k_max_angle(double* __restrict__ partial,
                                                  const float2* __restrict__ x, long len) {
  __shared__ double sm[16];
  double m = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < len;
       i += (long)gridDim.x * blockDim.x) {
    const float2 a = x[i];
    m = fmax(m, (double)fabsf(atan2f(a.y, a.x)));
  }
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 0) sm[wid] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = 0;
    for (int w = 0; w < nw; ++w) r = fmax(r, sm[w]);
    partial[blockIdx.x] = r;
  }
}
__global__ void k_max_finish(double* out, const double* partial, int nblk) {
  if (threadIdx.x) return;
  double r = 0;
  for (int i = 0; i < nblk; ++i) r = fmax(r, partial[i]);
  out[0] = r;
}
}  // namespace
}  // namespace pt

extern "C" int pt_k_tomo_resid(void* r, double* out, const void* K, const void* Ru,
                               const void* xi0, double scale, const double* scale_dev, long len,
                               pt_stream stream) {
  PT_REQUIRE(r && out && K && Ru && xi0, PT_ERR_ARG, "pt_k_tomo_resid: null argument");
  return seg_reduce<1>(out, len, 1,
                       FTomoResid{(float2*)r, (const float2*)K, (const float2*)Ru,
                                  (const float2*)xi0, SV{scale, scale_dev}},
                       (hipStream_t)stream);
}
extern "C" int pt_k_reg_grad(void* grad, double* out, const void* u, const void* xi1, double tau,
                             const double* tau_dev, int nz, int ny, int nx, pt_stream stream) {
  PT_REQUIRE(grad && out && u && xi1, PT_ERR_ARG, "pt_k_reg_grad: null argument");
  return seg_reduce<1>(out, (long)nz * ny * nx, 1,
                       FRegGrad{(float2*)grad, (const float2*)u, (const float2*)xi1,
                                SV{tau, tau_dev}, nz, ny, nx},
                       (hipStream_t)stream);
}
extern "C" int pt_k_dual(void* out, const void* lam, const void* a, const void* b, double c,
                         const double* c_dev, int inv, long len, pt_stream stream) {
  PT_REQUIRE(out && lam && b, PT_ERR_ARG, "pt_k_dual: null argument");
  return map(len,
             FDual{(float2*)out, (const float2*)lam, (const float2*)a, (const float2*)b,
                   SV{c, c_dev}, inv},
             (hipStream_t)stream);
}
extern "C" int pt_k_dot_diff(double* out, const void* a, const void* b, const void* c, long len,
                             pt_stream stream) {
  PT_REQUIRE(out && a && b && c, PT_ERR_ARG, "pt_k_dot_diff: null argument");
  return seg_reduce<2>(out, len, 1, FDotDiff{(const float2*)a, (const float2*)b, (const float2*)c},
                       (hipStream_t)stream);
}
extern "C" int pt_k_tv_norm(double* out, const void* phi, long plane, pt_stream stream) {
  PT_REQUIRE(out && phi, PT_ERR_ARG, "pt_k_tv_norm: null argument");
  return seg_reduce<1>(out, plane, 1, FTvNorm{(const float2*)phi, plane}, (hipStream_t)stream);
}
extern "C" int pt_k_lincomb3(void* z, double ar, double ai, const void* x, double br, double bi,
                             const void* y, double cr, double ci, const void* w, long len,
                             pt_stream stream) {
  PT_REQUIRE(z && x, PT_ERR_ARG, "pt_k_lincomb3: null argument");
  return map(len,
             FLincomb3{(float2*)z, make_float2((float)ar, (float)ai), (const float2*)x,
                       make_float2((float)br, (float)bi), (const float2*)y,
                       make_float2((float)cr, (float)ci), (const float2*)w},
             (hipStream_t)stream);
}
extern "C" int pt_k_axpy_seg(void* y, const double* a_dev, const void* x, long len, int nseg,
                             pt_stream stream) {
  PT_REQUIRE(y && a_dev && x, PT_ERR_ARG, "pt_k_axpy_seg: null argument");
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "pt_k_axpy_seg: nseg must divide len");
  return map(len, FAxpySeg{(float2*)y, a_dev, (const float2*)x, len / nseg}, (hipStream_t)stream);
}
extern "C" int pt_k_max_angle(double* out, const void* x, long len, pt_stream stream) {
  PT_REQUIRE(out && x, PT_ERR_ARG, "pt_k_max_angle: null argument");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = (int)std::min<long>(1024, std::max<long>(1, (len + RB * 8 - 1) / (RB * 8)));
  double* part;
  int rc = partial_buf((size_t)nblk, &part, st);
  if (rc) return rc;
  hipLaunchKernelGGL(k_max_angle, dim3(nblk), dim3(RB), 0, st, part, (const float2*)x, len);
  PT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_max_finish, dim3(1), dim3(64), 0, st, out, part, nblk);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

namespace pt {
namespace {
struct FIntensity {
  float* out; const float2* g; float s;
  __device__ void operator()(long i) const {
    const float2 a = g[i];
    const float m = hypotf(a.x, a.y);
    out[i] = m * m * s;
  }
};
}  // namespace
}  // namespace pt
extern "C" int pt_k_intensity(float* out, const void* g, float scale, long len, pt_stream stream) {
  PT_REQUIRE(out && g, PT_ERR_ARG, "pt_k_intensity: null argument");
  return map(len, FIntensity{out, (const float2*)g, scale}, (hipStream_t)stream);
}

extern "C" int pt_prof_start(const char* tag) {
  PT_REQUIRE(tag, PT_ERR_ARG, "pt_prof_start: null tag");
  std::lock_guard<std::mutex> lk(g_prof.mu);
  g_prof.on = true;
  g_prof.tag = tag;
  g_prof.used = 0;
  return PT_OK;
}

extern "C" int pt_prof_stop(double* total_ms, long* launches) {
  PT_REQUIRE(total_ms && launches, PT_ERR_ARG, "pt_prof_stop: null argument");
  std::lock_guard<std::mutex> lk(g_prof.mu);
  g_prof.on = false;
  double tot = 0.0;
  long cnt = 0;
  for (size_t i = 0; i + 1 < g_prof.used; i += 2) {
    PT_HIP(hipEventSynchronize(g_prof.ev[i + 1]));
    float ms = 0.f;
    PT_HIP(hipEventElapsedTime(&ms, g_prof.ev[i], g_prof.ev[i + 1]));
    tot += ms;
    ++cnt;
  }
  g_prof.used = 0;
  *total_ms = tot;
  *launches = cnt;
  return PT_OK;
}

extern "C" int pt_k_rho_minf(double* out, const void* h, const void* psi, const void* lamd,
                             const void* d, double rho, const double* rho_dev,
                             const double* gammas, int ngam, long len, int nseg,
                             const double* skip, pt_stream stream) {
  PT_REQUIRE(out && h && psi && lamd && d && gammas, PT_ERR_ARG, "pt_k_rho_minf: null argument");
  PT_REQUIRE(rho_dev || rho > 0, PT_ERR_ARG, "pt_k_rho_minf: rho must be positive");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_CAND, PT_ERR_ARG, "pt_k_rho_minf: 1 <= ngam <= 8");
  PT_REQUIRE(nseg > 0 && len % nseg == 0, PT_ERR_SIZE, "pt_k_rho_minf: nseg must divide len");
  return seg_reduce_n(out, len, nseg, ngam,
                      FRhoMinf{(const float2*)h, (const float2*)psi, (const float2*)lamd,
                               (const float2*)d, SV{rho, rho_dev}, gammas, ngam, len / nseg},
                      (hipStream_t)stream, skip);
}
int pt::rho_minf_partials(double** part, int* nblk, const void* h, const void* psi,
                          const void* lamd, const void* d, double rho, const double* rho_dev,
                          const double* gammas, int ngam, long len, int nseg, const double* skip,
                          hipStream_t st) {
  return seg_partials_n(part, nblk, len, nseg,
                        FRhoMinf{(const float2*)h, (const float2*)psi, (const float2*)lamd,
                                 (const float2*)d, SV{rho, rho_dev}, gammas, ngam, len / nseg},
                        st, skip);
}
extern "C" int pt_k_tomo_minf(double* out, const void* K, const void* Ru, const void* Rd,
                              const void* xi0, const double* gammas, int ngam, long len,
                              const double* skip, pt_stream stream) {
  PT_REQUIRE(out && K && Ru && Rd && xi0 && gammas, PT_ERR_ARG, "pt_k_tomo_minf: null argument");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_CAND, PT_ERR_ARG, "pt_k_tomo_minf: 1 <= ngam <= 8");
  return seg_reduce_n(out, len, 1, ngam,
                      FTomoMinf{(const float2*)K, (const float2*)Ru, (const float2*)Rd,
                                (const float2*)xi0, gammas, ngam},
                      (hipStream_t)stream, skip);
}
extern "C" int pt_k_reg_minf(double* out, const void* u, const void* d, const void* xi1,
                             const double* gammas, int ngam, int nz, int ny, int nx,
                             const double* skip, pt_stream stream) {
  PT_REQUIRE(out && u && d && xi1 && gammas, PT_ERR_ARG, "pt_k_reg_minf: null argument");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_CAND, PT_ERR_ARG, "pt_k_reg_minf: 1 <= ngam <= 8");
  return seg_reduce_n(out, (long)nz * ny * nx, 1, ngam,
                      FRegMinf{(const float2*)u, (const float2*)d, (const float2*)xi1, gammas,
                               ngam, nz, ny, nx},
                      (hipStream_t)stream, skip);
}

// ------------------------------------------------------------------ device-side decisions
// The scalar steps of the CG and ADMM loops, computed on the device so that an
// ADMM iteration enqueues without host round trips (and can be captured as a
// graph).  FP64, no contraction: the host restatement of each rule gives the
// same bits.
namespace pt {
namespace {
#pragma clang fp contract(off)
// Dai-Yuan (solver.py:195-196, 230-231): beta = ||g||^2 / sum(conj(d)(g - g0)),
// red[s] = {||g||^2, Re den, Im den}; beta = 0 when den is 0 or not finite
// (a zero step leaves g == g0, where the reference divides 0 by 0).
__global__ void k_dai_yuan(double* __restrict__ beta, const double* __restrict__ red, int nseg) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const double gn = red[3 * s], dr = red[3 * s + 1], di = red[3 * s + 2];
  const double den2 = dr * dr + di * di;
  double br = 0.0, bi = 0.0;
  if (den2 > 0.0 && isfinite(den2)) {
    br = gn * dr / den2;
    bi = -(gn * di) / den2;
    if (!isfinite(br) || !isfinite(bi)) br = bi = 0.0;
  }
  beta[2 * s] = br;
  beta[2 * s + 1] = bi;
}

// Halving line search (solver.py:171-177) for nseg independent segments, as
// sweeps of ngam candidates: cand[s][0] = 0, cand[s][j] = cur * 2^-(j-1).
// state[s] = {cur, done}; step[s] = {gamma, 0} once done.
__global__ void k_ls_begin(double* __restrict__ state, double* __restrict__ cand, int nseg,
                           int ngam) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const double cur = state[2 * s];
  state[2 * s + 1] = 0.0;
  cand[s * ngam] = 0.0;
  for (int j = 1; j < ngam; ++j) cand[s * ngam + j] = cur * ldexp(1.0, -(j - 1));
}

// f[s][j] = w[0]*f1[s][j] + w[1]*f2[s][j] (f2 may be null).  A segment accepts
// the first candidate that is not a strict ascent or is <= 1e-12 (then 0);
// otherwise its next sweep (ngam_next slots, written to cand_next) continues
// from half the last candidate.  With `last`, an unfinished segment ends at 0
// as the halving rule would.
__global__ void k_ls_select(double* __restrict__ state, const double* cand, double* cand_next,
                            double* __restrict__ step, const double* __restrict__ f1,
                            const double* __restrict__ f2, const double* __restrict__ w, int nseg,
                            int ngam, int ngam_next, int last) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  if (state[2 * s + 1] != 0.0) return;
  const double w0 = w[0], w1 = f2 ? w[1] : 0.0;
  const double* a = f1 + s * ngam;
  const double* b = f2 ? f2 + s * ngam : nullptr;
  ls_decide(state + 2 * s, step + 2 * s, cand + s * ngam, cand_next + s * ngam_next, ngam,
            ngam_next, last, [&](int j) { return w0 * a[j] + (b ? w1 * b[j] : 0.0); });
}

// cg_tomo's whole halving search (solver.py:171-183) in groups of kTLFirst
// halvings.  A sweep takes one or several groups: an evaluation (both functional
// terms, blockIdx.y) and a one-workgroup kernel that sums the partials in a fixed
// order and applies the halving rule; a sweep after the accepted step exits at once.
// 4 to 12 launches instead of the 31 of six sweeps of two reductions, their finishing
// passes and a selection.
// Which groups share a sweep: a sweep that exits costs 3.4 us, a group that need not
// have been evaluated 10 us at 96 x 64^2, 48 us at 192 x 128^2, 400 us at 384 x 256^2
// (bound: K, Ru, Rd, xi0, u, d, xi1 read once per group).  Up to kTLSmall blocks of
// 1024 elements the first group has a sweep and all others share one; up to kTLLarge
// the first two have one each (a third for the third group costs cg_tomo at 128^3 0.7 %,
// and steps below 2^-13 are rare); beyond that every group has.  Step accepted in the
// first / second / third group: 23 / 75 / 77 us (96 x 64^2), 68 / 120 / 310 us
// (192 x 128^2), 430 / 850 / 1260 us (384 x 256^2); with all groups after the first in
// one sweep the latter took 70 / 295 / 304 and 418 / 2420 / 2430 us.  Half the blocks
// up to kTLLarge: the selection then reads half the partials (at 192 x 128^2 75 -> 70
// us; at 384 x 256^2 435 -> 454).
constexpr int kTLFirst = 7;    // halvings per group (slot 0 is gamma = 0)
constexpr int kTLGroups = 6;   // groups in all: 42 halvings, 2 -> below 1e-12
constexpr int kTLBlocks = 2048;  // per term: 8 per CU
constexpr long kTLSmall = 1024, kTLLarge = 8192;
__global__ __launch_bounds__(RB) void k_tomo_ls_eval(double* __restrict__ partial, FTomoMinf ft,
                                                     long lenp, FRegMinf fr, long lenu,
                                                     const double* __restrict__ state, int g0,
                                                     int g1) {
  __shared__ double sm[PT_MAX_CAND * 16];
  __shared__ double cand[PT_MAX_CAND];
  if (g0 && state[1] != 0.0) return;
  const int term = blockIdx.y;
  for (int g = g0; g < g1; ++g) {
    __syncthreads();
    if (threadIdx.x <= kTLFirst)
      cand[threadIdx.x] =
          threadIdx.x ? state[0] * ldexp(1.0, -(g * kTLFirst + (int)threadIdx.x - 1)) : 0.0;
    __syncthreads();
    ft.gam = fr.gam = cand;
    double v[PT_MAX_CAND];
#pragma unroll
    for (int k = 0; k < PT_MAX_CAND; ++k) v[k] = 0.0;
    const long i0 = (long)blockIdx.x * blockDim.x + threadIdx.x, st = (long)gridDim.x * blockDim.x;
    if (term == 0)
      for (long i = i0; i < lenp; i += st) ft(i, v);
    else
      for (long i = i0; i < lenu; i += st) fr(i, v);
    block_sum<PT_MAX_CAND>(v, sm);
    if (threadIdx.x == 0)
#pragma unroll
      for (int k = 0; k < PT_MAX_CAND; ++k)
        partial[(((long)g * 2 + term) * gridDim.x + blockIdx.x) * PT_MAX_CAND + k] = v[k];
  }
}

// wave w sums the partials of (term w/8, candidate w%8); thread 0 decides
__global__ __launch_bounds__(1024) void k_tomo_ls_select(double* __restrict__ state,
                                                         double* __restrict__ step,
                                                         const double* __restrict__ partial,
                                                         const double* __restrict__ w, int nblk,
                                                         int g0, int g1) {
  __shared__ double f[2][PT_MAX_CAND];
  __shared__ int done;
  if (g0 && state[1] != 0.0) return;
  const double cur = state[0];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, term = wid >> 3, j = wid & 7;
  if (threadIdx.x == 0) {
    done = 0;
    if (!g0) state[1] = 0.0;
  }
  for (int g = g0; g < g1; ++g) {
    const double* src = partial + ((long)g * 2 + term) * nblk * PT_MAX_CAND + j;
    double s = 0.0;
#pragma unroll 4
    for (int b = lane; b < nblk; b += 64) s += src[(long)b * PT_MAX_CAND];
    s = wave_sum(s);
    __syncthreads();
    if (lane == 0) f[term][j] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int k = 1; k <= kTLFirst && !done; ++k) {
        const double gam = cur * ldexp(1.0, -(g * kTLFirst + k - 1));
        const double fz = w[0] * f[0][0] + w[1] * f[1][0];
        const double fk = w[0] * f[0][k] + w[1] * f[1][k];
        if (fz - fk < 0.0 && gam > 1e-12) continue;
        step[0] = gam <= 1e-12 ? 0.0 : gam;
        done = 1;
      }
      if (!done && g == kTLGroups - 1) {
        step[0] = 0.0;
        done = 1;
      }
    }
    __syncthreads();
    if (done) break;
  }
  if (threadIdx.x == 0 && done) {
    state[0] = step[0];
    state[1] = 1.0;
    step[1] = 0.0;
  }
}

// Residual balancing (solver.py:267-282).  norms = {||psi - h||^2,
// ||h - h0||^2, ||phi - e||^2, ||e - e0||^2}; the reference's
// ||rho (h - h0)||^2 is rho^2 ||h - h0||^2 (rho is a power of 2, so the
// scaling is exact).  rt = {rho, tau}, updated in place.
__global__ void k_penalty(double* __restrict__ rt, const double* __restrict__ norms) {
  if (threadIdx.x) return;
  double rho = rt[0], tau = rt[1];
  const double r = norms[0], s = rho * rho * norms[1];
  const double r2 = norms[2], s2 = tau * tau * norms[3];
  if (r > 10.0 * s) rho *= 2.0;
  else if (s > 10.0 * r) rho *= 0.5;
  if (r2 > 10.0 * s2) tau *= 2.0;
  else if (s2 > 10.0 * r2) tau *= 0.5;
  rt[0] = rho;
  rt[1] = tau;
}
#pragma clang fp contract(on)
}  // namespace
}  // namespace pt

extern "C" int pt_k_dai_yuan(double* beta, const double* red, int nseg, pt_stream stream) {
  PT_REQUIRE(beta && red && nseg > 0, PT_ERR_ARG, "pt_k_dai_yuan: bad argument");
  hipLaunchKernelGGL(k_dai_yuan, dim3((nseg + 63) / 64), dim3(64), 0, (hipStream_t)stream, beta,
                     red, nseg);
  PT_LAUNCH_CHECK();
  return PT_OK;
}
extern "C" int pt_k_tomo_linesearch(double* state, double* step, const void* K, const void* Ru,
                                    const void* Rd, const void* xi0, const void* u, const void* d,
                                    const void* xi1, const double* w, long len, int nz, int ny,
                                    int nx, pt_stream stream) {
  PT_REQUIRE(state && step && K && Ru && Rd && xi0 && u && d && xi1 && w, PT_ERR_ARG,
             "pt_k_tomo_linesearch: null argument");
  PT_REQUIRE(len > 0 && nz > 0 && ny > 0 && nx > 0, PT_ERR_SIZE,
             "pt_k_tomo_linesearch: sizes must be positive");
  hipStream_t st = (hipStream_t)stream;
  const long lenu = (long)nz * ny * nx;
  const long nb = (std::max(len, lenu) + RB * 4 - 1) / (RB * 4);
  const int nblk = (int)std::min<long>(nb <= kTLLarge ? kTLBlocks / 2 : kTLBlocks, nb);
  double* part;
  const int rc = partial_buf((size_t)kTLGroups * 2 * nblk * PT_MAX_CAND, &part, st);
  if (rc) return rc;
  const FTomoMinf ft{(const float2*)K, (const float2*)Ru, (const float2*)Rd, (const float2*)xi0,
                     nullptr, kTLFirst + 1};
  const FRegMinf fr{(const float2*)u, (const float2*)d, (const float2*)xi1, nullptr, kTLFirst + 1,
                    nz, ny, nx};
  // the first group of each sweep
  static constexpr int few[] = {0, 1, kTLGroups}, some[] = {0, 1, 2, kTLGroups},
                       all[] = {0, 1, 2, 3, 4, 5, kTLGroups};
  const int* at = nb <= kTLSmall ? few : nb <= kTLLarge ? some : all;
  for (; at[0] < kTLGroups; ++at) {
    const int g0 = at[0], g1 = at[1];
    hipLaunchKernelGGL(k_tomo_ls_eval, dim3(nblk, 2), dim3(RB), 0, st, part, ft, len, fr, lenu,
                       state, g0, g1);
    PT_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_tomo_ls_select, dim3(1), dim3(1024), 0, st, state, step, part, w, nblk,
                       g0, g1);
    PT_LAUNCH_CHECK();
  }
  return PT_OK;
}
extern "C" int pt_k_cg_resid(void* r, void* Ru, const void* Rd, const double* step, const void* K,
                             const void* xi0, const double* scale, long len, pt_stream stream) {
  PT_REQUIRE(r && Ru && K && xi0 && scale && (!Rd || step), PT_ERR_ARG,
             "pt_k_cg_resid: null argument");
  return map(len, FCgResid{(float2*)r, (float2*)Ru, (const float2*)Rd, step, (const float2*)K,
                           (const float2*)xi0, SV{0.0, scale}}, (hipStream_t)stream);
}
extern "C" int pt_k_cg_reg_grad(void* grad, const void* u, const void* xi1, const double* tau,
                                int nz, int ny, int nx, pt_stream stream) {
  PT_REQUIRE(grad && u && xi1 && tau, PT_ERR_ARG, "pt_k_cg_reg_grad: null argument");
  PT_REQUIRE(nz > 0 && ny > 0 && nx > 0 && (long)ny * nx <= 0x7fffff00L, PT_ERR_SIZE,
             "pt_k_cg_reg_grad: bad size");
  hipLaunchKernelGGL(k_cg_reg_grad, dim3((unsigned)((ny * nx + 255) / 256), std::min(nz, 65535)),
                     dim3(256), 0, (hipStream_t)stream,
                     FRegGrad{(float2*)grad, (const float2*)u, (const float2*)xi1, SV{0.0, tau},
                              nz, ny, nx});
  PT_LAUNCH_CHECK();
  return PT_OK;
}
extern "C" int pt_k_split_update(double* norms, void* phi, void* e, void* mu, const void* u,
                                 const double* tau, double alpha, int nz, int ny, int nx,
                                 pt_stream stream) {
  PT_REQUIRE(norms && phi && e && mu && u && tau, PT_ERR_ARG, "pt_k_split_update: null argument");
  PT_REQUIRE(nz > 0 && ny > 0 && nx > 0, PT_ERR_SIZE, "pt_k_split_update: sizes must be positive");
  return seg_reduce<2>(norms, (long)nz * ny * nx, 1,
                       FSplitTail{(float2*)phi, (float2*)e, (float2*)mu, (const float2*)u,
                                  SV{0.0, tau}, alpha, nz, ny, nx},
                       (hipStream_t)stream);
}
extern "C" int pt_k_object_update(double* norms, void* h, void* lamd, const void* psi,
                                  const void* Ru, double c, const double* pshift,
                                  const double* rho, long len, pt_stream stream) {
  PT_REQUIRE(norms && h && lamd && psi && Ru && pshift && rho, PT_ERR_ARG,
             "pt_k_object_update: null argument");
  PT_REQUIRE(len > 0, PT_ERR_SIZE, "pt_k_object_update: len must be positive");
  return seg_reduce<2>(norms, len, 1,
                       FObjectTail{(float2*)h, (float2*)lamd, (const float2*)psi,
                                   (const float2*)Ru, (float)c, pshift, SV{0.0, rho}},
                       (hipStream_t)stream);
}
extern "C" int pt_k_ls_begin(double* state, double* cand, int nseg, int ngam, pt_stream stream) {
  PT_REQUIRE(state && cand && nseg > 0, PT_ERR_ARG, "pt_k_ls_begin: bad argument");
  PT_REQUIRE(ngam >= 2 && ngam <= PT_MAX_CAND, PT_ERR_ARG, "pt_k_ls_begin: 2 <= ngam <= 8");
  hipLaunchKernelGGL(k_ls_begin, dim3((nseg + 63) / 64), dim3(64), 0, (hipStream_t)stream, state,
                     cand, nseg, ngam);
  PT_LAUNCH_CHECK();
  return PT_OK;
}
extern "C" int pt_k_ls_select(double* state, double* cand, double* cand_next, double* step,
                              const double* f1, const double* f2, const double* w, int nseg,
                              int ngam, int ngam_next, int last, pt_stream stream) {
  PT_REQUIRE(state && cand && cand_next && step && f1 && w && nseg > 0, PT_ERR_ARG,
             "pt_k_ls_select: bad argument");
  PT_REQUIRE(ngam >= 2 && ngam <= PT_MAX_CAND && ngam_next >= 2 && ngam_next <= PT_MAX_CAND,
             PT_ERR_ARG, "pt_k_ls_select: 2 <= ngam, ngam_next <= 8");
  PT_REQUIRE(cand_next != cand || ngam_next == ngam || nseg == 1, PT_ERR_ARG,
             "pt_k_ls_select: a sweep of another width needs its own candidate buffer");
  hipLaunchKernelGGL(k_ls_select, dim3((nseg + 63) / 64), dim3(64), 0, (hipStream_t)stream, state,
                     cand, cand_next, step, f1, f2, w, nseg, ngam, ngam_next, last);
  PT_LAUNCH_CHECK();
  return PT_OK;
}
extern "C" int pt_k_penalty(double* rho_tau, const double* norms, pt_stream stream) {
  PT_REQUIRE(rho_tau && norms, PT_ERR_ARG, "pt_k_penalty: null argument");
  hipLaunchKernelGGL(k_penalty, dim3(1), dim3(64), 0, (hipStream_t)stream, rho_tau, norms);
  PT_LAUNCH_CHECK();
  return PT_OK;
}
