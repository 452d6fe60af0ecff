// Ptychography operator for gfx950: probe x object patch, D x D far field.
//
// Replaces class ptychofft (src/cuda/ptychofft.cu, src/include/kernels.cuh
// kernels mul/mula/takeshifts/shifts/shiftsa) and fuses the CuPy chains of
// cg_ptycho (src/ptychotomo/solver.py:206-242).
//
// Layout: one 64-lane wavefront works on G = 64/D patches at a time; lane
// (slot = lane/D, r = lane%D) holds one frame row (D complex values in
// VGPRs).  The 2D FFT is an in-register row FFT, an LDS transpose (row stride
// D+1 to avoid bank conflicts), and an in-register column FFT, after which
// lane c holds far-field column c.  The frame is transposed relative to the
// object (kernels.cuh:251-263): frame row ix + ox holds object column
// stx + ix, frame column iy + oy holds object row sty + iy.
//
// Overlap-add (adjoint and fused gradient) is deterministic and free of
// global atomics: patches are binned by rounded position into B x B tiles
// per angle at set_scan_probe time; one wavefront owns a tile and
// accumulates its patches, in bin order, into an LDS tile extended by P-1
// (LDS adds issued by a single wavefront); the extended tiles go to scratch
// and a fold kernel sums the (at most 4) tiles covering each pixel in a fixed
// order.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"

struct pt_ptycho {
  int pt, nz, n, S, D, P;
  int ox, oy;
  float c;  // 1/sqrt(detx*dety)
  int B, EB, ntx, nty;
  long ntiles, nslots;
  float2* prb = nullptr;        // [P*P]
  int2* pos = nullptr;          // [pt*S] rounded (x, y); x < 0 -> skipped
  float2* shift = nullptr;      // [pt*S] shiftx*shifty
  int* tile_start = nullptr;    // [ntiles+1]
  int* tile_patch = nullptr;    // [nvalid]
  int* tile_slot = nullptr;     // [ntiles]
  float2* scratch = nullptr;    // [nslots*EB*EB]
  size_t scratch_cap = 0;       // elements
  double* partial = nullptr;    // minf partial sums
  size_t partial_cap = 0;       // doubles
  bool ready = false;
};

namespace pt {
namespace {

constexpr int WAVE = 64;

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }

// ------------------------------------------------------------------ transforms
// Forward 2D transform of the frame rows held by the wave (v = row r of the
// lane's patch) -> lane c holds far-field column c (in v).
template <int D>
__device__ __forceinline__ void frame_fwd(float2 (&v)[D], float2* T, int slot, int r) {
  reg_fft<D, -1>(v);
  float2* Ts = T + slot * D * (D + 1);
#pragma unroll
  for (int k = 0; k < D; ++k) Ts[r * (D + 1) + k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < D; ++k) v[k] = Ts[k * (D + 1) + r];
  __syncthreads();
  reg_fft<D, -1>(v);
}

// Wave-local LDS exchange: orders the wave's LDS accesses (LDS operations of
// one wavefront complete in issue order) without a workgroup barrier.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// D x D transposes through a per-wave float buffer (real, then imaginary
// parts: half the LDS of a float2 buffer).  Row stride D+1; the slot stride
// D(D+1) puts the two slots of a half-wave on disjoint banks.
template <int D, bool ROW_TO_COL>
__device__ __forceinline__ void transpose_w(float2 (&v)[D], float* Ts, int r) {
  float tmp[D];
#pragma unroll
  for (int k = 0; k < D; ++k) Ts[ROW_TO_COL ? r * (D + 1) + k : k * (D + 1) + r] = v[k].x;
  wave_sync();
#pragma unroll
  for (int k = 0; k < D; ++k) tmp[k] = Ts[ROW_TO_COL ? k * (D + 1) + r : r * (D + 1) + k];
  wave_sync();
#pragma unroll
  for (int k = 0; k < D; ++k) Ts[ROW_TO_COL ? r * (D + 1) + k : k * (D + 1) + r] = v[k].y;
  wave_sync();
#pragma unroll
  for (int k = 0; k < D; ++k) {
    v[k] = make_float2(tmp[k], Ts[ROW_TO_COL ? k * (D + 1) + r : r * (D + 1) + k]);
  }
  wave_sync();
}
// Forward / inverse frame transforms with the wave-local float buffer (T: this wave's
// G*D*(D+1) floats)
template <int D>
__device__ __forceinline__ void frame_fwd_w(float2 (&v)[D], float* T, int slot, int r) {
  reg_fft<D, -1>(v);
  transpose_w<D, true>(v, T + slot * D * (D + 1), r);
  reg_fft<D, -1>(v);
}
template <int D>
__device__ __forceinline__ void frame_inv_w(float2 (&v)[D], float* T, int slot, int r) {
  reg_fft<D, 1>(v);
  transpose_w<D, false>(v, T + slot * D * (D + 1), r);
  reg_fft<D, 1>(v);
}

// D x D transpose of FP64 complex frame elements through the same per-wave
// float buffer, one 32-bit word of every element at a time (low and high
// words of the real part, then of the imaginary part)
template <int D, bool ROW_TO_COL>
__device__ __forceinline__ void transpose_w64(double2 (&w)[D], float* Ts, int r) {
  int* Ti = reinterpret_cast<int*>(Ts);
  static_for<0, 4>([&](auto pc) {
    constexpr int part = decltype(pc)::value;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const double x = part < 2 ? w[k].x : w[k].y;
      Ti[ROW_TO_COL ? r * (D + 1) + k : k * (D + 1) + r] =
          (part & 1) ? __double2hiint(x) : __double2loint(x);
    }
    wave_sync();
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const int b = Ti[ROW_TO_COL ? k * (D + 1) + r : r * (D + 1) + k];
      double& x = part < 2 ? w[k].x : w[k].y;
      x = (part & 1) ? __hiloint2double(b, __double2loint(x))
                     : __hiloint2double(__double2hiint(x), b);
    }
    wave_sync();
  });
}

// Forward frame transform in FP64 arithmetic (double twiddles), FP32 in and
// out, the result scaled by s before it is rounded.  The fused gradient's
// Poisson residual d a/|a|^2 takes the far field's small entries relative to
// their own size; an FP32 transform's absolute rounding (~1e-7 of the
// frame's largest entry) is a large relative error there, and over tens of
// CG steps the FP32 trajectory then parts from the exact one by 3e-4 .. 1e-2
// depending on the FFT's operation order.  The FP64 transform leaves only
// the final rounding (relative, per entry).
// mid() is called between the two passes (loads in flight during the second).
template <int D, class F>
__device__ __forceinline__ void frame_fwd64_w(float2 (&v)[D], float* T, int slot, int r, float s,
                                              F mid) {
  double2 w[D];
#pragma unroll
  for (int k = 0; k < D; ++k) w[k] = make_double2((double)v[k].x, (double)v[k].y);
  reg_fft<D, -1>(w);
  transpose_w64<D, true>(w, T + slot * D * (D + 1), r);
  __builtin_amdgcn_sched_barrier(0);
  mid();
  reg_fft<D, -1>(w);
  const double sd = (double)s;
#pragma unroll
  for (int k = 0; k < D; ++k) v[k] = make_float2((float)(w[k].x * sd), (float)(w[k].y * sd));
}

// Load frame row r of patch p: c * prb[ix][iy] * psi[t][sty+iy][stx+ix]
template <int D>
__device__ __forceinline__ void load_frame_row(float2 (&v)[D], const float2* __restrict__ f,
                                               const float2* __restrict__ prb, int2 ps, int t, int r,
                                               int nz, int n, int P, int ox, int oy, float cs,
                                               bool active) {
  const int ix = r - ox;
  const bool rowin = active && ps.x >= 0 && ix >= 0 && ix < P;
  const float2* fp = f + ((long)t * nz + ps.y - oy) * n + ps.x + ix;
  const float2* pp = prb + (long)ix * P - oy;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int iy = k - oy;
    float2 val = make_float2(0.f, 0.f);
    if (rowin && iy >= 0 && iy < P) {
      float2 a = fp[(long)k * n];
      float2 b = pp[k];
      val = cscale(cmul(b, a), cs);
    }
    v[k] = val;
  }
}

// Split form of load_frame_row for kernels that issue all of a patch group's
// global loads before the first transpose: the probe column of the lane's
// frame row (c * prb[ix][iy], 0 outside the probe) once per wave, the raw
// object values per patch (0 outside), and their product.
template <int D>
__device__ __forceinline__ void probe_row(float2 (&pr)[D], const float2* __restrict__ prb, int r,
                                          int P, int ox, int oy, float cs) {
  const int ix = r - ox;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int iy = k - oy;
    pr[k] = (ix >= 0 && ix < P && iy >= 0 && iy < P) ? cscale(prb[(long)ix * P + iy], cs)
                                                     : make_float2(0.f, 0.f);
  }
}
template <int D>
__device__ __forceinline__ void load_rows(float2 (&v)[D], const float2* __restrict__ f, int2 ps,
                                          int t, int r, int nz, int n, int P, int ox, int oy,
                                          bool active) {
  const int ix = r - ox;
  const bool rowin = active && ps.x >= 0 && ix >= 0 && ix < P;
  const float2* fp = f + ((long)t * nz + ps.y - oy) * n + ps.x + ix;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int iy = k - oy;
    v[k] = (rowin && iy >= 0 && iy < P) ? fp[(long)k * n] : make_float2(0.f, 0.f);
  }
}
// v = cs * prb[ix][iy] * v, probe values read from memory (cached)
template <int D>
__device__ __forceinline__ void apply_probe(float2 (&v)[D], const float2* __restrict__ prb, int r,
                                            int P, int ox, int oy, float cs) {
  const int ix = r - ox;
  const float2* pp = prb + (long)ix * P - oy;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int iy = k - oy;
    v[k] = (ix >= 0 && ix < P && iy >= 0 && iy < P) ? cscale(cmul(pp[k], v[k]), cs)
                                                    : make_float2(0.f, 0.f);
  }
}

// ------------------------------------------------------------------ fwd
// INT = false: the far field with the per-patch phase (g); INT = true: only its
// intensity scaled by isc (out), in which the phase has no part: 165 MB written
// at 128^2, 192 angles, 16 x 16 frames instead of the far field written, read
// and squared in a second pass (98 + 96 -> 59 us).  Bound: the far field or
// intensity written.
template <int D, bool INT>
__global__ __launch_bounds__(WAVE) void k_fwd(float2* __restrict__ g, float* __restrict__ out,
                                              const float2* __restrict__ f,
                                              const float2* __restrict__ prb,
                                              const int2* __restrict__ pos,
                                              const float2* __restrict__ shift, int pt, int nz, int n,
                                              int S, int P, int ox, int oy, float cs, float isc) {
  constexpr int G = WAVE / D;
  // frames up to 16 x 16 transpose one float component at a time (half the LDS
  // of a complex buffer; at 64 x 64 that form spills registers) and read the
  // probe from LDS (a lane's probe column is P-strided in memory: one cache
  // line per lane and row)
  __shared__ float Tf[D <= 16 ? G * D * (D + 1) : 1];
  __shared__ float2 Tc[D <= 16 ? 1 : G * D * (D + 1)];
  __shared__ float2 prl[D <= 16 ? D * D : 1];
  const int lane = lane_id(), slot = lane / D, r = lane % D;
  if constexpr (D <= 16) {
    for (int i = lane; i < P * P; i += WAVE) prl[i] = prb[i];
    __syncthreads();
  }
  const long npatch = (long)pt * S;
  for (long grp = blockIdx.x; grp * G < npatch; grp += gridDim.x) {
    const long p = grp * G + slot;
    const bool active = p < npatch;
    int2 ps = active ? pos[p] : make_int2(-1, -1);
    const int t = active ? (int)(p / S) : 0;
    float2 v[D];
    if constexpr (D <= 16) {
      load_rows<D>(v, f, ps, t, r, nz, n, P, ox, oy, active);
      apply_probe<D>(v, prl, r, P, ox, oy, cs);
      frame_fwd_w<D>(v, Tf, slot, r);
    } else {
      load_frame_row<D>(v, f, prb, ps, t, r, nz, n, P, ox, oy, cs, active);
      frame_fwd<D>(v, Tc, slot, r);
    }
    if (!active) continue;
    if constexpr (INT) {
      float* op = out + p * D * D + r;
#pragma unroll
      for (int k = 0; k < D; ++k) op[k * D] = (v[k].x * v[k].x + v[k].y * v[k].y) * isc;
    } else {
      const float2 sh = shift[p];
      float2* gp = g + p * D * D + r;
#pragma unroll
      for (int k = 0; k < D; ++k) gp[k * D] = cmul(v[k], sh);
    }
  }
}

// ------------------------------------------------------------------ minf
// log|a| with |a| clamped below at 1e-32 as mlog does (solver.py:48-52), for
// s = |a|^2: the hardware log of s where s is a normal float; below that a
// is scaled by 2^64 first (|a| >= 1e-32 then gives a normal square).
__device__ __forceinline__ float log_abs(float2 a, float s) {
  if (s >= 1.17549435e-38f) return 0.5f * __logf(s);
  const float x = a.x * 1.8446744e19f, y = a.y * 1.8446744e19f;
  return fmaxf(0.5f * __logf(x * x + y * y) - 44.3614196f, -73.6827235f);
}

// log(1 + x) for x >= -15/16, without branches: u = fl(1 + x) and its rounding
// error c = x - (u - 1) (exact: u - 1 and the difference are representable
// for u in [1/16, 2^24]; for x in [-15/16, -1/2] u is exact and c = 0), then
// log1p(x) = ln u + log1p(c/u).  For u < 2,
// c/u is replaced by c (the difference, at most 2^-25 |x| / u, is under
// 9e-8 of |log1p(x)|); for u >= 2 the term is below 2^-24 against ln u >=
// 0.69 and is dropped.  ln u from the hardware base-2 log times ln 2; for
// |x| below FP32 resolution u = 1 and the result is c = x exactly.  Checked
// on gfx950 against the FP64 log1p over |x| in [1e-30, 1e3] (with c/u: at
// most 1.6e-7 relative).
__device__ __forceinline__ float log1p_step(float x) {
  const float u = 1.f + x;
  const float c = x - (u - 1.f);
  return __builtin_fmaf(__builtin_amdgcn_logf(u), 0.693147181f, u < 2.f ? c : 0.f);
}

// Candidate-independent part of the line-search sums, once per patch:
//   poisson:  w = 1/|a|^2 (hardware reciprocal) where |a|^2 >= 4 FLT_MIN,
//             else NaN (every candidate of that element then takes the
//             separate-log path of delta_part)
//   gaussian: w = |a|
template <int D, int MODEL>
__device__ __forceinline__ void delta_prep(const float2 (&a)[D], float (&w)[D]) {
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const float s0 = a[k].x * a[k].x + a[k].y * a[k].y;
    if constexpr (MODEL == PT_MODEL_POISSON)
      w[k] = s0 >= 4.70197740e-38f ? __builtin_amdgcn_rcpf(s0) : __builtin_nanf("");
    else
      w[k] = sqrtf(s0);
  }
}

// Line-search decision quantity of one lane's far-field column: the change
// f(gj) - f(0) of the data term, sum_k, with ag = a + gj*b formed in FP32 as
// the reference forms fpsi + gamma*fd (solver.py:172; a step below FP32
// resolution gives exactly 0).  Evaluated per element -- |ag|^2 - |a|^2 as a
// product of the (exact) difference and the sum, the log ratio as log1p --
// instead of as a difference of two large sums, whose FP32 rounding is of
// the size of the differences decided on near convergence.
//   poisson:  |ag|^2 - |a|^2 - 2 d (log|ag| - log|a|)
//   gaussian: (|ag| - sqrt d)^2 - (|a| - sqrt d)^2   (d holds sqrt d)
// w: delta_prep of a.
template <int D, int MODEL>
__device__ __forceinline__ float delta_part(const float2 (&a)[D], const float2 (&b)[D],
                                            const float (&d)[D], const float (&w)[D], float gj) {
  float part = 0.f;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const float2 ag = make_float2(a[k].x + gj * b[k].x, a[k].y + gj * b[k].y);
    const float dx = ag.x - a[k].x, dy = ag.y - a[k].y;
    const float ds = dx * (ag.x + a[k].x) + dy * (ag.y + a[k].y);
    if constexpr (MODEL == PT_MODEL_POISSON) {
      // log(|ag|^2 / |a|^2) as log1p of x = ds/|a|^2 = |ag|^2/|a|^2 - 1.  Rare
      // cases (a lane-uniform branch skipped when no lane needs it): x < -15/16,
      // where the candidate nearly cancels a and 1 + x loses the ratio to
      // rounding (there the ratio itself is taken), and |a|^2 or |ag|^2
      // below FLT_MIN (w = NaN; there mlog's clamp at 1e-32 decides and the
      // logs are taken separately).  For x in [-15/16, -1/2) 1 + x is exact,
      // so ln(1 + x) carries x's relative rounding (a few ulp) times
      // |x| / (1 + x) <= 15: under 3e-6 absolute against |ln(1 + x)| >= 0.69.
      // (With -1/2 as the threshold, large candidates -- the first sweep of a
      // step starts at gamma = 2 -- took the branch in most waves.)
      const float x = ds * w[k];
      float lr = log1p_step(x);
      if (!(x >= -0.9375f)) {
        // a through an empty asm statement: its log is candidate-independent,
        // and hoisted out of the candidate loop it would be taken for every
        // element (16 logs and registers per patch) instead of only here
        float2 a0 = a[k];
        asm volatile("" : "+v"(a0.x), "+v"(a0.y));
        const float sg = ag.x * ag.x + ag.y * ag.y;
        const float s0 = a0.x * a0.x + a0.y * a0.y;
        if (s0 >= 4.70197740e-38f && sg >= 1.17549435e-38f)
          lr = __builtin_amdgcn_logf(sg * w[k]) * 0.693147181f;
        else
          lr = 2.f * (log_abs(ag, sg) - log_abs(a0, s0));
      }
      part += ds - d[k] * lr;
    } else {
      const float sg = ag.x * ag.x + ag.y * ag.y;
      const float den = w[k] + sqrtf(sg);
      const float dm = den > 0.f ? ds / den : 0.f;
      part += ds - 2.f * d[k] * dm;
    }
  }
  return part;
}

// Absolute data term at gamma = 0 (take_lagr's lagr[0], solver.py:294-296)
template <int D>
__device__ __forceinline__ float data_term(const float2 (&a)[D], const float (&d)[D], int model) {
  float part = 0.f;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const float s2 = a[k].x * a[k].x + a[k].y * a[k].y;
    if (model == PT_MODEL_POISSON) {
      part += s2 - 2.f * d[k] * log_abs(a[k], s2);
    } else {
      const float e = sqrtf(s2) - d[k];
      part += e * e;
    }
  }
  return part;
}

// Sums over patches, per chunk, of the data term's change f(gamma_j) - f(0)
// at ngam step candidates (lagr = 0), or of the absolute data term of
// take_lagr (lagr != 0, gamma = 0 only); one partial per (chunk, block) in
// partial[(c*gridDim.x + b)*ngam + j].  The candidate
// loop is not unrolled and its FP64 accumulators rotate in registers; the
// LDS footprint is the transpose buffer only.
#define PT_MAX_GAM 8
template <int D, int MODEL>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 3 : 1)))
void k_minf(double* __restrict__ partial,
                                               const float2* __restrict__ f,
                                               const float2* __restrict__ dir,
                                               const float* __restrict__ data,
                                               const float2* __restrict__ prb,
                                               const int2* __restrict__ pos,
                                               const double* __restrict__ gammas, int ngam,
                                               int chunk, int nz, int n, int S, int P, int ox,
                                               int oy, float cs, float cp, float cd, int model,
                                               int lagr, const double* __restrict__ skip) {
  constexpr int G = WAVE / D;
  __shared__ float T[G * D * (D + 1)];
  const int lane = lane_id(), slot = lane / D, r = lane % D;
  const int c = blockIdx.y, bx = blockIdx.x;
  // chunks whose line search has finished (skip[2*c+1] != 0) are not evaluated
  if (skip && skip[2 * c + 1] != 0.0) return;
  __shared__ float gsh[PT_MAX_GAM];
  if (lane < PT_MAX_GAM) gsh[lane] = lane < ngam ? (float)gammas[(long)c * ngam + lane] : 0.f;
  __syncthreads();
  double acc[PT_MAX_GAM];
#pragma unroll
  for (int j = 0; j < PT_MAX_GAM; ++j) acc[j] = 0.0;
  const long npatch = (long)chunk * S;
  const long base = (long)c * chunk * S;
  for (long grp = bx; grp * G < npatch; grp += gridDim.x) {
    const long pl = grp * G + slot;
    const bool active = pl < npatch;
    const long p = base + pl;
    int2 ps = active ? pos[p] : make_int2(-1, -1);
    const int t = active ? (int)(p / S) : 0;
    float2 a[D], b[D];
    float d[D];
    // every global load of the group first (one memory round trip)
    load_rows<D>(a, f, ps, t, r, nz, n, P, ox, oy, active);
    if (dir) load_rows<D>(b, dir, ps, t, r, nz, n, P, ox, oy, active);
    {
      const float* dp = data + (active ? p : 0) * D * D + r;
#pragma unroll
      for (int k = 0; k < D; ++k) d[k] = active ? dp[k * D] : 0.f;
    }
    apply_probe<D>(a, prb, r, P, ox, oy, cs);
    frame_fwd_w<D>(a, T, slot, r);
    if (dir) {
      apply_probe<D>(b, prb, r, P, ox, oy, cs);
      frame_fwd_w<D>(b, T, slot, r);
    } else {
#pragma unroll
      for (int k = 0; k < D; ++k) b[k] = make_float2(0.f, 0.f);
    }
    if (!active) continue;
    float dterm = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      d[k] = d[k] * cd;
      a[k] = cscale(a[k], cp);
      b[k] = cscale(b[k], cp);
      if (model == PT_MODEL_GAUSSIAN) {
        d[k] = sqrtf(d[k]);
      } else if (lagr) {
        dterm += d[k] - 2.f * d[k] * logf(fmaxf(sqrtf(d[k]), 1e-32f));
      }
    }
    // fpsi + gamma*fd formed element-wise in FP32 (solver.py:172): a step
    // below FP32 resolution leaves the term bit-identical to gamma = 0.
    // Candidate j accumulates into acc[0]; the accumulators rotate once per
    // candidate slot (8 rotations per patch group restore their order).
    if (lagr) {
      acc[0] += (double)(data_term<D>(a, d, model) - dterm);
      continue;
    }
    float w[D];
    delta_prep<D, MODEL>(a, w);
#pragma unroll 1
    for (int j = 0; j < PT_MAX_GAM; ++j) {
      // gamma = 0 (candidate 0 of a sweep) changes nothing: its sum stays 0
      if (j < ngam && gsh[j] != 0.f) {
        const float gj = gsh[j];
        const float part = delta_part<D, MODEL>(a, b, d, w, gj);
        acc[0] += (double)part;
      }
      const double t0 = acc[0];
#pragma unroll
      for (int q = 0; q < PT_MAX_GAM - 1; ++q) acc[q] = acc[q + 1];
      acc[PT_MAX_GAM - 1] = t0;
    }
  }
#pragma unroll
  for (int j = 0; j < PT_MAX_GAM; ++j) {
    if (j >= ngam) break;
    const double v = wave_sum(acc[j]);
    if (lane == 0) partial[((long)c * gridDim.x + bx) * ngam + j] = v;
  }
}

// ------------------------------------------------------------------ one wave per frame
// Frame transforms of large detectors with 16 values per lane.  A lane that
// holds a whole frame row (k_minf, tile_body) needs D complex values per array:
// at D = 32 one wave per SIMD fits, at D = 64 the line search spills (10 ms for
// a sweep over 14400 frames).
//
// D = 32: two lanes per row.  Lane l = 2 ix + s holds the row's elements
// 2 j + s, j < 16: a 16-point FFT in registers, then one radix-2 step between
// the two lanes (DPP), after which lane s holds outputs k + 16 s.  The same along
// the columns after an LDS exchange: lane l = 2 ky + s ends with far-field
// elements (kx = m + 16 s, ky), m < 16.
//
// D = 64, probes up to 16 pixels: only 16 x 16 frame elements are not zero.  With
// o the probe's offset, output 4 k1 + k0 of a line is
//   W^(o (4 k1 + k0)) sum_j (x_j W_64^(j k0)) W_16^(j k1):
// four 16-point FFTs of twisted inputs (K = 4 sub-transforms).  Lane l = ix + 16
// k0 transforms a row's sub-transform k0; after the exchange lane l = ky takes
// its column's four sub-transforms in turn (kx = 4 m + c).  5 FFTs of 16 points
// per lane and frame.  The factor W^(o k) has modulus 1 and is left out: the
// functional only sees moduli, and the gradient's residual commutes with it.
template <int D>
struct WaveFrame;

// the partner lane's value (lane ^ 1)
__device__ __forceinline__ int dpp_xor1(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true);
}
__device__ __forceinline__ float lane_xor1(float x) {
  return __int_as_float(dpp_xor1(__float_as_int(x)));
}
__device__ __forceinline__ double lane_xor1(double x) {
  return __hiloint2double(dpp_xor1(__double2hiint(x)), dpp_xor1(__double2loint(x)));
}

// 32-bit words of the 16 complex values of a lane exchanged through the
// wave's LDS buffer: value j goes to wr(j), comes back from rd(j)
template <typename C, class FW, class FR>
__device__ __forceinline__ void wave_exchange(C (&v)[16], float* Ts, FW wr, FR rd) {
  using R = decltype(v[0].x);
  int* Ti = reinterpret_cast<int*>(Ts);
  constexpr int words = sizeof(C) / 4;
  static_for<0, words>([&](auto pc) {
    constexpr int part = decltype(pc)::value;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const R x = part < words / 2 ? v[j].x : v[j].y;
      if constexpr (words == 2) Ti[wr(j)] = __float_as_int(x);
      else Ti[wr(j)] = (part & 1) ? __double2hiint(x) : __double2loint(x);
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int b = Ti[rd(j)];
      R& x = part < words / 2 ? v[j].x : v[j].y;
      if constexpr (words == 2) x = __int_as_float(b);
      else x = (part & 1) ? __hiloint2double(b, __double2loint(x))
                          : __hiloint2double(__double2hiint(x), b);
    }
    wave_sync();
  });
}

template <>
struct WaveFrame<32> {
  static constexpr int kSub = 1;            // column sub-transforms
  static constexpr int kBuf = 32 * 33;      // floats of the exchange buffer
  int l, s;
  __device__ explicit WaveFrame(int lane) : l(lane), s(lane & 1) {}
  // frame element of value j before the transform; far-field element after it
  __device__ int ix() const { return l >> 1; }
  __device__ int iy(int j) const { return 2 * j + s; }
  __device__ int ky() const { return l >> 1; }
  __device__ int kx(int m, int) const { return m + 16 * s; }
  __device__ int wr(int j) const { return (l >> 1) * 33 + j + 16 * s; }
  __device__ int rd(int j) const { return (2 * j + s) * 33 + (l >> 1); }
  template <typename C>
  __device__ __forceinline__ void fwd32(C (&v)[16]) const {
    using R = decltype(v[0].x);
    const R sg = s ? (R)-1 : (R)1;
    reg_fft<16, -1>(v);
    static_for<0, 16>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const C t = twiddle_ct<32, k, -1>(v[k]);
      const C u = cmake(t, s ? t.x : v[k].x, s ? t.y : v[k].y);
      v[k] = cmake(t, lane_xor1(u.x) + sg * u.x, lane_xor1(u.y) + sg * u.y);
    });
  }
  __device__ __forceinline__ void inv32(float2 (&v)[16]) const {
    const float sg = s ? -1.f : 1.f;
    static_for<0, 16>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      const float2 u = make_float2(lane_xor1(v[k].x) + sg * v[k].x,
                                   lane_xor1(v[k].y) + sg * v[k].y);
      const float2 t = twiddle_ct<32, k, 1>(u);
      v[k] = make_float2(s ? t.x : u.x, s ? t.y : u.y);
    });
    reg_fft<16, 1>(v);
  }
  // probe element of value j as it enters the transform (tw unused)
  __device__ float2 twist(float2 x, int, const double2*) const { return x; }
  template <typename C>
  __device__ __forceinline__ void rows(C (&v)[16], float* T, const double2*) const {
    fwd32(v);
    wave_exchange(v, T, [&](int j) { return wr(j); }, [&](int j) { return rd(j); });
  }
  template <typename C>
  __device__ __forceinline__ void cols(const C (&x)[16], C (&y)[16], int, const double2*) const {
#pragma unroll
    for (int j = 0; j < 16; ++j) y[j] = x[j];
    fwd32(y);
  }
  // z += column inverse of sub-transform c (c = 0: the whole)
  __device__ __forceinline__ void cols_inv(float2 (&y)[16], float2 (&z)[16], int,
                                           const double2*) const {
    inv32(y);
#pragma unroll
    for (int j = 0; j < 16; ++j) z[j] = y[j];
  }
  __device__ __forceinline__ void rows_inv(float2 (&z)[16], float* T, const double2*) const {
    wave_exchange(z, T, [&](int j) { return rd(j); }, [&](int j) { return wr(j); });
    inv32(z);
  }
  // frame values of a lane after rows_inv: all 16, element (ix, iy(j))
  static constexpr int kOut = 16;
  __device__ int out_iy(int j) const { return iy(j); }
  __device__ float2 out(const float2 (&z)[16], int j) const { return z[j]; }
  __device__ __forceinline__ void combine(float2 (&)[16]) const {}
};

template <>
struct WaveFrame<64> {
  static constexpr int kSub = 4;
  static constexpr int kBuf = 16 * 68;
  int l, k0;
  __device__ explicit WaveFrame(int lane) : l(lane), k0(lane >> 4) {}
  __device__ int ix() const { return l & 15; }
  __device__ int iy(int j) const { return j; }
  __device__ int ky() const { return l; }
  __device__ int kx(int m, int c) const { return 4 * m + c; }
  __device__ int wr(int k1) const { return (l & 15) * 68 + 4 * k1 + k0; }
  __device__ int rd(int i) const { return i * 68 + l; }
  // tw[m] = exp(-2 pi i m / 64)
  static __device__ __forceinline__ float2 mul(float2 x, double2 w) {
    return cmul(x, make_float2((float)w.x, (float)w.y));
  }
  static __device__ __forceinline__ double2 mul(double2 x, double2 w) {
    return make_double2(x.x * w.x - x.y * w.y, x.x * w.y + x.y * w.x);
  }
  static __device__ __forceinline__ float2 mulc(float2 x, double2 w) {
    return cmulc(x, make_float2((float)w.x, (float)w.y));
  }
  __device__ float2 twist(float2 x, int j, const double2* tw) const {
    return mul(x, tw[(j * k0) & 63]);
  }
  // FP32 rows take inputs whose probe carries the twist, FP64 rows twist here
  __device__ __forceinline__ void rows(float2 (&v)[16], float* T, const double2*) const {
    reg_fft<16, -1>(v);
    wave_exchange(v, T, [&](int j) { return wr(j); }, [&](int j) { return rd(j); });
  }
  __device__ __forceinline__ void rows(double2 (&v)[16], float* T, const double2* tw) const {
#pragma unroll
    for (int j = 1; j < 16; ++j) v[j] = mul(v[j], tw[(j * k0) & 63]);
    reg_fft<16, -1>(v);
    wave_exchange(v, T, [&](int j) { return wr(j); }, [&](int j) { return rd(j); });
  }
  template <typename C>
  __device__ __forceinline__ void cols(const C (&x)[16], C (&y)[16], int c,
                                       const double2* tw) const {
    y[0] = x[0];
#pragma unroll
    for (int j = 1; j < 16; ++j) y[j] = mul(x[j], tw[(j * c) & 63]);
    reg_fft<16, -1>(y);
  }
  __device__ __forceinline__ void cols_inv(float2 (&y)[16], float2 (&z)[16], int c,
                                           const double2* tw) const {
    reg_fft<16, 1>(y);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float2 t = mulc(y[j], tw[(j * c) & 63]);
      z[j] = c ? cadd(z[j], t) : t;
    }
  }
  __device__ __forceinline__ void rows_inv(float2 (&z)[16], float* T, const double2* tw) const {
    wave_exchange(z, T, [&](int j) { return rd(j); }, [&](int j) { return wr(j); });
    reg_fft<16, 1>(z);
#pragma unroll
    for (int j = 1; j < 16; ++j) z[j] = mulc(z[j], tw[(j * k0) & 63]);
  }
  // sum over the four lanes of a row: lane k0 keeps elements 4 k0 .. 4 k0 + 3
  static constexpr int kOut = 4;
  __device__ int out_iy(int j) const { return 4 * k0 + j; }
  __device__ float2 out(const float2 (&z)[16], int j) const { return z[j]; }
  __device__ __forceinline__ void combine(float2 (&z)[16]) const {
    half_sum<8>(z, k0 >> 1, 32);
    half_sum<4>(z, k0 & 1, 16);
  }
  template <int H>
  __device__ __forceinline__ void half_sum(float2 (&z)[16], int up, int mask) const {
#pragma unroll
    for (int i = 0; i < H; ++i) {
      const float2 keep = make_float2(up ? z[H + i].x : z[i].x, up ? z[H + i].y : z[i].y);
      const float2 give = make_float2(up ? z[i].x : z[H + i].x, up ? z[i].y : z[H + i].y);
      z[i] = make_float2(keep.x + __shfl_xor(give.x, mask, 64),
                         keep.y + __shfl_xor(give.y, mask, 64));
    }
  }
};

// exp(-2 pi i m / 64) into LDS (64 x 64 frames)
template <int D>
__device__ __forceinline__ void stage_tw64(double2* tw) {
  if constexpr (D == 64)
    if (threadIdx.x < 64) tw[threadIdx.x] = make_double2(cospi(threadIdx.x / 32.0), -sinpi(threadIdx.x / 32.0));
}

// the probe, scaled and twisted, in lane order: prl[j * WAVE + lane] (all W waves)
template <int W, int D>
__device__ __forceinline__ void stage_probe(float2* prl, const float2* __restrict__ prb,
                                            const WaveFrame<D>& fr, int wave, int lane, int P, int o,
                                            float scale, const double2* tw) {
  const int px = fr.ix() - o;
#pragma unroll
  for (int k = 0; k < 16 / W; ++k) {
    const int j = wave + W * k;
    const int py = fr.iy(j) - o;
    float2 q = make_float2(0.f, 0.f);
    if (px >= 0 && px < P && py >= 0 && py < P)
      q = fr.twist(cscale(prb[(long)px * P + py], scale), j, tw);
    prl[j * WAVE + lane] = q;
  }
}
// a lane's 16 object values of the patch whose first pixel is f[0] (0 outside
// the probe, read unconditionally).  f is uniform over the wave: the loads take
// scalar bases and unsigned 32-bit byte offsets, one for all values of a lane
// where the probe fills the transform's window.
template <class V>
__device__ __forceinline__ V load_at(const V* f, unsigned byte) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(f) + byte);
}
template <int D>
__device__ __forceinline__ void load_frame(float2 (&a)[16], const float2* __restrict__ f,
                                           const WaveFrame<D>& fr, int n, int P, int o) {
  const int px = fr.ix() - o;
  if (P == (D == 32 ? 32 : 16)) {
    const unsigned off = (unsigned)(fr.iy(0) * n + px) * sizeof(float2);
#pragma unroll
    for (int j = 0; j < 16; ++j) a[j] = load_at(f + (D == 32 ? 2 : 1) * j * n, off);
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int py = fr.iy(j) - o;
      const bool in = px >= 0 && px < P && py >= 0 && py < P;
      a[j] = load_at(f, in ? (unsigned)(py * n + px) * sizeof(float2) : 0u);
      if (!in) a[j] = make_float2(0.f, 0.f);
    }
  }
}
// the wave's number within the workgroup, as a scalar: what depends on it alone
// (the patch, its position and addresses) is computed once per wave
__device__ __forceinline__ int wave_uniform() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
}

// Line-search sums of k_minf (lagr = 0) for 32 x 32 frames and for 64 x 64
// frames with probes up to 16 pixels: one wave per patch, kMinfWWaves waves per
// workgroup, one partial per (chunk, workgroup).  A workgroup takes a
// contiguous range of patches and the workgroups run in XCD-contiguous order,
// since neighbouring patches read overlapping object rows.  The probe, scaled
// to the far field and twisted, is staged in LDS in lane order.
// Bound: vector issue and the LDS exchanges, two waves per SIMD (221 registers;
// held to three waves it spills 47 and measured 8 % slower).  Four CG steps'
// sweeps: 119 k frames of 32 x 32 8.9 -> 3.4 ms, 14.4 k frames of 64 x 64 with a
// 16 x 16 probe 40 -> 1.26 ms (a lane per frame row before).
constexpr int kMinfWWaves = 4;
template <int D, int MODEL>
__global__ __launch_bounds__(WAVE * kMinfWWaves, 2)
void k_minf_wave(double* __restrict__ partial, const float2* __restrict__ f,
                 const float2* __restrict__ dir, const float* __restrict__ data,
                 const float2* __restrict__ prb, const int2* __restrict__ pos,
                 const double* __restrict__ gammas, int ngam, int chunk, int nz, int n, int S,
                 int P, int ox, float scale, float cd, const double* __restrict__ skip) {
  using F = WaveFrame<D>;
  __shared__ float2 prl[16 * WAVE];
  __shared__ float Tb[kMinfWWaves][F::kBuf];
  __shared__ double2 tw[D == 64 ? 64 : 1];
  __shared__ float gsh[PT_MAX_GAM];
  __shared__ double red[kMinfWWaves][PT_MAX_GAM];
  const int c = blockIdx.y;
  if (skip && skip[2 * c + 1] != 0.0) return;
  const int wave = wave_uniform(), lane = lane_id();
  const F fr(lane);
  const int o = D == 32 ? ox : 0;           // frame offset of the probe window
  stage_tw64<D>(tw);
  if (threadIdx.x < PT_MAX_GAM)
    gsh[threadIdx.x] = threadIdx.x < ngam ? (float)gammas[(long)c * ngam + threadIdx.x] : 0.f;
  __syncthreads();
  stage_probe<kMinfWWaves>(prl, prb, fr, wave, lane, P, o, scale, tw);
  __syncthreads();
  float* T = Tb[wave];
  double acc[PT_MAX_GAM];
#pragma unroll
  for (int j = 0; j < PT_MAX_GAM; ++j) acc[j] = 0.0;
  const long npatch = (long)chunk * S, base = (long)c * npatch;
  const long per = (npatch + gridDim.x - 1) / gridDim.x;
  const long b0 = (long)xcd_contig(blockIdx.x, gridDim.x) * per;
  const long b1 = min(b0 + per, npatch);
  for (long pl = b0 + wave; pl < b1; pl += kMinfWWaves) {
    const long p = base + pl;
    const int2 ps = pos[p];
    if (ps.x < 0) continue;  // a skipped patch has no far field: its sums do not change
    const int t = (int)(p / S);
    const long at = ((long)t * nz + ps.y) * n + ps.x;
    float2 a[16], b[16];
    load_frame<D>(a, f + at, fr, n, P, o);
    load_frame<D>(b, dir + at, fr, n, P, o);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float2 q = prl[j * WAVE + lane];
      a[j] = cmul(q, a[j]);
      b[j] = cmul(q, b[j]);
    }
    fr.rows(a, T, tw);
    fr.rows(b, T, tw);
    const float* dp = data + p * D * D;
#pragma unroll 1
    for (int sub = 0; sub < F::kSub; ++sub) {
      float d[16], w[16];
#pragma unroll
      for (int m = 0; m < 16; ++m) d[m] = load_at(dp, (unsigned)(fr.kx(m, sub) * D + fr.ky()) * 4u);
      float2 ya[16], yb[16];
      fr.cols(a, ya, sub, tw);
      fr.cols(b, yb, sub, tw);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        d[m] *= cd;
        if (MODEL == PT_MODEL_GAUSSIAN) d[m] = sqrtf(d[m]);
      }
      delta_prep<16, MODEL>(ya, w);
#pragma unroll 1
      for (int j = 0; j < PT_MAX_GAM; ++j) {
        if (j < ngam && gsh[j] != 0.f) acc[0] += (double)delta_part<16, MODEL>(ya, yb, d, w, gsh[j]);
        const double t0 = acc[0];
#pragma unroll
        for (int q = 0; q < PT_MAX_GAM - 1; ++q) acc[q] = acc[q + 1];
        acc[PT_MAX_GAM - 1] = t0;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < PT_MAX_GAM; ++j) {
    const double v = wave_sum(acc[j]);
    if (lane == 0) red[wave][j] = v;
  }
  __syncthreads();
  if (threadIdx.x < ngam) {
    double v = 0.0;
    for (int w = 0; w < kMinfWWaves; ++w) v += red[w][threadIdx.x];
    partial[((long)c * gridDim.x + blockIdx.x) * ngam + threadIdx.x] = v;
  }
}

// k_fwd for 32 x 32 frames and for 64 x 64 frames with probes up to 16 pixels.  A
// wave takes one patch while that needs at most kFwdWBlocks workgroups (four per
// CU), beyond that up to four, which share the staged probe.  Four in a row from the
// first patch on left few frames to a fraction of the CUs: 968 frames of 32 x 32 19
// -> 7.8 us, 392 of 64 x 64 42 -> 12 us; at 26912 frames of 32 x 32 four per wave
// take 59 us.  Bound there: the far field written (3.7 TB/s).
constexpr int kFwdWBlocks = 1024;
template <int D, bool INT>
__global__ __launch_bounds__(WAVE * kMinfWWaves, 3)
void k_fwd_wave(float2* __restrict__ g, float* __restrict__ out, const float2* __restrict__ f,
                const float2* __restrict__ prb, const int2* __restrict__ pos,
                const float2* __restrict__ shift, long npatch, int nz, int n, int S, int P, int ox,
                float cs, float isc) {
  using F = WaveFrame<D>;
  __shared__ float2 prl[16 * WAVE];
  __shared__ float Tb[kMinfWWaves][F::kBuf];
  __shared__ double2 tw[D == 64 ? 64 : 1];
  const int wave = wave_uniform(), lane = lane_id();
  const F fr(lane);
  const int o = D == 32 ? ox : 0;
  stage_tw64<D>(tw);
  __syncthreads();
  stage_probe<kMinfWWaves>(prl, prb, fr, wave, lane, P, o, cs, tw);
  __syncthreads();
  const long per = (npatch + gridDim.x - 1) / gridDim.x;
  const long b0 = (long)xcd_contig(blockIdx.x, gridDim.x) * per;
  const long b1 = min(b0 + per, npatch);
  for (long p = b0 + wave; p < b1; p += kMinfWWaves) {
    const int2 ps = pos[p];
    const long at = ((p / S) * nz + max(ps.y, 0)) * n + max(ps.x, 0);
    float2 a[16];
    load_frame<D>(a, f + at, fr, n, P, o);
    // a skipped patch (x < 0) has a zero far field
#pragma unroll
    for (int j = 0; j < 16; ++j)
      a[j] = ps.x < 0 ? make_float2(0.f, 0.f) : cmul(prl[j * WAVE + lane], a[j]);
    fr.rows(a, Tb[wave], tw);
    const float2 sh = shift[p];
    const long e0 = p * D * D;
#pragma unroll 1
    for (int sub = 0; sub < F::kSub; ++sub) {
      float2 y[16];
      fr.cols(a, y, sub, tw);
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int kx = fr.kx(m, sub), e = kx * D + fr.ky();
        if constexpr (INT) {
          (out + e0)[e] = (y[m].x * y[m].x + y[m].y * y[m].y) * isc;
        } else {
          float2 v = cmul(y[m], sh);
          if constexpr (D == 64) v = F::mul(v, tw[(ox * (kx + fr.ky())) & 63]);
          (g + e0)[e] = v;
        }
      }
    }
  }
}

// Line-search sums of k_minf (lagr = 0), organised by the overlap-add
// tiles: a workgroup of kMinfWaves waves takes one tile, stages the psi and
// d pixels of its EB x EB extended region once in LDS as (psi, d) pairs
// (coalesced rows; the tile's patches then read their frames from LDS
// instead of each loading D overlapping rows from memory) and evaluates the
// tile's patches G at a time, wave w taking groups w, w + kMinfWaves, ...
// A workgroup takes tiles blockIdx.x, blockIdx.x + gridDim.x, ... of its
// chunk (blockIdx.y), kMinfTiles of them: a sweep in which every chunk has
// finished its search (skip) then costs a quarter of the workgroup launches,
// and one in which a single chunk is open still fills the device.  Per-patch arithmetic is that of
// k_minf.  The tiles' sums add up in LDS; one partial per workgroup in
// partial[(c*ngam + j)*gx + workgroup].
// FULL: the probe covers the frame (P = D, no offset): no bounds selects,
// and the probe in LDS is pre-scaled by cs*cp (the far field is linear in
// the probe), so the frames need no scaling after the transform.
constexpr int kMinfWaves = 2;
constexpr int kMinfStage = 16;  // staged pixels per thread: EB*EB <= 64*kMinfWaves*kMinfStage
constexpr int kMinfTiles = 4;   // tiles per workgroup (the grid is capped at tpc / kMinfTiles)
// Arguments of one line-search launch (one instance of a group)
struct MinfTileArgs {
  double* partial;
  const float2* f;
  const float2* dir;
  const float* data;
  const float2* prb;
  const int2* pos;
  const int* tile_start;
  const int* tile_patch;
  const double* gammas;
  const double* skip;
  const float2* hh;
  const float2* lamd;
  const double* rho_dev;
  double* partial_rho;
  double rho_host;
  int ngam, chunk, nty, ntx, B, EB, nz, n, P, ox, oy;
  float cs, cp, cd;
};

// Up to kGroupMax instances of one kernel in one launch: instance i takes
// workgroups start[i] .. start[i+1]-1 (its own grid, flattened); the
// arguments travel by value in the kernel-argument segment.
constexpr int kGroupMax = 8;
template <class A>
struct Group {
  A a[kGroupMax];
  int start[kGroupMax + 1];
  int gx[kGroupMax];  // x extent of each instance's own grid
  int n;
};
// instance of workgroup b (uniform per workgroup)
template <class A>
__device__ __forceinline__ int group_find(const Group<A>& g, int b) {
  int i = 0;
  while (i + 1 < g.n && b >= g.start[i + 1]) ++i;
  return i;
}

// tot[j] += the wave's sum of acc[j], j < ngam: lane j adds sum j, one LDS update for
// all (one per candidate by lane 0 held the wave for each one's read: 5 halvings at
// 64^2, 32 angles, 16 x 16 frames 132 -> 127 us, 7 halvings with 8 x 8 frames 137 ->
// 131 us, at 256^2, 96 angles 776 -> 762 us)
template <int NG>
__device__ __forceinline__ void add_lane_sums(const double (&acc)[NG], int ngam, double* tot,
                                              int lane) {
  double mine = 0.0;
#pragma unroll
  for (int j = 0; j < NG; ++j) {
    if (j >= ngam) break;
    const double v = wave_sum(acc[j]);
    mine = lane == j ? v : mine;
  }
  if (lane < NG) tot[lane] += mine;
}

template <int D, int MODEL, int NG, bool FULL>
__device__ __forceinline__ void minf_tile_body(const MinfTileArgs& A, int c, int bx, int gxn) {
  double* __restrict__ partial = A.partial;
  const float2* __restrict__ f = A.f;
  const float2* __restrict__ dir = A.dir;
  const float* __restrict__ data = A.data;
  const float2* __restrict__ prb = A.prb;
  const int2* __restrict__ pos = A.pos;
  const int* __restrict__ tile_start = A.tile_start;
  const int* __restrict__ tile_patch = A.tile_patch;
  const double* __restrict__ gammas = A.gammas;
  const double* __restrict__ skip = A.skip;
  const float2* __restrict__ hh = A.hh;
  const float2* __restrict__ lamd = A.lamd;
  const double* __restrict__ rho_dev = A.rho_dev;
  double* __restrict__ partial_rho = A.partial_rho;
  const double rho_host = A.rho_host;
  const int ngam = A.ngam, chunk = A.chunk, nty = A.nty, ntx = A.ntx, B = A.B, EB = A.EB;
  const int nz = A.nz, n = A.n, P = A.P, ox = A.ox, oy = A.oy;
  const float cs = A.cs, cp = A.cp, cd = A.cd;
  constexpr int G = WAVE / D;
  // LDS: EB*EB (psi, d) pairs, the probe (P*P), then the transpose buffers
  extern __shared__ float4 lds_pd[];
  if (skip && skip[2 * c + 1] != 0.0) return;
  const int wave = threadIdx.x / WAVE, lane = lane_id(), slot = lane / D, r = lane % D;
  float2* prl = reinterpret_cast<float2*>(lds_pd + EB * EB);
  float* T = reinterpret_cast<float*>(prl + ((P * P + 1) & ~1)) + wave * G * D * (D + 1);
  const float pscale = FULL ? cs * cp : 1.f;
  // FULL (P = D): the probe staged transposed, [iy][ix], so that the lanes of a
  // frame (rows ix) read consecutive words for each column iy; row-major, the
  // 16 lanes' reads fell on two banks.  Otherwise row-major for apply_probe.
  for (int i = threadIdx.x; i < P * P; i += blockDim.x) {
    if constexpr (FULL) prl[(i % D) * D + i / D] = cscale(prb[i], pscale);
    else prl[i] = cscale(prb[i], pscale);
  }
  __shared__ float gsh[NG];
  __shared__ double tot[2][kMinfWaves][NG];  // data term, rho term; each wave adds to its own
  if (lane < NG) tot[0][wave][lane] = tot[1][wave][lane] = 0.0;
  const int tpa = nty * ntx, tpc = chunk * tpa;
  if (threadIdx.x < NG)
    gsh[threadIdx.x] = threadIdx.x < ngam ? (float)gammas[(long)c * ngam + threadIdx.x] : 0.f;
  const float rho = (float)(rho_dev ? rho_dev[0] : rho_host);
  const int ix = r - ox;
  for (int tb = bx; tb < tpc; tb += gxn) {
    const long tile = (long)c * tpc + tb;
    const int t = (int)(tile / tpa);
    const int rem = (int)(tile - (long)t * tpa);
    const int y0 = (rem / ntx) * B, x0 = (rem % ntx) * B;
    const int beg = tile_start[tile], end = tile_start[tile + 1];
    __syncthreads();  // the previous tile's frames are read (and the probe staged)
    if (end > beg) {
      // all loads of the region first (one memory round trip), then the
      // stores.  The thread index is passed through an empty asm statement:
      // the staging offsets are then recomputed per tile instead of being
      // hoisted out of the tile loop (where kMinfStage offsets and masks
      // would hold registers through the whole patch loop)
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));
      const float2* fz = f + (long)t * nz * n;
      const float2* dz = dir + (long)t * nz * n;
      float2 va[kMinfStage], vb[kMinfStage];
#pragma unroll
      for (int u = 0; u < kMinfStage; ++u) {
        const int i = tid + u * WAVE * kMinfWaves;
        const int yy = i / EB, xx = i - yy * EB;
        const int y = y0 + yy, x = x0 + xx;
        const bool in = i < EB * EB && y < nz && x < n;
        va[u] = in ? fz[(long)y * n + x] : make_float2(0.f, 0.f);
        vb[u] = in ? dz[(long)y * n + x] : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int u = 0; u < kMinfStage; ++u) {
        const int i = tid + u * WAVE * kMinfWaves;
        if (i < EB * EB) lds_pd[i] = make_float4(va[u].x, va[u].y, vb[u].x, vb[u].y);
      }
    }
    __syncthreads();
    double acc[NG];  // candidate slots (NG >= ngam)
#pragma unroll
    for (int j = 0; j < NG; ++j) acc[j] = 0.0;
    for (int i0 = beg + wave * G; i0 < end; i0 += kMinfWaves * G) {
      const int ii = i0 + slot;
      const bool active = ii < end;
      // a slot past the tile's last patch recomputes the tile's first one
      // (in bounds, results dropped)
      const long p = tile_patch[active ? ii : beg];
      const int2 ps = pos[p];
      float2 a[D], b[D];
      if constexpr (FULL) {
        const float4* src = lds_pd + (ps.y - y0) * EB + ps.x + r - x0;
        const float2* pp = prl + r;
#pragma unroll
        for (int k = 0; k < D; ++k) {
          const float4 v = src[k * EB];
          const float2 q = pp[k * D];
          a[k] = cmul(q, make_float2(v.x, v.y));
          b[k] = cmul(q, make_float2(v.z, v.w));
        }
        frame_fwd_w<D>(a, T, slot, r);
        frame_fwd_w<D>(b, T, slot, r);
      } else {
        const bool rowin = ix >= 0 && ix < P;
        const float4* src = lds_pd + (ps.y - oy - y0) * EB + ps.x + ix - x0;
#pragma unroll
        for (int k = 0; k < D; ++k) {
          const int iy = k - oy;
          float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
          if (rowin && iy >= 0 && iy < P) v = src[k * EB];
          a[k] = make_float2(v.x, v.y);
          b[k] = make_float2(v.z, v.w);
        }
        apply_probe<D>(a, prl, r, P, ox, oy, cs);
        frame_fwd_w<D>(a, T, slot, r);
        apply_probe<D>(b, prl, r, P, ox, oy, cs);
        frame_fwd_w<D>(b, T, slot, r);
#pragma unroll
        for (int k = 0; k < D; ++k) {
          a[k] = cscale(a[k], cp);
          b[k] = cscale(b[k], cp);
        }
      }
      if (!active) continue;
      // the data column after the transforms: loaded earlier, it would hold
      // D registers through them
      float d[D];
      {
        const float* dp = data + p * D * D + r;
#pragma unroll
        for (int k = 0; k < D; ++k) d[k] = dp[k * D];
      }
#pragma unroll
      for (int k = 0; k < D; ++k) {
        d[k] = d[k] * cd;
        if (MODEL == PT_MODEL_GAUSSIAN) d[k] = sqrtf(d[k]);
      }
      float w[D];
      delta_prep<D, MODEL>(a, w);
#pragma unroll 1
      for (int j = 0; j < NG; ++j) {
        if (j < ngam && gsh[j] != 0.f) acc[0] += (double)delta_part<D, MODEL>(a, b, d, w, gsh[j]);
        const double t0 = acc[0];
#pragma unroll
        for (int q = 0; q < NG - 1; ++q) acc[q] = acc[q + 1];
        acc[NG - 1] = t0;
      }
    }
    add_lane_sums<NG>(acc, ngam, tot[0][wave], lane);
    if (!hh) continue;
    // The functional's rho term (solver.py:213), change of
    // |h - (psi + g*d) + lamd/rho|^2 from g = 0 per pixel, over the pixels
    // this tile owns: its B x B core, and for the last tile of a row or
    // column of tiles everything up to the object's edge (inside the
    // extended region), so the tiles of an angle partition it.  psi and d
    // were just staged from the same lines (cached).
    const int ty = rem / ntx, tx = rem % ntx;
    const int wy = (ty == nty - 1 ? nz : y0 + B) - y0, wx = (tx == ntx - 1 ? n : x0 + B) - x0;
#pragma unroll
    for (int j = 0; j < NG; ++j) acc[j] = 0.0;
    for (int i = threadIdx.x; i < wy * wx; i += blockDim.x) {
      const int yy = i / wx, xx = i - yy * wx;
      const long o = ((long)t * nz + y0 + yy) * n + x0 + xx;
      const float2 a = hh[o], pv = f[o], l = lamd[o], dd = dir[o];
      const float lx = l.x / rho, ly = l.y / rho;
      const float r0x = a.x - pv.x + lx, r0y = a.y - pv.y + ly;
#pragma unroll
      for (int j = 0; j < NG; ++j) {
        if (j < ngam) {
          const float g = gsh[j];
          const float tx2 = pv.x + g * dd.x, ty2 = pv.y + g * dd.y;
          const float rx = a.x - tx2 + lx, ry = a.y - ty2 + ly;
          acc[j] += (double)((rx - r0x) * (rx + r0x) + (ry - r0y) * (ry + r0y));
        }
      }
    }
    add_lane_sums<NG>(acc, ngam, tot[1][wave], lane);
  }
  __syncthreads();
  const int term = wave, j = lane;  // two waves: wave 0 the data term, wave 1 the rho term
  static_assert(kMinfWaves == 2, "one wave per term");
  if (j < ngam && (term == 0 || hh))
    (term ? partial_rho : partial)[((long)c * ngam + j) * gxn + bx] = tot[term][0][j] + tot[term][1][j];
}

template <int D, int MODEL, int NG, bool FULL>
__global__ __launch_bounds__(WAVE * kMinfWaves) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 3 : 1)))
void k_minf_tile(MinfTileArgs A) {
  minf_tile_body<D, MODEL, NG, FULL>(A, blockIdx.y, blockIdx.x, gridDim.x);
}
// the same for a group of instances (grid: the instances' (gx x nchunk) grids
// flattened, chunk-major)
template <int D, int MODEL, int NG, bool FULL>
__global__ __launch_bounds__(WAVE * kMinfWaves) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 3 : 1)))
void k_minf_tile_group(Group<MinfTileArgs> g) {
  const int i = group_find(g, blockIdx.x);
  const int local = blockIdx.x - g.start[i], gx = g.gx[i];
  minf_tile_body<D, MODEL, NG, FULL>(g.a[i], local / gx, local % gx, gx);
}

// Sums of the k_minf_tile partials (layout [chunk][gamma][block]): one
// 256-thread workgroup per (chunk, gamma), thread-strided sums in block
// order, then the fixed-shape workgroup tree (deterministic).
__global__ __launch_bounds__(256) void k_reduce_partials_t(double* __restrict__ out,
                                                           const double* __restrict__ partial,
                                                           long nblk, int ngam,
                                                           const double* __restrict__ skip) {
  __shared__ double sm[16];
  const int c = blockIdx.x, j = blockIdx.y;
  if (skip && skip[2 * c + 1] != 0.0) return;
  const double* src = partial + ((long)c * ngam + j) * nblk;
  double v[1] = {0.0};
  for (long b = threadIdx.x; b < nblk; b += blockDim.x) v[0] += src[b];
  block_sum<1>(v, sm);
  if (threadIdx.x == 0) out[c * ngam + j] = v[0];
}

// One reduction of k_reduce_partials_t (one instance of a group)
struct ReduceArgs {
  double* out;
  const double* partial;
  const double* skip;
  long nblk;
};
// grid (flattened chunks of the instances, ngam); g.gx: chunks per instance
__global__ __launch_bounds__(256) void k_reduce_partials_group(Group<ReduceArgs> g, int ngam) {
  __shared__ double sm[16];
  const int i = group_find(g, blockIdx.x);
  const ReduceArgs& A = g.a[i];
  const int c = blockIdx.x - g.start[i], j = blockIdx.y;
  if (A.skip && A.skip[2 * c + 1] != 0.0) return;
  const double* src = A.partial + ((long)c * ngam + j) * A.nblk;
  double v[1] = {0.0};
  for (long b = threadIdx.x; b < A.nblk; b += blockDim.x) v[0] += src[b];
  block_sum<1>(v, sm);
  if (threadIdx.x == 0) A.out[c * ngam + j] = v[0];
}

// Sums of a sweep's partials of both terms and its decision, one workgroup per
// chunk: a wave per (term, candidate) adds the partials in a fixed order, then one
// lane applies the halving rule.  The two reductions and the selection this
// replaces (and, off the tile path, the rho term's second pass) were 62 of some 330
// launches of an ADMM iteration, each 3.5 us in small problems: iteration at 64^3
// 1.99 -> 1.87 ms, 4 CG steps at 128^2, 64 angles, 64 x 64 frames 3.13 -> 3.02 ms.
// The line search on tiles writes a partial per workgroup (an eighth of one per
// wave and tile), since one workgroup per chunk reads them: 7 us at 256^3.
struct LsFinishArgs {
  double* state;
  const double* cand;
  double* cand_next;
  double* step;
  const double* w;       // weights of the two terms
  const double* p[2];    // partials of chunk c, candidate j, block b:
  long cs[2], js[2], bs[2];  // p[c*cs + j*js + b*bs]
  int nb[2];
  int ngam, ngam_next, last;
};
__device__ __forceinline__ void ls_finish_body(const LsFinishArgs& A, int c) {
  __shared__ double f[2][PT_MAX_GAM];
  const int wid = threadIdx.x / WAVE, lane = lane_id();
  if (A.state[2 * c + 1] != 0.0) return;
  const int term = wid / PT_MAX_GAM, j = wid % PT_MAX_GAM;
  if (j < A.ngam) {
    const double* src = A.p[term] + c * A.cs[term] + j * A.js[term];
    const long bs = A.bs[term];
    const int nb = A.nb[term];
    double s = 0.0;
#pragma unroll 8
    for (int b = lane; b < nb; b += WAVE) s += src[b * bs];
    s = wave_sum(s);
    if (lane == 0) f[term][j] = s;
  }
  __syncthreads();
  if (threadIdx.x) return;
  const double w0 = A.w[0], w1 = A.w[1];
  ls_decide(A.state + 2 * c, A.step + 2 * c, A.cand + c * A.ngam, A.cand_next + c * A.ngam_next,
            A.ngam, A.ngam_next, A.last, [&](int k) {
#pragma clang fp contract(off)
              return w0 * f[0][k] + w1 * f[1][k];
            });
}
__global__ __launch_bounds__(1024) void k_ls_finish(LsFinishArgs A) {
  ls_finish_body(A, blockIdx.x);
}
// the same for a group of instances (their chunks flattened): the same sums in the
// same order, so that a grouped sweep decides as the instance's own would
__global__ __launch_bounds__(1024) void k_ls_finish_group(Group<LsFinishArgs> g) {
  const int i = group_find(g, blockIdx.x);
  ls_finish_body(g.a[i], blockIdx.x - g.start[i]);
}

// LDS bytes of a k_minf_tile workgroup
inline size_t minf_tile_lds_bytes(int D, int EB, int P) {
  return sizeof(float4) * (size_t)EB * EB + sizeof(float2) * (size_t)((P * P + 1) & ~1) +
         sizeof(float) * (size_t)kMinfWaves * (64 / D) * D * (D + 1);
}

__global__ __launch_bounds__(64) void k_reduce_partials(double* __restrict__ out,
                                                         const double* __restrict__ partial,
                                                         int nblk, int ngam,
                                                         const double* __restrict__ skip) {
  // one wave per (chunk, gamma): lane-strided sums in block order, then a
  // fixed-shape wave tree (deterministic)
  const int c = blockIdx.x, j = blockIdx.y, lane = threadIdx.x;
  if (skip && skip[2 * c + 1] != 0.0) return;
  double s = 0.0;
  for (int b = lane; b < nblk; b += WAVE) s += partial[((long)c * nblk + b) * ngam + j];
  s = wave_sum(s);
  if (lane == 0) out[c * ngam + j] = s;
}

// ------------------------------------------------------------------ tiles
enum { TILE_ADJ = 0, TILE_GRAD = 1 };

// Waves per overlap-add workgroup.  Waves of one workgroup would share the
// LDS tile and have to add in turn (barrier-separated, deterministic); one
// wave per tile avoids the serialisation, and small tiles keep many tiles
// resident per CU.
template <int D>
constexpr int tile_waves() { return 1; }

// Arguments of one overlap-add tile launch (one instance of a group)
struct TileArgs {
  float2* scratch;
  const float2* gin;
  const float2* f;
  const float* data;
  const float2* prb;
  const int2* pos;
  const float2* shift;
  const int* tile_start;
  const int* tile_patch;
  const int* tile_slot;
  int nty, ntx, B, EB, nz, n, S, P, ox, oy;
  float cs, cp, cd, out_scale;
};

// a * b with the roundings spelled out: the gradient's FP64 transform takes the
// rounded products, and the Poisson residual magnifies a change of their last bits
// where the far field is small, so which product a multiply-add rounds first is not
// left to the compiler (it chose otherwise for 8 x 8 frames that fill the detector
// than for the rest)
__device__ __forceinline__ float2 cmul_fma(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x));
}

// body of workgroup b of nb (one per tile).  MODEL: the gradient's data model (any
// value for the adjoint).  FULL: the probe covers the frame, so every frame
// element is added without a bounds check.
// The data column is loaded between the two passes of the FP64 transform: loaded
// with the object rows it held D registers through the first pass, and with the
// run-time model and bounds masks the 16 x 16 gradient took 256 registers and
// spilled 31 of them.  Now 130, three waves per SIMD (the LDS tile's limit); at
// 256^3, 384 angles, 1.43 M frames 1.54 -> 1.19 ms per launch.  Bound: vector issue
// of the FP64 transform, residual and inverse (about 1700 instructions per four
// frames, 1.0 ms).  The loads do not branch: a branch between the passes splits
// the FP64 transform into two blocks, the compiler contracts its products
// differently, and the gradient differs in the last bit.
template <int D, int MODE, int MODEL, bool FULL>
__device__ __forceinline__ void tile_body(const TileArgs& A, int b, int nb) {
  float2* __restrict__ scratch = A.scratch;
  const float2* __restrict__ gin = A.gin;
  const float2* __restrict__ f = A.f;
  const float* __restrict__ data = A.data;
  const float2* __restrict__ prb = A.prb;
  const int2* __restrict__ pos = A.pos;
  const float2* __restrict__ shift = A.shift;
  const int* __restrict__ tile_start = A.tile_start;
  const int* __restrict__ tile_patch = A.tile_patch;
  const int* __restrict__ tile_slot = A.tile_slot;
  const int nty = A.nty, ntx = A.ntx, B = A.B, EB = A.EB, nz = A.nz, n = A.n;
  const int P = FULL ? D : A.P, ox = FULL ? 0 : A.ox, oy = FULL ? 0 : A.oy;
  const float cs = A.cs, cp = A.cp, cd = A.cd, out_scale = A.out_scale;
  constexpr int G = WAVE / D;
  constexpr int W = tile_waves<D>();
  extern __shared__ float lds_f[];
  float2* acc = reinterpret_cast<float2*>(lds_f);          // EB*EB
  const int wave = threadIdx.x / WAVE;
  float* T = lds_f + 2 * EB * EB + wave * G * D * (D + 1);  // this wave's buffer
  // XCD-contiguous tile order: adjacent tiles' extended regions overlap (5.9
  // -> 5.6 ms per 256^3 iteration; the line-search and forward kernels
  // measured slower with it -- line search 12.5 -> 15.7 ms -- and keep the
  // hardware order)
  const long tile = xcd_contig(b, nb);
  const int slotid = tile_slot[tile];
  if (slotid < 0) return;
  const int lane = lane_id(), slot = lane / D, r = lane % D;
  const int tpa = nty * ntx;
  const int t = (int)(tile / tpa);
  const int rem = (int)(tile - (long)t * tpa);
  const int y0 = (rem / ntx) * B, x0 = (rem % ntx) * B;
  for (int i = threadIdx.x; i < EB * EB; i += W * WAVE) acc[i] = make_float2(0.f, 0.f);
  __syncthreads();
  const int beg = tile_start[tile], end = tile_start[tile + 1];
  const int ix = r - ox;
  // probe column of this lane's frame row in registers (frames up to 32 x 32;
  // 64 x 64 frames read it from memory, which is cached)
  constexpr int NPR = D <= 32 ? D : 1;
  float2 pr[NPR];
  if constexpr (D <= 32) probe_row<D>(pr, prb, r, P, ox, oy, 1.0f);
  auto prv = [&](int k) -> float2 {
    if constexpr (D <= 32) return pr[k];
    const int iy = k - oy;
    return (ix >= 0 && ix < P && iy >= 0 && iy < P) ? prb[(long)ix * P + iy]
                                                    : make_float2(0.f, 0.f);
  };
  for (int i0 = beg; i0 < end; i0 += W * G) {
    const int ii = i0 + wave * G + slot;
    const bool active = ii < end;
    const long p = active ? tile_patch[ii] : 0;
    const int2 ps = active ? pos[p] : make_int2(-1, -1);
    float2 v[D];
    if constexpr (MODE == TILE_ADJ) {
      // lane c loads far-field column c, removes the per-patch phase
      if (active) {
        const float2 sh = shift[p];
        const float2* gp = gin + p * D * D + r;
#pragma unroll
        for (int k = 0; k < D; ++k) v[k] = cmulc(gp[k * D], sh);
      } else {
#pragma unroll
        for (int k = 0; k < D; ++k) v[k] = make_float2(0.f, 0.f);
      }
    } else {
      load_rows<D>(v, f, ps, t, r, nz, n, P, ox, oy, active);
#pragma unroll
      for (int k = 0; k < D; ++k) v[k] = cscale(cmul_fma(prv(k), v[k]), cs);
      // a = coefptycho * F(c * prb * psi), rounded once after an FP64 transform
      float dv[D];
      frame_fwd64_w<D>(v, T, slot, r, cp, [&]() {
        const float* dp = data + p * D * D + r;
#pragma unroll
        for (int k = 0; k < D; ++k) dv[k] = dp[k * D];  // patch 0's where not active
      });
      // residual in the unshifted frame (the per-patch unimodular factor of
      // kernels.cuh:319-355 cancels: r(s*a) = s*r(a), F* removes s again)
      if (active) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
          const float d = dv[k] * cd;
          const float2 a = v[k];
          const float aa = a.x * a.x + a.y * a.y;
          float2 res;
          if constexpr (MODEL == PT_MODEL_POISSON) {
            // IEEE division: where |a| is small the quotient's relative error
            // becomes a large absolute error of the residual, and a 1-ulp
            // reciprocal there moves a 36-step CG run 6x farther from FP64
            const float q = d / (aa + 1e-32f);
            res = make_float2(a.x - q * a.x, a.y - q * a.y);
          } else {
            const float m = sqrtf(aa);
            const float sd = sqrtf(d);
            if (m > 0.f) {
              const float q = sd / m;
              res = make_float2(a.x - q * a.x, a.y - q * a.y);
            } else {
              // angle(0) = 0 in the shifted frame: r = -sqrt(d) there
              const float2 sh = shift[p];
              res = make_float2(-sd * sh.x, sd * sh.y);
            }
          }
          v[k] = res;
        }
      }
    }
    frame_inv_w<D>(v, T, slot, r);
    // overlap-add of c*conj(prb)*frame into the LDS tile.  The G patches of a
    // wave overlap, so they are added one slot at a time, in slot order
    // (deterministic): within a slot every lane owns distinct pixels, so a
    // plain LDS read-add-write (all 16 rows read first, then written) needs
    // no atomics; waves of a workgroup take turns.
    const bool adds = active && ps.x >= 0 && ix >= 0 && ix < P;
    const int col = ps.x + ix - x0;
    const int rowb = ps.y - oy - y0;
#pragma unroll
    for (int k = 0; k < D; ++k) v[k] = cscale(cmulc(v[k], prv(k)), out_scale);
    constexpr int KB = D < 8 ? D : 8;   // rows read before they are written back
#pragma unroll 1
    for (int w = 0; w < W; ++w) {
      if (w == wave) {
#pragma unroll 1
        for (int sl = 0; sl < G; ++sl) {
          if (sl == slot && adds) {
#pragma unroll
            for (int k0 = 0; k0 < D; k0 += KB) {
              float2 cur[KB];
#pragma unroll
              for (int kk = 0; kk < KB; ++kk) {
                const int iy = k0 + kk - oy;
                if (iy >= 0 && iy < P) cur[kk] = acc[(rowb + k0 + kk) * EB + col];
              }
#pragma unroll
              for (int kk = 0; kk < KB; ++kk) {
                const int iy = k0 + kk - oy;
                if (iy >= 0 && iy < P)
                  acc[(rowb + k0 + kk) * EB + col] = cadd(cur[kk], v[k0 + kk]);
              }
            }
          }
          wave_sync();
        }
      }
      if constexpr (W > 1) __syncthreads();
    }
  }
  if constexpr (W == 1) wave_sync();
  else __syncthreads();
  float2* out = scratch + (long)slotid * EB * EB;
  for (int i = threadIdx.x; i < EB * EB; i += W * WAVE) out[i] = acc[i];
}
template <int D, int MODE, int MODEL, bool FULL>
__global__ __launch_bounds__(WAVE * tile_waves<D>()) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 3 : 1))) void k_tile(TileArgs A) {
  tile_body<D, MODE, MODEL, FULL>(A, blockIdx.x, gridDim.x);
}
// the same for a group of instances (their tile grids flattened)
template <int D, int MODE, int MODEL, bool FULL>
__global__ __launch_bounds__(WAVE * tile_waves<D>()) __attribute__((amdgpu_waves_per_eu(D <= 16 ? 3 : 1)))
void k_tile_group(Group<TileArgs> g) {
  const int i = group_find(g, blockIdx.x);
  tile_body<D, MODE, MODEL, FULL>(g.a[i], blockIdx.x - g.start[i], g.gx[i]);
}

// tile_body for 32 x 32 frames and for 64 x 64 frames with probes up to 16
// pixels (WaveFrame): kTileW waves per tile, each taking every kTileW-th of the
// tile's patches, adding to the shared LDS tile in turn (a barrier between
// turns), so the order of the sums is the list's.  With one wave per tile the 30
// KB tiles left one wave per SIMD.  Bound: the FP64 transform's issue (0.44 of
// 0.67 ms at 119 k frames of 32 x 32) and the LDS exchanges at two waves per SIMD.
// What depends on the patch alone is scalar (wave_uniform, load_at), the data model
// a template argument: gradient of 119 k frames of 32 x 32 1.09 -> 0.67 ms (with
// 64-bit addresses per lane and value, and both models' code, it spilled 58
// registers), of 14.4 k of 64 x 64 0.44 -> 0.35 ms; a lane per frame row took 1.04
// and 1.18 ms.  Adjoint of 20 k frames of 32 x 32 72 us.
// (Six waves for the 32 x 32 gradient, 160 registers and three waves per SIMD,
// measured 1.01 ms against 0.67: more turns at the shared tile.)
constexpr int kTileW = 4;
template <int D, int MODE, int MODEL>
__device__ __forceinline__ void tile_body_w(const TileArgs& A, int b, int nb) {
  using F = WaveFrame<D>;
  const int EB = A.EB, n = A.n, P = A.P;
  extern __shared__ float lds_f[];
  float2* acc = reinterpret_cast<float2*>(lds_f);
  double2* tw = reinterpret_cast<double2*>(lds_f + ((2 * EB * EB + 3) & ~3) + 2 * WAVE);
  const int wave = wave_uniform(), lane = lane_id();
  float2* prl = reinterpret_cast<float2*>(tw + (D == 64 ? 64 : 0));
  float* T = reinterpret_cast<float*>(prl + (MODE == TILE_GRAD ? 16 * WAVE : 0)) + wave * F::kBuf;
  const long tile = xcd_contig(b, nb);
  const int slotid = A.tile_slot[tile];
  if (slotid < 0) return;
  const int tpa = A.nty * A.ntx;
  const int t = (int)(tile / tpa), rem = (int)(tile - (long)t * tpa);
  const int y0 = (rem / A.ntx) * A.B, x0 = (rem % A.ntx) * A.B;
  for (int i = threadIdx.x; i < EB * EB; i += kTileW * WAVE) acc[i] = make_float2(0.f, 0.f);
  stage_tw64<D>(tw);
  const F fr(lane);
  const int o = D == 32 ? A.ox : 0;
  const int px = fr.ix() - o;
  const bool colin = px >= 0 && px < P;
  // gradient: the probe times c = 1/D (exact) staged in lane order, untwisted.  The
  // adjoint uses it once per patch and reads it from memory: 8 KB more would cost
  // it a workgroup per CU (91 -> 99 us at 20 k frames of 32 x 32).
  if constexpr (MODE == TILE_GRAD) {
    for (int j = wave; j < 16; j += kTileW) {
      const int py = fr.iy(j) - o;
      const bool in = colin && py >= 0 && py < P;
      prl[j * WAVE + lane] = in ? cscale(A.prb[(long)px * P + py], A.cs) : make_float2(0.f, 0.f);
    }
  }
  const float oscale = MODE == TILE_GRAD ? A.out_scale / A.cs : A.out_scale;
  __syncthreads();
  const int beg = A.tile_start[tile], end = A.tile_start[tile + 1];
  for (int i0 = beg; i0 < end; i0 += kTileW) {
    const int ii = i0 + wave;
    const bool active = ii < end;
    int2 ps = make_int2(0, 0);
    float2 z[16];
    if (active) {
      const long p = A.tile_patch[ii];
      ps = A.pos[p];
      const float2 sh = A.shift[p];
      double2 x[MODE == TILE_GRAD ? 16 : 1];
      if constexpr (MODE == TILE_GRAD) {
        // a = coefptycho * F(c * prb * psi), rounded once after an FP64 transform
        const long at = ((long)t * A.nz + ps.y) * n + ps.x;
        float2 v[16];
        load_frame<D>(v, A.f + at, fr, n, P, o);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float2 q = cmul_fma(prl[j * WAVE + lane], v[j]);
          x[j] = make_double2((double)q.x, (double)q.y);
        }
        fr.rows(x, T, tw);
      }
#pragma unroll 1
      for (int sub = 0; sub < F::kSub; ++sub) {
        float2 y[16];
        const long e0 = p * D * D;
        if constexpr (MODE == TILE_ADJ) {
          // the per-patch phase removed; at D = 64 also the factor W^(o k) of the
          // probe's offset, which the sub-transforms leave out
#pragma unroll
          for (int m = 0; m < 16; ++m) y[m] = cmulc(load_at(A.gin + e0, (unsigned)(fr.kx(m, sub) * D + fr.ky()) * 8u), sh);
          if constexpr (D == 64) {
#pragma unroll
            for (int m = 0; m < 16; ++m)
              y[m] = F::mulc(y[m], tw[(A.ox * (fr.kx(m, sub) + fr.ky())) & 63]);
          }
        } else {
          {
            double2 yd[16];
            fr.cols(x, yd, sub, tw);
            const double sd = (double)A.cp;
#pragma unroll
            for (int m = 0; m < 16; ++m)
              y[m] = make_float2((float)(yd[m].x * sd), (float)(yd[m].y * sd));
          }
          __builtin_amdgcn_sched_barrier(0);  // the data after the FP64 transform: registers
          float dv[16];
#pragma unroll
          for (int m = 0; m < 16; ++m) dv[m] = load_at(A.data + e0, (unsigned)(fr.kx(m, sub) * D + fr.ky()) * 4u);
          // residual as in tile_body
#pragma unroll
          for (int m = 0; m < 16; ++m) {
            const float d = dv[m] * A.cd;
            const float2 a = y[m];
            const float aa = a.x * a.x + a.y * a.y;
            float2 res;
            if constexpr (MODEL == PT_MODEL_POISSON) {
              const float q = d / (aa + 1e-32f);
              res = make_float2(a.x - q * a.x, a.y - q * a.y);
            } else {
              const float mo = sqrtf(aa);
              const float sd = sqrtf(d);
              const float q = sd / mo;
              res = make_float2(a.x - q * a.x, a.y - q * a.y);
              if (!(mo > 0.f)) {
                // angle(0) = 0 in the shifted frame
                res = make_float2(-sd * sh.x, sd * sh.y);
                if constexpr (D == 64)
                  res = F::mulc(res, tw[(A.ox * (fr.kx(m, sub) + fr.ky())) & 63]);
              }
            }
            y[m] = res;
          }
        }
        fr.cols_inv(y, z, sub, tw);
      }
      fr.rows_inv(z, T, tw);
      fr.combine(z);
#pragma unroll
      for (int j = 0; j < F::kOut; ++j) {
        float2 q;
        if constexpr (MODE == TILE_GRAD) {
          q = prl[(D == 64 ? fr.out_iy(j) : j) * WAVE + lane];
        } else {
          const int py = fr.out_iy(j) - o;
          q = A.prb[colin && py >= 0 && py < P ? (long)px * P + py : 0];
        }
        z[j] = cscale(cmulc(z[j], q), oscale);
      }
    }
    // tile index of each kept value; values outside the probe go to a slot of
    // the lane's own behind the tile, so that the additions need no branches
    int at[F::kOut];
#pragma unroll
    for (int j = 0; j < F::kOut; ++j) {
      const int fy = fr.out_iy(j), py = fy - o;
      at[j] = colin && py >= 0 && py < P ? (ps.y + py - y0) * EB + ps.x + px - x0
                                         : EB * EB + lane;
    }
#pragma unroll 1
    for (int w = 0; w < kTileW; ++w) {
      if (w == wave && active) {
        // all reads, then all writes: the lane's pixels are distinct
        float2 cur[F::kOut];
#pragma unroll
        for (int j = 0; j < F::kOut; ++j) cur[j] = acc[at[j]];
#pragma unroll
        for (int j = 0; j < F::kOut; ++j) acc[at[j]] = cadd(cur[j], z[j]);
      }
      __syncthreads();
    }
  }
  float2* out = A.scratch + (long)slotid * EB * EB;
  for (int i = threadIdx.x; i < EB * EB; i += kTileW * WAVE) out[i] = acc[i];
}
template <int D, int MODE, int MODEL>
__global__ __launch_bounds__(WAVE * kTileW, 2) void k_tile_w(TileArgs A) {
  tile_body_w<D, MODE, MODEL>(A, blockIdx.x, gridDim.x);
}
template <int D, int MODE, int MODEL>
__global__ __launch_bounds__(WAVE * kTileW, 2) void k_tile_w_group(Group<TileArgs> g) {
  const int i = group_find(g, blockIdx.x);
  tile_body_w<D, MODE, MODEL>(g.a[i], blockIdx.x - g.start[i], g.gx[i]);
}
// LDS bytes of a k_tile_w workgroup
template <int D, int MODE>
inline size_t tile_w_lds_bytes(int EB) {
  return sizeof(float) * (size_t)(((2 * EB * EB + 3) & ~3) + 2 * WAVE) +
         (D == 64 ? 64 * sizeof(double2) : 0) +
         (MODE == TILE_GRAD ? sizeof(float2) * (size_t)16 * WAVE : 0) +
         sizeof(float) * (size_t)kTileW * WaveFrame<D>::kBuf;
}
// whether a handle's frames run one wave per frame (WaveFrame)
inline bool wave_frames(const pt_ptycho* h) {
  return h->D == 32 || (h->D == 64 && h->P <= 16);
}

// LDS bytes of a k_tile workgroup
inline size_t tile_lds_bytes(int D, int EB) {
  const int W = 1, G = 64 / D;
  return sizeof(float2) * (size_t)EB * EB + sizeof(float) * (size_t)W * G * D * (D + 1);
}

// Arguments of one fold launch (one instance of a group)
struct FoldArgs {
  float2* out;
  const float2* scratch;
  const int* tile_slot;
  const float2* psi;
  const float2* hh;
  const float2* lamd;
  const double* rho_dev;
  float rhov;
  int pt, nz, n, nty, ntx, B, EB;
};

template <int MODE>
__device__ __forceinline__ void fold_body(const FoldArgs& A, long blk) {
  float2* __restrict__ out = A.out;
  const float2* __restrict__ scratch = A.scratch;
  const int* __restrict__ tile_slot = A.tile_slot;
  const float2* __restrict__ psi = A.psi;
  const float2* __restrict__ hh = A.hh;
  const float2* __restrict__ lamd = A.lamd;
  const double* __restrict__ rho_dev = A.rho_dev;
  const float rhov = A.rhov;
  const int pt = A.pt, nz = A.nz, n = A.n, nty = A.nty, ntx = A.ntx, B = A.B, EB = A.EB;
  const long idx = blk * blockDim.x + threadIdx.x;
  const long total = (long)pt * nz * n;
  if (idx >= total) return;
  const int x = (int)(idx % n);
  const long tz = idx / n;
  const int y = (int)(tz % nz);
  const int t = (int)(tz / nz);
  float2 s = make_float2(0.f, 0.f);
  // tiles whose extended region [t*B, t*B + EB) contains the pixel, in
  // ascending order (fixed summation order)
  const int ylo = y - EB + 1, xlo = x - EB + 1;
  const int ty0 = ylo <= 0 ? 0 : (ylo + B - 1) / B, ty1 = min(y / B, nty - 1);
  const int tx0 = xlo <= 0 ? 0 : (xlo + B - 1) / B, tx1 = min(x / B, ntx - 1);
  for (int ty = ty0; ty <= ty1; ++ty) {
    const int ly = y - ty * B;
    for (int tx = tx0; tx <= tx1; ++tx) {
      const int lx = x - tx * B;
      const int sl = tile_slot[((long)t * nty + ty) * ntx + tx];
      if (sl < 0) continue;
      s = cadd(s, scratch[(long)sl * EB * EB + ly * EB + lx]);
    }
  }
  if constexpr (MODE == TILE_GRAD) {
    // grad -= rho*(h - psi + lamd/rho)   (solver.py:225)
    const float rho = rho_dev ? (float)rho_dev[0] : rhov;
    const float2 h = hh[idx], p = psi[idx], l = lamd[idx];
    const float ir = 1.0f / rho;
    const float2 q = make_float2(h.x - p.x + l.x * ir, h.y - p.y + l.y * ir);
    s = make_float2(s.x - rho * q.x, s.y - rho * q.y);
  }
  out[idx] = s;
}
template <int MODE>
__global__ void k_fold(FoldArgs A) {
  fold_body<MODE>(A, blockIdx.x);
}
template <int MODE>
__global__ void k_fold_group(Group<FoldArgs> g) {
  const int i = group_find(g, blockIdx.x);
  fold_body<MODE>(g.a[i], blockIdx.x - g.start[i]);
}

// ------------------------------------------------------------------ set-up kernels
__global__ void k_setup_pos(int2* __restrict__ pos, float2* __restrict__ shift,
                            const float* __restrict__ scan, long np) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float sx = scan[i], sy = scan[np + i];
  const float rx = roundf(sx), ry = roundf(sy);
  // a negative rounded coordinate marks the patch as skipped (x = -1), in y too:
  // the kernels test x
  pos[i] = rx < 0.f || ry < 0.f ? make_int2(-1, -1) : make_int2((int)rx, (int)ry);
  // takeshifts (kernels.cuh:306-317): e^{2 pi i frac(x)} * e^{2 pi i frac(y)}
  double ax = 2.0 * kPi * (double)(sx - rx), ay = 2.0 * kPi * (double)(sy - ry);
  double cx = cos(ax), sxn = sin(ax), cy = cos(ay), syn = sin(ay);
  float2 a = make_float2((float)cx, (float)sxn), b = make_float2((float)cy, (float)syn);
  shift[i] = cmul(a, b);
}

int launch_blocks(long work, int per_block, int cap) {
  long b = (work + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return (int)b;
}

template <int D, bool INT>
int run_fwd(pt_ptycho* h, float2* g, float* out, const float2* f, float scale, float isc,
            hipStream_t st) {
  constexpr int G = WAVE / D;
  const long np = (long)h->pt * h->S;
  ProfScope prof("ptycho_fwd", st);
  if constexpr (D >= 32) {
    if (wave_frames(h)) {
      const int nw = (int)std::min<long>(4, 1 + (np - 1) / (kMinfWWaves * kFwdWBlocks));
      const int nb = launch_blocks(np, nw * kMinfWWaves, 1 << 20);
      hipLaunchKernelGGL((k_fwd_wave<D, INT>), dim3(nb), dim3(WAVE * kMinfWWaves), 0, st, g, out, f,
                         h->prb, h->pos, h->shift, np,
                         h->nz, h->n, h->S, h->P, h->ox, h->c * scale, isc);
      PT_LAUNCH_CHECK();
      return PT_OK;
    }
  }
  if constexpr (D != 32)
    hipLaunchKernelGGL((k_fwd<D, INT>), dim3(launch_blocks(np, G, 1 << 20)), dim3(WAVE), 0, st, g,
                       out, f, h->prb, h->pos, h->shift, h->pt, h->nz, h->n, h->S, h->P, h->ox,
                       h->oy, h->c * scale, isc);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// the probe covers the frame (no offset): the FULL kernels
template <int D>
inline bool minf_full(const pt_ptycho* h) {
  return h->P == D && h->ox == 0 && h->oy == 0;
}
// fn(k_tile<...>, k_tile_group<...>) for the model and probe form (frames of 64
// x 64 come here with a probe beyond 16 pixels, rarely the whole frame: one form)
template <int D, int MODE, class F>
inline void tile_dispatch(int model, bool full, F&& fn) {
  auto by_full = [&](auto model_c) {
    constexpr int M = decltype(model_c)::value;
    if constexpr (D <= 16) {
      if (full) {
        fn(k_tile<D, MODE, M, true>, k_tile_group<D, MODE, M, true>);
        return;
      }
    }
    fn(k_tile<D, MODE, M, false>, k_tile_group<D, MODE, M, false>);
  };
  if constexpr (MODE == TILE_ADJ) by_full(std::integral_constant<int, PT_MODEL_POISSON>());
  else if (model == PT_MODEL_POISSON) by_full(std::integral_constant<int, PT_MODEL_POISSON>());
  else by_full(std::integral_constant<int, PT_MODEL_GAUSSIAN>());
}

inline TileArgs tile_args(const pt_ptycho* h, const float2* gin, const float2* f, const float* data,
                          float cp, float cd, float out_scale) {
  TileArgs A;
  A.scratch = h->scratch; A.gin = gin; A.f = f; A.data = data; A.prb = h->prb; A.pos = h->pos;
  A.shift = h->shift; A.tile_start = h->tile_start; A.tile_patch = h->tile_patch;
  A.tile_slot = h->tile_slot; A.nty = h->nty; A.ntx = h->ntx; A.B = h->B; A.EB = h->EB;
  A.nz = h->nz; A.n = h->n; A.S = h->S; A.P = h->P; A.ox = h->ox; A.oy = h->oy;
  A.cs = h->c; A.cp = cp; A.cd = cd; A.out_scale = out_scale;
  return A;
}

template <int D, int MODE>
int run_tiles(pt_ptycho* h, const float2* gin, const float2* f, const float* data, float cp,
              float cd, float out_scale, int model, hipStream_t st) {
  const TileArgs A = tile_args(h, gin, f, data, cp, cd, out_scale);
  ProfScope prof(MODE == TILE_GRAD ? "ptycho_grad_tile" : "ptycho_adj_tile", st);
  if constexpr (D >= 32) {
    if (wave_frames(h)) {
      auto kern = MODE == TILE_ADJ || model == PT_MODEL_POISSON
                      ? k_tile_w<D, MODE, PT_MODEL_POISSON>
                      : k_tile_w<D, MODE, MODE == TILE_ADJ ? PT_MODEL_POISSON : PT_MODEL_GAUSSIAN>;
      const size_t lds = tile_w_lds_bytes<D, MODE>(h->EB);
      hipLaunchKernelGGL(kern, dim3((unsigned)h->ntiles), dim3(WAVE * kTileW), lds, st, A);
      PT_LAUNCH_CHECK();
      return PT_OK;
    }
  }
  if constexpr (D != 32)
    tile_dispatch<D, MODE>(model, minf_full<D>(h), [&](auto kern, auto) {
      hipLaunchKernelGGL(kern, dim3((unsigned)h->ntiles), dim3(WAVE * tile_waves<D>()),
                         tile_lds_bytes(D, h->EB), st, A);
    });
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// Partial-sum buffer of a line-search launch: the handle's buffer, grown on
// demand, or (fixed != nullptr) a caller-provided fixed buffer of fixed_cap
// doubles that is never reallocated.
inline int minf_partials(pt_ptycho* h, size_t need, double* fixed, size_t fixed_cap,
                         double** out) {
  if (fixed) {
    PT_REQUIRE(need <= fixed_cap, PT_ERR_SIZE,
               "pt_ptycho_minf_noalloc: " + std::to_string(need) + " partial sums (on overlap-add "
                   "tiles counted as one per wave, tile and candidate) exceed the fixed buffer's " +
                   std::to_string(fixed_cap) + " (fewer angles per call, or pt_ptycho_minf)");
    *out = fixed;
    return PT_OK;
  }
  if (need > h->partial_cap) {
    if (h->partial) PT_HIP(hipFree(h->partial));
    h->partial = nullptr;
    PT_HIP(hipMalloc(&h->partial, need * sizeof(double)));
    h->partial_cap = need;
  }
  *out = h->partial;
  return PT_OK;
}

// Optional rho term of the line search (pt_ptycho_linesearch): sums of the
// change of |h - (psi + g*d) + lamd/rho|^2 per chunk into f2.
struct RhoTerm {
  const float2* hh = nullptr;
  const float2* lamd = nullptr;
  double rho = 0.0;
  const double* rho_dev = nullptr;
  double* f2 = nullptr;
  LsFinishArgs* fin = nullptr;  // set: finish the sweep with k_ls_finish instead of sums and f2
};

// whether a line search of this handle runs on the overlap-add tiles: frames
// up to 16 x 16 whose extended tile fits the staging, where a tile holds on
// average at least one patch per slot of its workgroup (sparser tiles would
// leave lanes idle); otherwise each patch reads its frame rows directly
// (32 x 32 frames: 63 x 63 extended tiles)
template <int D>
inline bool minf_tile_path(const pt_ptycho* h) {
  constexpr int G = WAVE / D;
  if constexpr (D > 16) return false;
  const bool dense = (long)h->S >= (long)kMinfWaves * G * h->nty * h->ntx;
  return dense && minf_tile_lds_bytes(D, h->EB, h->P) <= 64 * 1024 &&
         h->EB * h->EB <= WAVE * kMinfWaves * kMinfStage;
}
inline int minf_tile_gx(const pt_ptycho* h, int chunk) {
  return (chunk * h->nty * h->ntx + kMinfTiles - 1) / kMinfTiles;
}
inline MinfTileArgs minf_tile_args(const pt_ptycho* h, double* part, double* part_rho,
                                   const float2* f, const float2* dir, const float* data,
                                   const double* gammas, int ngam, int chunk, float cp, float cd,
                                   const double* skip, const RhoTerm& rt) {
  MinfTileArgs A;
  A.partial = part; A.f = f; A.dir = dir; A.data = data; A.prb = h->prb; A.pos = h->pos;
  A.tile_start = h->tile_start; A.tile_patch = h->tile_patch; A.gammas = gammas; A.skip = skip;
  A.hh = rt.hh; A.lamd = rt.lamd; A.rho_dev = rt.rho_dev; A.partial_rho = part_rho;
  A.rho_host = rt.rho; A.ngam = ngam; A.chunk = chunk; A.nty = h->nty; A.ntx = h->ntx;
  A.B = h->B; A.EB = h->EB; A.nz = h->nz; A.n = h->n; A.P = h->P; A.ox = h->ox; A.oy = h->oy;
  A.cs = h->c; A.cp = cp; A.cd = cd;
  return A;
}
// fn(k_minf_tile<...>, k_minf_tile_group<...>) for the model, probe form
// and candidate count: the accumulator count is a template argument
// (registers): 3, 5 and 6 slots cover the solver's sweeps (gamma = 0 and 1,
// 2, 4 or 5 halvings), 8 any other ngam
template <int D, class F>
inline void minf_dispatch(int model, bool full, int ngam, F&& fn) {
  auto by_ng = [&](auto model_c, auto full_c) {
    constexpr int M = decltype(model_c)::value;
    constexpr bool FU = decltype(full_c)::value;
    if (ngam <= 3) fn(k_minf_tile<D, M, 3, FU>, k_minf_tile_group<D, M, 3, FU>);
    else if (ngam <= 5) fn(k_minf_tile<D, M, 5, FU>, k_minf_tile_group<D, M, 5, FU>);
    else if (ngam <= 6) fn(k_minf_tile<D, M, 6, FU>, k_minf_tile_group<D, M, 6, FU>);
    else fn(k_minf_tile<D, M, PT_MAX_GAM, FU>, k_minf_tile_group<D, M, PT_MAX_GAM, FU>);
  };
  using Poi = std::integral_constant<int, PT_MODEL_POISSON>;
  using Gau = std::integral_constant<int, PT_MODEL_GAUSSIAN>;
  if (model == PT_MODEL_POISSON) {
    if (full) by_ng(Poi(), std::true_type());
    else by_ng(Poi(), std::false_type());
  } else {
    if (full) by_ng(Gau(), std::true_type());
    else by_ng(Gau(), std::false_type());
  }
}

// the partials of a line search on tiles, as k_ls_finish reads them
inline void ls_tile_partials(LsFinishArgs* F, const double* part, const double* part_rho, int nbt) {
  for (int t = 0; t < 2; ++t) {
    F->p[t] = t ? part_rho : part;
    F->cs[t] = (long)F->ngam * nbt; F->js[t] = nbt; F->bs[t] = 1; F->nb[t] = nbt;
  }
}

template <int D>
int run_minf(pt_ptycho* h, double* sums, const float2* f, const float2* dir, const float* data,
             const double* gammas, int ngam, int chunk, float cp, float cd, int model, int lagr,
             const double* skip, hipStream_t st, double* fixed, size_t fixed_cap,
             const RhoTerm& rt = RhoTerm()) {
  constexpr int G = WAVE / D;
  const int nchunk = h->pt / chunk;
  // line-search sums over the overlap-add tiles (frames read from LDS)
  const size_t tl = minf_tile_lds_bytes(D, h->EB, h->P);
  if constexpr (D <= 16) if (!lagr && dir && minf_tile_path<D>(h)) {
    const int nbt = minf_tile_gx(h, chunk);
    const size_t nper = (size_t)nchunk * nbt * ngam;
    // a fixed buffer's limit counts one partial per wave and tile, as the interface
    // states it (the kernel writes one per workgroup)
    const size_t need = fixed ? (size_t)nchunk * chunk * h->nty * h->ntx * kMinfWaves * ngam : nper;
    double* part;
    int rc = minf_partials(h, rt.hh ? 2 * need : need, fixed, fixed_cap, &part);
    if (rc) return rc;
    double* part_rho = rt.hh ? part + nper : nullptr;
    {
      ProfScope prof("ptycho_minf", st);
      const MinfTileArgs A = minf_tile_args(h, part, part_rho, f, dir, data, gammas, ngam, chunk,
                                            cp, cd, skip, rt);
      minf_dispatch<D>(model, minf_full<D>(h), ngam, [&](auto kern, auto) {
        hipLaunchKernelGGL(kern, dim3(nbt, nchunk), dim3(WAVE * kMinfWaves), tl, st, A);
      });
    }
    PT_LAUNCH_CHECK();
    if (rt.fin) {
      ls_tile_partials(rt.fin, part, part_rho, nbt);
      hipLaunchKernelGGL(k_ls_finish, dim3(nchunk), dim3(1024), 0, st, *rt.fin);
      PT_LAUNCH_CHECK();
      return PT_OK;
    }
    hipLaunchKernelGGL(k_reduce_partials_t, dim3(nchunk, ngam), dim3(256), 0, st, sums, part,
                       (long)nbt, ngam, skip);
    PT_LAUNCH_CHECK();
    if (rt.hh) {
      hipLaunchKernelGGL(k_reduce_partials_t, dim3(nchunk, ngam), dim3(256), 0, st, rt.f2,
                         part_rho, (long)nbt, ngam, skip);
      PT_LAUNCH_CHECK();
    }
    return PT_OK;
  }
  long np = (long)chunk * h->S;
  int nb = launch_blocks(np, 4 * G, std::max(1, 20480 / nchunk));
  bool wave = false;
  if constexpr (D >= 32) {
    wave = wave_frames(h) && !lagr && dir;
    if (wave) nb = std::max(1, nb / kMinfWWaves);
  }
  double* part;
  int rc = minf_partials(h, (size_t)nchunk * nb * ngam, fixed, fixed_cap, &part);
  if (rc) return rc;
  {
  ProfScope prof(lagr ? "ptycho_lagr" : "ptycho_minf", st);
  if constexpr (D >= 32) {
    if (wave) {
      auto kern = model == PT_MODEL_POISSON ? k_minf_wave<D, PT_MODEL_POISSON>
                                            : k_minf_wave<D, PT_MODEL_GAUSSIAN>;
      hipLaunchKernelGGL(kern, dim3(nb, nchunk), dim3(WAVE * kMinfWWaves), 0, st, part, f, dir,
                         data, h->prb, h->pos, gammas, ngam, chunk, h->nz, h->n, h->S, h->P,
                         h->ox, h->c * cp, cd, skip);
    }
  }
  if (wave) {
  } else if (model == PT_MODEL_POISSON)
    hipLaunchKernelGGL((k_minf<D, PT_MODEL_POISSON>), dim3(nb, nchunk), dim3(WAVE), 0, st,
                       part, f, dir, data, h->prb, h->pos, gammas, ngam, chunk, h->nz, h->n,
                       h->S, h->P, h->ox, h->oy, h->c, cp, cd, model, lagr, skip);
  else
    hipLaunchKernelGGL((k_minf<D, PT_MODEL_GAUSSIAN>), dim3(nb, nchunk), dim3(WAVE), 0, st,
                       part, f, dir, data, h->prb, h->pos, gammas, ngam, chunk, h->nz, h->n,
                       h->S, h->P, h->ox, h->oy, h->c, cp, cd, model, lagr, skip);
  }
  PT_LAUNCH_CHECK();
  if (rt.fin) {
    LsFinishArgs& F = *rt.fin;
    double* pr;
    int nbr;
    rc = rho_minf_partials(&pr, &nbr, rt.hh, f, rt.lamd, dir, rt.rho, rt.rho_dev, gammas, ngam,
                           (long)h->pt * h->nz * h->n, nchunk, skip, st);
    if (rc) return rc;
    F.p[0] = part; F.cs[0] = (long)nb * ngam; F.js[0] = 1; F.bs[0] = ngam; F.nb[0] = nb;
    F.p[1] = pr; F.cs[1] = (long)nbr * 8; F.js[1] = 1; F.bs[1] = 8; F.nb[1] = nbr;
    hipLaunchKernelGGL(k_ls_finish, dim3(nchunk), dim3(1024), 0, st, F);
    PT_LAUNCH_CHECK();
    return PT_OK;
  }
  hipLaunchKernelGGL(k_reduce_partials, dim3(nchunk, ngam), dim3(64), 0, st, sums, part, nb,
                     ngam, skip);
  PT_LAUNCH_CHECK();
  if (rt.hh)   // per-patch kernel: the rho term as its own fused pass
    return pt_k_rho_minf(rt.f2, rt.hh, f, rt.lamd, dir, rt.rho, rt.rho_dev, gammas, ngam,
                         (long)h->pt * h->nz * h->n, nchunk, skip, (pt_stream)st);
  return PT_OK;
}

inline FoldArgs fold_args(const pt_ptycho* h, float2* out, const float2* psi, const float2* hh,
                          const float2* lamd, float rho, const double* rho_dev) {
  FoldArgs A;
  A.out = out; A.scratch = h->scratch; A.tile_slot = h->tile_slot; A.psi = psi; A.hh = hh;
  A.lamd = lamd; A.rho_dev = rho_dev; A.rhov = rho; A.pt = h->pt; A.nz = h->nz; A.n = h->n;
  A.nty = h->nty; A.ntx = h->ntx; A.B = h->B; A.EB = h->EB;
  return A;
}
inline int fold_blocks(const pt_ptycho* h) {
  return (int)(((long)h->pt * h->nz * h->n + 255) / 256);
}

template <int MODE>
int run_fold(pt_ptycho* h, float2* out, const float2* psi, const float2* hh, const float2* lamd,
             float rho, const double* rho_dev, hipStream_t st) {
  ProfScope prof("ptycho_fold", st);
  hipLaunchKernelGGL(k_fold<MODE>, dim3(fold_blocks(h)), dim3(256), 0, st,
                     fold_args(h, out, psi, hh, lamd, rho, rho_dev));
  PT_LAUNCH_CHECK();
  return PT_OK;
}

#define PT_DISPATCH_D(D, CALL)                         \
  switch (D) {                                         \
    case 8: { constexpr int DD = 8; return CALL; }     \
    case 16: { constexpr int DD = 16; return CALL; }   \
    case 32: { constexpr int DD = 32; return CALL; }   \
    case 64: { constexpr int DD = 64; return CALL; }   \
    default: set_error("unsupported detector size"); return PT_ERR_SIZE; \
  }

int fwd_impl(pt_ptycho* h, void* g, const void* f, float scale, pt_stream stream) {
  PT_REQUIRE(h && g && f, PT_ERR_ARG, "pt_ptycho_fwd: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_fwd: set_scan_probe not called");
  hipStream_t st = (hipStream_t)stream;
  PT_DISPATCH_D(h->D, (run_fwd<DD, false>(h, (float2*)g, nullptr, (const float2*)f, scale, 0.f, st)));
}

template <int MODE>
int tiles_impl(pt_ptycho* h, float2* out, const float2* gin, const float2* f, const float* data,
               const float2* hh, const float2* lamd, double rho, const double* rho_dev, float cp,
               float cd, float out_scale, int model, hipStream_t st) {
  int rc;
  switch (h->D) {
    case 8: rc = run_tiles<8, MODE>(h, gin, f, data, cp, cd, out_scale, model, st); break;
    case 16: rc = run_tiles<16, MODE>(h, gin, f, data, cp, cd, out_scale, model, st); break;
    case 32: rc = run_tiles<32, MODE>(h, gin, f, data, cp, cd, out_scale, model, st); break;
    case 64: rc = run_tiles<64, MODE>(h, gin, f, data, cp, cd, out_scale, model, st); break;
    default: set_error("unsupported detector size"); return PT_ERR_SIZE;
  }
  if (rc) return rc;
  return run_fold<MODE>(h, out, f, hh, lamd, (float)rho, rho_dev, st);
}

// The extended tile takes what a workgroup of one wave (k_tile) leaves of this after
// its transpose buffers.  12 KB for frames up to 16 x 16 (13 resident per CU; a 16 x
// 16 probe gets 16 x 16 pixel tiles, extended to 31 x 31).  40 KB for larger frames:
// a 32 x 32 probe gets 32 x 32 pixel tiles extended to 63 x 63, where in 12 KB the
// tiles would shrink to 8 pixels -- one patch per tile at step 8 and ~25 overlapping
// tiles summed per pixel by the fold.  One wave per frame (k_tile_w) keeps these tiles
// and adds the buffers of its four waves and the staged probe: 57 KB for the gradient
// of 32 x 32 frames, 51 KB for 64 x 64 ones with a 16 x 16 probe, two workgroups per CU.
constexpr size_t kTileLdsBudget = 12 * 1024;
constexpr size_t kTileLdsBudgetLarge = 40 * 1024;

}  // namespace
}  // namespace pt

using namespace pt;

extern "C" int pt_ptycho_create(int ptheta, int nz, int n, int ntheta0, int nscan, int detx,
                                int dety, int nprb, pt_ptycho** out) {
  (void)ntheta0;
  PT_REQUIRE(out, PT_ERR_ARG, "pt_ptycho_create: null output handle");
  *out = nullptr;
  PT_REQUIRE(ptheta > 0 && nz > 0 && n > 0 && nscan > 0 && nprb > 0, PT_ERR_SIZE,
             "pt_ptycho_create: sizes must be positive");
  PT_REQUIRE(detx == dety, PT_ERR_SIZE, "pt_ptycho_create: detx must equal dety");
  PT_REQUIRE(detx == 8 || detx == 16 || detx == 32 || detx == 64, PT_ERR_SIZE,
             "pt_ptycho_create: detector size must be 8, 16, 32 or 64");
  PT_REQUIRE(nprb <= detx && nprb <= n && nprb <= nz, PT_ERR_SIZE,
             "pt_ptycho_create: probe larger than detector or object");
  pt_ptycho* h = new pt_ptycho();
  h->pt = ptheta; h->nz = nz; h->n = n; h->S = nscan; h->D = detx; h->P = nprb;
  h->ox = (detx - nprb) / 2;
  h->oy = (dety - nprb) / 2;
  h->c = 1.0f / sqrtf((float)(detx * dety));
  // tile size from the LDS budget: the extended tile takes what the
  // transpose buffers leave, and at least P+7 pixels
  const size_t tbytes = tile_lds_bytes(detx, 0);
  const size_t budget = detx >= 32 ? kTileLdsBudgetLarge : kTileLdsBudget;
  const size_t left = budget > tbytes + 4096 ? budget - tbytes : 4096;
  const long maxe = (long)std::sqrt((double)left / sizeof(float2));
  int EB = (int)std::max<long>(maxe, nprb + 7);
  int B = EB - (nprb - 1);
  h->B = B; h->EB = EB;
  h->ntx = (n - nprb) / B + 1;
  h->nty = (nz - nprb) / B + 1;
  h->ntiles = (long)ptheta * h->ntx * h->nty;
  long np = (long)ptheta * nscan;
  auto fail = [&](hipError_t e, const char* what) {
    set_error(std::string("pt_ptycho_create: ") + what + ": " + hipGetErrorString(e));
    pt_ptycho_destroy(h);
    return PT_ERR_HIP;
  };
  hipError_t e;
  if ((e = hipMalloc(&h->prb, sizeof(float2) * nprb * nprb))) return fail(e, "prb");
  if ((e = hipMalloc(&h->pos, sizeof(int2) * np))) return fail(e, "pos");
  if ((e = hipMalloc(&h->shift, sizeof(float2) * np))) return fail(e, "shift");
  if ((e = hipMalloc(&h->tile_start, sizeof(int) * (h->ntiles + 1)))) return fail(e, "tiles");
  if ((e = hipMalloc(&h->tile_patch, sizeof(int) * std::max<long>(np, 1)))) return fail(e, "tiles");
  if ((e = hipMalloc(&h->tile_slot, sizeof(int) * h->ntiles))) return fail(e, "tiles");
  *out = h;
  return PT_OK;
}

extern "C" int pt_ptycho_destroy(pt_ptycho* h) {
  if (!h) return PT_OK;
  (void)hipFree(h->prb);
  (void)hipFree(h->pos);
  (void)hipFree(h->shift);
  (void)hipFree(h->tile_start);
  (void)hipFree(h->tile_patch);
  (void)hipFree(h->tile_slot);
  (void)hipFree(h->scratch);
  (void)hipFree(h->partial);
  delete h;
  return PT_OK;
}

extern "C" int pt_ptycho_set_scan_probe(pt_ptycho* h, const float* scan, const void* prb,
                                        pt_stream stream) {
  PT_REQUIRE(h && scan && prb, PT_ERR_ARG, "pt_ptycho_set_scan_probe: null argument");
  hipStream_t st = (hipStream_t)stream;
  const long np = (long)h->pt * h->S;
  PT_HIP(hipMemcpyAsync(h->prb, prb, sizeof(float2) * h->P * h->P, hipMemcpyDeviceToDevice, st));
  int nb = (int)((np + 255) / 256);
  hipLaunchKernelGGL(k_setup_pos, dim3(nb), dim3(256), 0, st, h->pos, h->shift, scan, np);
  PT_LAUNCH_CHECK();
  // bin valid patches by tile (host; geometry is static between calls)
  std::vector<int2> pos(np);
  PT_HIP(hipMemcpyAsync(pos.data(), h->pos, sizeof(int2) * np, hipMemcpyDeviceToHost, st));
  PT_HIP(hipStreamSynchronize(st));
  std::vector<int> cnt(h->ntiles + 1, 0);
  for (long i = 0; i < np; ++i) {
    const int2 p = pos[i];
    if (p.x < 0 || p.y < 0) continue;
    if (p.x > h->n - h->P || p.y > h->nz - h->P) {
      set_error("pt_ptycho_set_scan_probe: scan position places the probe outside the object");
      h->ready = false;
      return PT_ERR_ARG;
    }
    const long t = i / h->S;
    const long tile = (t * h->nty + p.y / h->B) * h->ntx + p.x / h->B;
    cnt[tile + 1]++;
  }
  for (long i = 0; i < h->ntiles; ++i) cnt[i + 1] += cnt[i];
  std::vector<int> fillp(cnt.begin(), cnt.end() - 1);
  std::vector<int> list(std::max<long>(cnt[h->ntiles], 1));
  for (long i = 0; i < np; ++i) {
    const int2 p = pos[i];
    if (p.x < 0 || p.y < 0) continue;
    const long t = i / h->S;
    const long tile = (t * h->nty + p.y / h->B) * h->ntx + p.x / h->B;
    list[fillp[tile]++] = (int)i;
  }
  std::vector<int> slot(h->ntiles, -1);
  long ns = 0;
  for (long i = 0; i < h->ntiles; ++i)
    if (cnt[i + 1] > cnt[i]) slot[i] = (int)ns++;
  h->nslots = ns;
  size_t need = (size_t)std::max<long>(ns, 1) * h->EB * h->EB;
  if (need > h->scratch_cap) {
    if (h->scratch) PT_HIP(hipFree(h->scratch));
    h->scratch = nullptr;
    PT_HIP(hipMalloc(&h->scratch, need * sizeof(float2)));
    h->scratch_cap = need;
  }
  PT_HIP(hipMemcpyAsync(h->tile_start, cnt.data(), sizeof(int) * (h->ntiles + 1),
                        hipMemcpyHostToDevice, st));
  PT_HIP(hipMemcpyAsync(h->tile_patch, list.data(), sizeof(int) * list.size(),
                        hipMemcpyHostToDevice, st));
  PT_HIP(hipMemcpyAsync(h->tile_slot, slot.data(), sizeof(int) * h->ntiles,
                        hipMemcpyHostToDevice, st));
  PT_HIP(hipStreamSynchronize(st));
  h->ready = true;
  return PT_OK;
}

extern "C" int pt_ptycho_fwd(pt_ptycho* h, void* g, const void* f, pt_stream stream) {
  return fwd_impl(h, g, f, 1.0f, stream);
}
extern "C" int pt_ptycho_fwd_scaled(pt_ptycho* h, void* g, const void* f, float scale,
                                    pt_stream stream) {
  return fwd_impl(h, g, f, scale, stream);
}

extern "C" int pt_ptycho_intensity(pt_ptycho* h, float* out, const void* f, float scale,
                                   float iscale, pt_stream stream) {
  PT_REQUIRE(h && out && f, PT_ERR_ARG, "pt_ptycho_intensity: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_intensity: set_scan_probe not called");
  hipStream_t st = (hipStream_t)stream;
  PT_DISPATCH_D(h->D, (run_fwd<DD, true>(h, nullptr, out, (const float2*)f, scale, iscale, st)));
}

static int adj_impl(pt_ptycho* h, void* f, const void* g, float scale, pt_stream stream) {
  PT_REQUIRE(h && g && f, PT_ERR_ARG, "pt_ptycho_adj: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_adj: set_scan_probe not called");
  return tiles_impl<TILE_ADJ>(h, (float2*)f, (const float2*)g, nullptr, nullptr, nullptr,
                              nullptr, 0.0, nullptr, 1.0f, 1.0f, h->c * scale, 0,
                              (hipStream_t)stream);
}
extern "C" int pt_ptycho_adj(pt_ptycho* h, void* f, const void* g, pt_stream stream) {
  return adj_impl(h, f, g, 1.0f, stream);
}
extern "C" int pt_ptycho_adj_scaled(pt_ptycho* h, void* f, const void* g, float scale,
                                    pt_stream stream) {
  return adj_impl(h, f, g, scale, stream);
}

extern "C" int pt_ptycho_grad(pt_ptycho* h, void* grad, const void* psi, const float* data,
                              const void* hh, const void* lamd, double rho, const double* rho_dev,
                              float coefptycho, float coefdata, int model, pt_stream stream) {
  PT_REQUIRE(h && grad && psi && data && hh && lamd, PT_ERR_ARG, "pt_ptycho_grad: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_grad: set_scan_probe not called");
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             "pt_ptycho_grad: bad model");
  PT_REQUIRE(rho_dev || rho > 0, PT_ERR_ARG, "pt_ptycho_grad: rho must be positive");
  return tiles_impl<TILE_GRAD>(h, (float2*)grad, nullptr, (const float2*)psi, data,
                               (const float2*)hh, (const float2*)lamd, rho, rho_dev, coefptycho,
                               coefdata,
                               h->c * coefptycho, model, (hipStream_t)stream);
}

// no handle twice in a group call (each launch writes the handle's scratch)
template <class A>
static bool distinct_handles(const A* a, int n) {
  std::vector<const pt_ptycho*> hs;
  for (int i = 0; i < n; ++i) hs.push_back(a[i].h);
  std::sort(hs.begin(), hs.end());
  return std::adjacent_find(hs.begin(), hs.end()) == hs.end();
}

// One k_tile_group and one k_fold_group launch (the gradient of
// pt_ptycho_grad) for the instances idx (at most kGroupMax, detector D, all or
// none with one wave per frame, all or none with a probe that covers the frame)
template <int D, bool WF>
static int run_grad_group(const pt_ptycho_grad_args* a, const int* idx, int n, int model,
                          bool full, hipStream_t st) {
  Group<TileArgs> g;
  Group<FoldArgs> fg;
  size_t lds = 0;
  int tot = 0, totf = 0;
  for (int k = 0; k < n; ++k) {
    const pt_ptycho_grad_args& x = a[idx[k]];
    const pt_ptycho* h = x.h;
    g.a[k] = tile_args(h, nullptr, (const float2*)x.psi, x.data, x.coefptycho, x.coefdata,
                       h->c * x.coefptycho);
    g.gx[k] = h->ntiles;
    g.start[k] = tot;
    tot += h->ntiles;
    fg.a[k] = fold_args(h, (float2*)x.grad, (const float2*)x.psi, (const float2*)x.hh,
                        (const float2*)x.lamd, (float)x.rho, x.rho_dev);
    fg.gx[k] = fold_blocks(h);
    fg.start[k] = totf;
    totf += fg.gx[k];
    if constexpr (WF) lds = std::max(lds, tile_w_lds_bytes<D, TILE_GRAD>(h->EB));
    else lds = std::max(lds, tile_lds_bytes(D, h->EB));
  }
  g.start[n] = tot;
  fg.start[n] = totf;
  g.n = fg.n = n;
  {
    ProfScope prof("ptycho_grad_tile", st);
    if constexpr (WF) {
      auto kern = model == PT_MODEL_POISSON ? k_tile_w_group<D, TILE_GRAD, PT_MODEL_POISSON>
                                            : k_tile_w_group<D, TILE_GRAD, PT_MODEL_GAUSSIAN>;
      hipLaunchKernelGGL(kern, dim3(tot), dim3(WAVE * kTileW), lds, st, g);
    } else {
      tile_dispatch<D, TILE_GRAD>(model, full, [&](auto, auto kern) {
        hipLaunchKernelGGL(kern, dim3(tot), dim3(WAVE * tile_waves<D>()), lds, st, g);
      });
    }
  }
  PT_LAUNCH_CHECK();
  {
    ProfScope prof("ptycho_fold", st);
    hipLaunchKernelGGL(k_fold_group<TILE_GRAD>, dim3(totf), dim3(256), 0, st, fg);
  }
  PT_LAUNCH_CHECK();
  return PT_OK;
}

extern "C" int pt_ptycho_grad_group(const pt_ptycho_grad_args* a, int n, int model,
                                    pt_stream stream) {
  PT_REQUIRE(n >= 0 && (a || n == 0), PT_ERR_ARG, "pt_ptycho_grad_group: bad argument");
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             "pt_ptycho_grad_group: bad model");
  // D = 8 and 16 (probe partial / full), 32, 64 (one wave per frame), 64
  std::vector<int> bins[7];
  for (int i = 0; i < n; ++i) {
    const pt_ptycho_grad_args& x = a[i];
    PT_REQUIRE(x.h && x.grad && x.psi && x.data && x.hh && x.lamd, PT_ERR_ARG,
               "pt_ptycho_grad_group: null argument in instance " + std::to_string(i));
    PT_REQUIRE(x.h->ready, PT_ERR_STATE,
               "pt_ptycho_grad_group: set_scan_probe not called for instance " +
                   std::to_string(i));
    PT_REQUIRE(x.rho_dev || x.rho > 0, PT_ERR_ARG,
               "pt_ptycho_grad_group: rho must be positive (instance " + std::to_string(i) + ")");
    const int D = x.h->D;
    const int b = D == 8    ? (minf_full<8>(x.h) ? 1 : 0)
                  : D == 16 ? 2 + (minf_full<16>(x.h) ? 1 : 0)
                  : D == 32 ? 4
                            : wave_frames(x.h) ? 5 : 6;
    bins[b].push_back(i);
  }
  PT_REQUIRE(distinct_handles(a, n), PT_ERR_ARG,
             "pt_ptycho_grad_group: a handle appears twice (its tile scratch would be shared)");
  hipStream_t st = (hipStream_t)stream;
  for (int b = 0; b < 7; ++b) {
    for (size_t k0 = 0; k0 < bins[b].size(); k0 += kGroupMax) {
      const int m = (int)std::min<size_t>(kGroupMax, bins[b].size() - k0);
      const int* idx = bins[b].data() + k0;
      int rc;
      switch (b) {
        case 0:
        case 1: rc = run_grad_group<8, false>(a, idx, m, model, b == 1, st); break;
        case 2:
        case 3: rc = run_grad_group<16, false>(a, idx, m, model, b == 3, st); break;
        case 4: rc = run_grad_group<32, true>(a, idx, m, model, false, st); break;
        case 5: rc = run_grad_group<64, true>(a, idx, m, model, false, st); break;
        default: rc = run_grad_group<64, false>(a, idx, m, model, false, st); break;
      }
      if (rc) return rc;
    }
  }
  return PT_OK;
}

static int minf_impl(pt_ptycho* h, double* sums, const void* psi, const void* dir,
                     const float* data, const double* gammas, int ngam, int chunk,
                     float coefptycho, float coefdata, int model, int lagr, const double* skip,
                     pt_stream stream, double* fixed, size_t fixed_cap) {
  PT_REQUIRE(h && sums && psi && data && gammas, PT_ERR_ARG, "pt_ptycho_minf: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_minf: set_scan_probe not called");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_GAM, PT_ERR_ARG, "pt_ptycho_minf: 1 <= ngam <= 8");
  PT_REQUIRE(chunk > 0 && h->pt % chunk == 0, PT_ERR_SIZE,
             "pt_ptycho_minf: chunk must divide the number of angles");
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             "pt_ptycho_minf: bad model");
  hipStream_t st = (hipStream_t)stream;
  PT_DISPATCH_D(h->D, (run_minf<DD>(h, sums, (const float2*)psi, (const float2*)dir, data, gammas,
                                     ngam, chunk, coefptycho, coefdata, model, lagr, skip, st,
                                     fixed, fixed_cap)));
}

extern "C" int pt_ptycho_linesearch(pt_ptycho* h, double* f1, double* f2, const void* psi,
                                    const void* dir, const float* data, const void* hh,
                                    const void* lamd, double rho, const double* rho_dev,
                                    const double* gammas, int ngam, int chunk, float coefptycho,
                                    float coefdata, int model, const double* skip,
                                    pt_stream stream) {
  PT_REQUIRE(h && f1 && f2 && psi && dir && data && hh && lamd && gammas, PT_ERR_ARG,
             "pt_ptycho_linesearch: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_ptycho_linesearch: set_scan_probe not called");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_GAM, PT_ERR_ARG, "pt_ptycho_linesearch: 1 <= ngam <= 8");
  PT_REQUIRE(chunk > 0 && h->pt % chunk == 0, PT_ERR_SIZE,
             "pt_ptycho_linesearch: chunk must divide the number of angles");
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             "pt_ptycho_linesearch: bad model");
  PT_REQUIRE(rho_dev || rho > 0, PT_ERR_ARG, "pt_ptycho_linesearch: rho must be positive");
  RhoTerm rt;
  rt.hh = (const float2*)hh;
  rt.lamd = (const float2*)lamd;
  rt.rho = rho;
  rt.rho_dev = rho_dev;
  rt.f2 = f2;
  hipStream_t st = (hipStream_t)stream;
  PT_DISPATCH_D(h->D, (run_minf<DD>(h, f1, (const float2*)psi, (const float2*)dir, data, gammas,
                                     ngam, chunk, coefptycho, coefdata, model, 0, skip, st,
                                     nullptr, 0, rt)));
}

// the sweep's arguments checked (of instance inst of a group, or inst = -1); its
// decision's arguments
static int sweep_args(const pt_ptycho_linesearch_args& a, const pt_ptycho_sweep_args& s, int ngam,
                      int ngam_next, int last, int model, int inst, LsFinishArgs* F) {
  auto err = [&](const char* msg) {
    return inst < 0 ? std::string("pt_ptycho_linesearch_sweep: ") + msg
                    : std::string("pt_ptycho_linesearch_sweep_group: ") + msg + " (instance " +
                          std::to_string(inst) + ")";
  };
  PT_REQUIRE(a.h && a.psi && a.dir && a.data && a.hh && a.lamd && a.gammas && a.skip &&
                 s.cand_next && s.step && s.w,
             PT_ERR_ARG, err("null argument"));
  const pt_ptycho* h = a.h;
  PT_REQUIRE(h->ready, PT_ERR_STATE, err("set_scan_probe not called"));
  PT_REQUIRE(ngam >= 2 && ngam <= PT_MAX_GAM && ngam_next >= 2 && ngam_next <= PT_MAX_GAM,
             PT_ERR_ARG, err("2 <= ngam, ngam_next <= 8"));
  PT_REQUIRE(a.chunk > 0 && h->pt % a.chunk == 0, PT_ERR_SIZE,
             err("chunk must divide the number of angles"));
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             err("bad model"));
  PT_REQUIRE(a.rho_dev || a.rho > 0, PT_ERR_ARG, err("rho must be positive"));
  PT_REQUIRE(s.cand_next != a.gammas || ngam_next == ngam || h->pt == a.chunk, PT_ERR_ARG,
             err("a sweep of another width needs its own candidate buffer"));
  *F = LsFinishArgs{};
  F->state = const_cast<double*>(a.skip);
  F->cand = a.gammas; F->cand_next = s.cand_next; F->step = s.step; F->w = s.w;
  F->ngam = ngam; F->ngam_next = ngam_next; F->last = last;
  return PT_OK;
}

static RhoTerm rho_term(const pt_ptycho_linesearch_args& a, LsFinishArgs* fin) {
  RhoTerm rt;
  rt.hh = (const float2*)a.hh;
  rt.lamd = (const float2*)a.lamd;
  rt.rho = a.rho;
  rt.rho_dev = a.rho_dev;
  rt.f2 = a.f2;
  rt.fin = fin;
  return rt;
}

extern "C" int pt_ptycho_linesearch_sweep(const pt_ptycho_linesearch_args* a, double* cand_next,
                                          double* step, const double* w, int ngam, int ngam_next,
                                          int last, int model, pt_stream stream) {
  PT_REQUIRE(a, PT_ERR_ARG, "pt_ptycho_linesearch_sweep: null argument");
  LsFinishArgs F;
  const int rc = sweep_args(*a, {cand_next, step, w}, ngam, ngam_next, last, model, -1, &F);
  if (rc) return rc;
  pt_ptycho* h = a->h;
  const RhoTerm rt = rho_term(*a, &F);
  hipStream_t st = (hipStream_t)stream;
  PT_DISPATCH_D(h->D, (run_minf<DD>(h, nullptr, (const float2*)a->psi, (const float2*)a->dir,
                                    a->data, a->gammas, ngam, a->chunk, a->coefptycho,
                                    a->coefdata, model, 0, a->skip, st, nullptr, 0, rt)));
}

// One launch of k_minf_tile_group and the two grouped reductions, or the grouped
// decisions (fin, by instance), for the instances idx (at most kGroupMax, all on the
// tile path with detector D and the same probe form)
template <int D>
static int run_minf_group(const pt_ptycho_linesearch_args* a, LsFinishArgs* fin, const int* idx,
                          int n, int ngam, int model, bool full, hipStream_t st) {
  Group<MinfTileArgs> g;
  Group<ReduceArgs> r1, r2;
  Group<LsFinishArgs> gf;
  size_t lds = 0;
  int tot = 0, totc = 0;
  for (int k = 0; k < n; ++k) {
    const pt_ptycho_linesearch_args& x = a[idx[k]];
    pt_ptycho* h = x.h;
    const int nchunk = h->pt / x.chunk;
    const int nbt = minf_tile_gx(h, x.chunk);
    const size_t nper = (size_t)nchunk * nbt * ngam;
    double* part;
    int rc = minf_partials(h, 2 * nper, nullptr, 0, &part);
    if (rc) return rc;
    g.a[k] = minf_tile_args(h, part, part + nper, (const float2*)x.psi, (const float2*)x.dir,
                            x.data, x.gammas, ngam, x.chunk, x.coefptycho, x.coefdata, x.skip,
                            rho_term(x, nullptr));
    g.gx[k] = nbt;
    g.start[k] = tot;
    tot += g.gx[k] * nchunk;
    r1.a[k] = ReduceArgs{x.f1, part, x.skip, (long)nbt};
    r2.a[k] = ReduceArgs{x.f2, part + nper, x.skip, (long)nbt};
    if (fin) {
      ls_tile_partials(&fin[idx[k]], part, part + nper, nbt);
      gf.a[k] = fin[idx[k]];
    }
    r1.gx[k] = r2.gx[k] = gf.gx[k] = nchunk;
    r1.start[k] = r2.start[k] = gf.start[k] = totc;
    totc += nchunk;
    lds = std::max(lds, minf_tile_lds_bytes(D, h->EB, h->P));
  }
  g.start[n] = tot;
  r1.start[n] = r2.start[n] = gf.start[n] = totc;
  g.n = r1.n = r2.n = gf.n = n;
  {
    ProfScope prof("ptycho_minf", st);
    minf_dispatch<D>(model, full, ngam, [&](auto, auto kern) {
      hipLaunchKernelGGL(kern, dim3(tot), dim3(WAVE * kMinfWaves), lds, st, g);
    });
  }
  PT_LAUNCH_CHECK();
  if (fin) {
    hipLaunchKernelGGL(k_ls_finish_group, dim3(totc), dim3(1024), 0, st, gf);
    PT_LAUNCH_CHECK();
    return PT_OK;
  }
  hipLaunchKernelGGL(k_reduce_partials_group, dim3(totc, ngam), dim3(256), 0, st, r1, ngam);
  PT_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_reduce_partials_group, dim3(totc, ngam), dim3(256), 0, st, r2, ngam);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// groups of (detector size, probe form) on the tile path, kGroupMax at a time; every
// other instance by single(i)
template <class F>
static int minf_groups(const pt_ptycho_linesearch_args* a, LsFinishArgs* fin, int n, int ngam,
                       int model, hipStream_t st, F single) {
  std::vector<int> bins[4];  // D = 8 / 16, probe partial / full
  for (int i = 0; i < n; ++i) {
    const pt_ptycho* h = a[i].h;
    int b = -1;
    if (h->D == 8 && minf_tile_path<8>(h)) b = minf_full<8>(h) ? 1 : 0;
    if (h->D == 16 && minf_tile_path<16>(h)) b = 2 + (minf_full<16>(h) ? 1 : 0);
    if (b >= 0) {
      bins[b].push_back(i);
      continue;
    }
    const int rc = single(i);
    if (rc) return rc;
  }
  for (int b = 0; b < 4; ++b) {
    for (size_t k0 = 0; k0 < bins[b].size(); k0 += kGroupMax) {
      const int m = (int)std::min<size_t>(kGroupMax, bins[b].size() - k0);
      const int* idx = bins[b].data() + k0;
      const int rc = b < 2 ? run_minf_group<8>(a, fin, idx, m, ngam, model, b == 1, st)
                           : run_minf_group<16>(a, fin, idx, m, ngam, model, b == 3, st);
      if (rc) return rc;
    }
  }
  return PT_OK;
}

extern "C" int pt_ptycho_linesearch_group(const pt_ptycho_linesearch_args* a, int n, int ngam,
                                          int model, pt_stream stream) {
  PT_REQUIRE(n >= 0 && (a || n == 0), PT_ERR_ARG, "pt_ptycho_linesearch_group: bad argument");
  PT_REQUIRE(ngam >= 1 && ngam <= PT_MAX_GAM, PT_ERR_ARG,
             "pt_ptycho_linesearch_group: 1 <= ngam <= 8");
  PT_REQUIRE(model == PT_MODEL_POISSON || model == PT_MODEL_GAUSSIAN, PT_ERR_ARG,
             "pt_ptycho_linesearch_group: bad model");
  for (int i = 0; i < n; ++i) {
    const pt_ptycho_linesearch_args& x = a[i];
    PT_REQUIRE(x.h && x.f1 && x.f2 && x.psi && x.dir && x.data && x.hh && x.lamd && x.gammas,
               PT_ERR_ARG, "pt_ptycho_linesearch_group: null argument in instance " +
                               std::to_string(i));
    PT_REQUIRE(x.h->ready, PT_ERR_STATE,
               "pt_ptycho_linesearch_group: set_scan_probe not called for instance " +
                   std::to_string(i));
    PT_REQUIRE(x.chunk > 0 && x.h->pt % x.chunk == 0, PT_ERR_SIZE,
               "pt_ptycho_linesearch_group: chunk must divide the number of angles (instance " +
                   std::to_string(i) + ")");
    PT_REQUIRE(x.rho_dev || x.rho > 0, PT_ERR_ARG,
               "pt_ptycho_linesearch_group: rho must be positive (instance " + std::to_string(i) +
                   ")");
  }
  PT_REQUIRE(distinct_handles(a, n), PT_ERR_ARG,
             "pt_ptycho_linesearch_group: a handle appears twice (its partial sums would be "
             "shared)");
  return minf_groups(a, nullptr, n, ngam, model, (hipStream_t)stream, [&](int i) {
    const pt_ptycho_linesearch_args& x = a[i];
    return pt_ptycho_linesearch(x.h, x.f1, x.f2, x.psi, x.dir, x.data, x.hh, x.lamd, x.rho,
                                x.rho_dev, x.gammas, ngam, x.chunk, x.coefptycho, x.coefdata,
                                model, x.skip, stream);
  });
}

extern "C" int pt_ptycho_linesearch_sweep_group(const pt_ptycho_linesearch_args* a,
                                                const pt_ptycho_sweep_args* s, int n, int ngam,
                                                int ngam_next, int last, int model,
                                                pt_stream stream) {
  PT_REQUIRE(n >= 0 && ((a && s) || n == 0), PT_ERR_ARG,
             "pt_ptycho_linesearch_sweep_group: bad argument");
  std::vector<LsFinishArgs> fin(n);
  for (int i = 0; i < n; ++i) {
    const int rc = sweep_args(a[i], s[i], ngam, ngam_next, last, model, i, &fin[i]);
    if (rc) return rc;
  }
  PT_REQUIRE(distinct_handles(a, n), PT_ERR_ARG,
             "pt_ptycho_linesearch_sweep_group: a handle appears twice (its partial sums would "
             "be shared)");
  return minf_groups(a, fin.data(), n, ngam, model, (hipStream_t)stream, [&](int i) {
    return pt_ptycho_linesearch_sweep(&a[i], s[i].cand_next, s[i].step, s[i].w, ngam, ngam_next,
                                      last, model, stream);
  });
}

extern "C" int pt_ptycho_minf(pt_ptycho* h, double* sums, const void* psi, const void* dir,
                              const float* data, const double* gammas, int ngam, int chunk,
                              float coefptycho, float coefdata, int model, int lagr,
                              const double* skip, pt_stream stream) {
  return minf_impl(h, sums, psi, dir, data, gammas, ngam, chunk, coefptycho, coefdata, model,
                   lagr, skip, stream, nullptr, 0);
}

// Partial sums of pt_ptycho_minf_noalloc: one fixed array per device (16
// MiB, held until the process ends).  Every slot a launch reads is written
// by the same launch, so nothing needs clearing; calls that overlap on one
// device share it and race.
static __device__ __align__(256) double scratch[PT_MINF_NOALLOC_PARTIALS];

namespace {
std::mutex g_scratch_mu;
std::vector<double*> g_scratch_ptr;   // per device: address of `scratch` there
}  // namespace

// Device address of this device's `scratch`, looked up on the device's first
// call (host code uses the address, never the symbol itself).
static int scratch_on_current_device(double** out) {
  int dev = 0;
  PT_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize(dev + 1, nullptr);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    PT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    PT_REQUIRE(p, PT_ERR_HIP, "pt_ptycho_minf_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return PT_OK;
}

extern "C" int pt_ptycho_minf_noalloc(pt_ptycho* h, double* sums, const void* psi,
                                      const void* dir, const float* data, const double* gammas,
                                      int ngam, int chunk, float coefptycho, float coefdata,
                                      int model, int lagr, const double* skip, pt_stream stream) {
  double* part = nullptr;
  int rc = scratch_on_current_device(&part);
  if (rc) return rc;
  return minf_impl(h, sums, psi, dir, data, gammas, ngam, chunk, coefptycho, coefdata, model,
                   lagr, skip, stream, part, PT_MINF_NOALLOC_PARTIALS);
}
