// USFFT Radon transform for gfx950.
//
// Replaces class radonusfft (src/cuda/radonusfft.cu + kernels.cuh kernels
// divphi, unpaddivphi, fftshiftc, fftshift1c, wrap, wrapadj, takexy, gather,
// scatter, circ, pad, pad2) and its three cuFFT plans.
//
// Same mathematics as the reference chain (gridding on the 2N x 2N oversampled
// grid, N = 3n/2), restructured:
//  * The checkerboard multiplications around each FFT are centred DFTs; they
//    are realised as index rotations on load/store (free).
//  * The 2L-point centred DFT of an input that is non-zero only on the
//    central L points splits into two L-point DFTs (even outputs: plain
//    input; odd outputs: input twisted by exp(-i pi j/L)).  All FFTs are
//    Stockham transforms of N points (the forward's grid lines and the detector
//    lines) or n points (the adjoint's grid lines): for n = 64, 96, 128, 192, 256
//    and 512 register line FFTs (24 points per lane; n-point lines of a power of
//    two 16), compile-time passes with LDS only for the exchanges between them,
//    otherwise LDS transforms with a run-time mixed-radix plan (2/3/4/5/8).
//  * pad2 + circ + divphi are applied while loading the object rows; the
//    adjoint's unpaddivphi + circ + crop are applied while storing them.  The
//    adjoint only needs the n x n object points (the forward transforms the
//    N x N extended object), so its grid is 2n x 2n and its lines have n points.
//  * The periodic halo of the gridding grid (wrap/wrapadj) is an index
//    modulo the grid edge.
//  * Grid buffers hold pairs of slices interleaved, so that a grid point of a
//    pair is one 16-byte access.
//  * gather: 8 x 8 Kaiser-Bessel taps (see below) from grid tiles staged in LDS.
//  * scatter: deterministic and free of atomics.  At set_theta time every
//    8 x 8 grid tile gets the list of polar samples whose footprint covers
//    part of it (wrapadj folded into the periodic offsets); one wavefront owns
//    a (tile, list chunk, slices) work item and accumulates the tile as FP32
//    matrix-core products; tiles with several chunks sum their partials in a
//    fixed order in a fix-up kernel.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"

namespace {
constexpr int kTile = 32;                // gather tile edge (grid points)
constexpr int kWorkMax = 256;            // samples per gather work item
}  // namespace

struct pt_tomo {
  int ntheta, pz, n, N;
  int pzs;                   // pz rounded up to whole blocks of 8 slices
  pt::LinePlan plan, plann;  // lines of N and of n points
  float2* tw = nullptr;      // [N] exp(-2 pi i m/N)
  float2* twist = nullptr;   // [N] exp(-i pi j/N), j = idx - N/2
  float2* twn = nullptr;     // [n], [n]: the same for n
  float2* twistn = nullptr;
  float* dphi = nullptr;     // [N] forward: 1/(kernel's transform) at a/(2N), a = idx - N/2
  float* dphia = nullptr;    // [n] adjoint: the same at a/(2n), a = idx - n/2
  float* filt = nullptr;     // [N] detector-frequency filter of the adjoint, or null
  int2* mrange = nullptr;    // [N] circ mask column range [lo, hi) per row
  float2* spos = nullptr;    // [ntheta*N] sample positions (x, y)
  int2* sfloor = nullptr;    // [ntheta*N] floor(2N*x), floor(2N*y)
  float* wfwd = nullptr;     // [ntheta*N][16] gridding weights, forward and adjoint
  float* wadj = nullptr;
  // buffers of both directions (pz rounded up to whole blocks)
  float2* A = nullptr;       // fwd [pz/2][N][2N][2], adj [pz/2][n][2n][2]
  float2* Bg = nullptr;      // fwd [pz/2][2N][2N][2], adj [pz/2][2n][2n][2]
  float2* Q = nullptr;       // polar samples: fwd [pz/2][sample][2], adj [sample][pzs]
  // gather bins: samples by kTile x kTile tile of their floor position
  int ntile1 = 0;            // tiles per axis
  int* wi_tile = nullptr;    // [nwi] tile index
  int2* wi_range = nullptr;  // [nwi] [s0, s1) into bin_sample
  int* bin_sample = nullptr; // [ntheta*N]
  int nwi = 0;
  // scatter: per 8 x 8 tile of the 2n x 2n grid, the samples whose footprint covers it
  int nts = 0;               // tiles per axis
  int2* ent = nullptr;       // [nent] sample, footprint origin - tile: x + 8 | y << 8
  int* swi_tile = nullptr;   // [nswi]
  int2* swi_range = nullptr; // [nswi] entry range
  int* swi_slot = nullptr;   // [nswi] partial slot, -1 = direct write
  int4* sfix = nullptr;      // [nfix] (tile, first slot, nslots, 0)
  int nswi = 0, nfix = 0, szb = 1;
  float2* spart = nullptr;   // [nslots][pzs/2][64][2]
  int rows_per_wg = 1, cols_per_wg = 1, adj_lines = 1;
  int line_kind = PT_LINES_AUTO;  // line passes: register FFT where N allows, or generic
  bool ready = false;
};

namespace pt {
namespace {

// ------------------------------------------------------------------ grid disc
// The polar samples lie within the disc of radius h of the 2h x 2h grid (h = N
// forward, n adjoint), their footprints (kW points wide, folded into the grid by
// periodicity, which only brings them nearer to the centre) within h + 6.  The
// grid's corners outside, 1 - pi/4 of it, are neither written nor read: 250 MB less
// to write for the column pass at 256^3 (0.48 -> 0.46 ms), and in the adjoint as
// much less to write and read in all (column pass 185 -> 169 us, operator 788 ->
// 752 us; 180^2 x 21 slices 100 -> 94 us).  The points between the disc and the
// samples' footprints are written as zeros.
constexpr int kDiscMargin = 6;
// largest |ky| within the disc at column offset kx from the centre (one more than
// needed at most)
__host__ __device__ inline int disc_rows(int kx, int h) {
  const int r = h + kDiscMargin;
  return (int)sqrtf((float)(r * r - kx * kx)) + 1;
}

// ------------------------------------------------------------------ forward row pass
// For rows q of slice z: x[p] = mask*u[clamp]*dphi[q]*dphi[p] (pad2, circ,
// divphi), centred 2N-point DFT along p -> A[z/2][q][kx][z%2], kx = k' + N.
// (A last pair with one slice carries a copy of it in the other half.)
// A workgroup takes `rows` of the pair's 2 N (row, slice) lines.
__global__ __launch_bounds__(256) void k_row_fwd(float2* __restrict__ A, const float2* __restrict__ u,
                          const float2* __restrict__ tw, const float2* __restrict__ twist,
                          const float* __restrict__ dphi, const int2* __restrict__ mrange,
                          LinePlan plan, int n, int rows, int pz) {
  extern __shared__ float2 lds[];
  const int N = plan.N, r0 = blockIdx.x * rows;
  const int o = N / 6;
  const int nl = 2 * rows;  // line 2r: plain, 2r+1: twisted
  float2* lb = lds + nl * (N + 1);  // ping-pong partner
  float2* twl = lb + nl * (N + 1);
  for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = tw[i];
  for (int i = threadIdx.x; i < nl * N; i += blockDim.x) {
    const int line = i / N, c = i - line * N;
    const int r = r0 + (line >> 1), q = r >> 1;
    const int z = min(2 * (int)blockIdx.y + (r & 1), pz - 1);
    float2 val = make_float2(0.f, 0.f);
    if (q < N) {
      const int2 mr = mrange[q];
      if (c >= mr.x && c < mr.y) {
        const int uy = min(max(q - o, 0), n - 1), ux = min(max(c - o, 0), n - 1);
        val = cscale(u[((long)z * n + uy) * n + ux], dphi[q] * dphi[c]);
        if (line & 1) val = cmul(val, twist[c]);
      }
    }
    // centred -> rotated index a' = (c + N/2) mod N
    int a = c + N / 2;
    if (a >= N) a -= N;
    lds[line * (N + 1) + a] = val;
  }
  __syncthreads();
  const float2* res = lds_fft_pp<-1>(lds, lb, N + 1, nl, plan, twl, threadIdx.x, blockDim.x);
  for (int i = threadIdx.x; i < nl * N; i += blockDim.x) {
    const int line = i / N, b = i - line * N;
    const int r = r0 + (line >> 1), q = r >> 1;
    if (q >= N) continue;
    const int m = b < N / 2 ? b : b - N;  // centred frequency
    const int kx = 2 * m + N + (line & 1);
    A[(((long)blockIdx.y * N + q) * (2 * N) + kx) * 2 + (r & 1)] = res[line * (N + 1) + b];
  }
}

// ------------------------------------------------------------------ forward column pass
// Column tiles run in XCD-contiguous order (xcd_contig): neighbouring tiles
// read the same cache lines of the rows (8 columns = 64 bytes per row).
//
// C = 2^lc of the 4N columns (kx, slice) of one slice pair z per workgroup:
// y[q] = A[z][q][kx] -> centred 2N-point DFT along q -> B[z][ky][kx], as the plain N-point DFT
// (even ky - N) and the twisted one (odd ky - N) run one after the other in
// the same C padded LDS lines (ping-pong pair).  The N x C tile stays in
// registers between the two; the twiddle table is staged in LDS.
constexpr int kColVpt = 12;  // tile values per thread: N * C <= 256 * kColVpt
__global__ __launch_bounds__(256) void k_col_fwd(float2* __restrict__ Bg, const float2* __restrict__ A,
                          const float2* __restrict__ tw, const float2* __restrict__ twist,
                          LinePlan plan, int lc) {
  extern __shared__ float2 lds[];
  const int N = plan.N, W = 4 * N, S = N + 1, C = 1 << lc;  // W: columns of a slice pair
  const int gx = (W + C - 1) >> lc;
  const int L = xcd_contig(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int z = L / gx, k0 = (L - z * gx) << lc;
  float2* la = lds;
  float2* lb = la + C * S;
  float2* twl = lb + C * S;
  for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = tw[i];
  const int nv = (N * C + 255) >> 8;
  const float2* Az = A + (long)z * N * W + k0;
  float2 reg[kColVpt];
#pragma unroll
  for (int v = 0; v < kColVpt; ++v) {
    if (v < nv) {
      const int i = threadIdx.x + v * 256;
      const int q = i >> lc, cc = i & (C - 1);
      reg[v] = (q < N && k0 + cc < W) ? Az[(long)q * W + cc] : make_float2(0.f, 0.f);
    }
  }
  float2* Bz = Bg + (long)z * (2 * N) * W + k0;
  for (int par = 0; par < 2; ++par) {
#pragma unroll
    for (int v = 0; v < kColVpt; ++v) {
      if (v < nv) {
        const int i = threadIdx.x + v * 256;
        const int q = i >> lc, cc = i & (C - 1);
        if (q < N) {
          int a = q + N / 2;  // centred -> rotated
          if (a >= N) a -= N;
          la[cc * S + a] = par ? cmul(reg[v], twist[q]) : reg[v];
        }
      }
    }
    __syncthreads();
    const float2* res = lds_fft_pp<-1>(la, lb, S, C, plan, twl, threadIdx.x, blockDim.x);
    for (int i = threadIdx.x; i < N * C; i += blockDim.x) {
      const int r = i >> lc, cc = i & (C - 1);
      if (k0 + cc >= W) continue;
      const int m = r - N / 2;  // ky - N = 2m + par
      const int b = m < 0 ? m + N : m;
      if (abs(2 * m + par) <= disc_rows(((k0 + cc) >> 1) - N, N))
        Bz[(long)(2 * m + par + N) * W + cc] = res[cc * S + b];
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ gridding kernel
// Interpolation between the oversampled grid and the polar samples with the
// Kaiser-Bessel kernel I0(beta sqrt(1 - (2d/w)^2)) / I0(beta) of width w = 8
// grid points, beta as pi sqrt((w/s)^2 (s - 1/2)^2 - 0.8) = 18.6389 for oversampling
// s = 2 (Beatty, Nishimura and Pauly 2005).  kBeta is 4.5e-6 below that expression,
// for which the aliasing error is the same to 1e-4 of itself (5.25e-8 rms over the
// object); kernel and transform use the one value.  Its Fourier transform
// w sinh(r)/r / I0(beta), r = sqrt(beta^2 - (pi w xi)^2), is divided out of the
// object points (dphi).  The reference's Gaussian with 15 x 15 taps
// (kernels.cuh:97-158, eps = 1e-6) approximates the same nonuniform Fourier
// sums: in 64 bits, on white-noise objects, it is 2.5e-7 from the direct sums,
// this kernel with 8 x 8 taps 6e-8 (7 taps: 6e-7).
constexpr int kW = 8;
constexpr int kWLo = kW / 2 - 1;  // taps floor(x) - kWLo .. floor(x) + kW/2
constexpr double kBeta = 18.638856593895362;

__host__ __device__ inline double bessel_i0(double x) {
  const double t = 0.25 * x * x;
  double term = 1.0, sum = 1.0;
#pragma unroll
  for (int k = 1; k < 64; ++k) {
    term *= t * (1.0 / ((double)k * k));
    sum += term;
  }
  return sum;
}
// 1 / Fourier transform of the kernel at frequency xi (cycles per grid point)
double kb_inverse_ft(double xi) {
  const double a = kPi * kW * xi, r = std::sqrt(kBeta * kBeta - a * a);
  return r * bessel_i0(kBeta) / (kW * std::sinh(r));
}

// Weights of all samples, FP64 rounded to FP32: w[s][0..7] of the columns
// floor(G x) - 3 .. floor(G x) + 4, w[s][8..15] of the rows (y).
__global__ __launch_bounds__(256) void k_kb_weights(float* __restrict__ w,
                                                    const float2* __restrict__ spos, long ns,
                                                    int G, double peak) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= ns * 2 * kW) return;
  const int k = (int)(i % (2 * kW));
  const float2 p = spos[i / (2 * kW)];
  const double x = (double)G * (double)(k < kW ? p.x : p.y);
  const double d = (floor(x) - kWLo + (k % kW) - x) / (kW / 2);
  w[i] = (float)(bessel_i0(kBeta * sqrt(fmax(0.0, 1.0 - d * d))) / peak);
}

// ------------------------------------------------------------------ gather
// One workgroup per (32 x 32 grid tile bin chunk, zper slice pairs): the
// tile plus the footprint's halo (periodic in 2N) is staged in LDS as
// [y][x][slice of the pair]; each lane interpolates its polar samples with
// separable weights held in registers for all of the workgroup's pairs.
// Output G[z/2][sample][z%2].  The loads of the next pair's tile are in flight
// (registers) while a pair is interpolated from LDS.
// Bound: LDS reads, 64 taps x 16 bytes per sample and slice pair (0.25 ms at
// 256^3, 384 angles, at 128 bytes per cycle and CU), beside 1.5 GB of grid and
// samples (0.3 ms): 0.38 ms per launch there, 1.44 ms with the 15 x 15
// Gaussian taps; at 32^2 x 8 slices, 48 angles, 169 -> 8 us.  One sample per
// lane: with two, the weights and the reads in flight took 211 registers (two
// waves per SIMD, 0.54 ms); 512 lanes per workgroup measured 1 % slower.
constexpr int kGE = kTile + kW - 1;                                // staged tile edge
constexpr int kGatherStage = (kGE * kGE + kWorkMax - 1) / kWorkMax;  // staged points per lane
typedef float f4v __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(kWorkMax, 4) void k_gather_tile(
    f4v* __restrict__ G, const f4v* __restrict__ Bg, const f4v* __restrict__ wts,
    const int2* __restrict__ sfloor, const int* __restrict__ wi_tile,
    const int2* __restrict__ wi_range, const int* __restrict__ bin_sample, int N, int ntile1,
    int ns, int npair, int zper) {
  __shared__ f4v lds4[kGatherStage * kWorkMax];  // [y][x], then slots of the staging's last round
  const int twoN = 2 * N;
  // XCD-contiguous order: adjacent tiles' staged regions overlap
  const int lw = xcd_contig(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int zb = lw / gridDim.x;
  const int wi = lw - zb * gridDim.x;
  const int jp0 = zb * zper, jp1 = min(jp0 + zper, npair);
  const int tile = wi_tile[wi];
  const int ty0 = (tile / ntile1) * kTile, tx0 = (tile % ntile1) * kTile;
  const int2 rg = wi_range[wi];
  // this lane's sample, its weights and its footprint's offset in the staged tile
  const int bi = rg.x + threadIdx.x;
  const int sid = bi < rg.y ? bin_sample[bi] : -1;
  const int2 f = sfloor[max(sid, 0)];
  const int off = sid < 0 ? 0 : (f.y + N - ty0) * kGE + f.x + N - tx0;
  const f4v* wp = wts + (long)max(sid, 0) * (2 * kW / 4);
  const f4v wx[2] = {wp[0], wp[1]}, wy[2] = {wp[2], wp[3]};
  // grid offsets of this lane's staged points
  int goff[kGatherStage];
#pragma unroll
  for (int u = 0; u < kGatherStage; ++u) {
    const int i = min((int)threadIdx.x + u * kWorkMax, kGE * kGE - 1);
    const int y = i / kGE, x = i - y * kGE;
    int gy = ty0 - kWLo + y, gx = tx0 - kWLo + x;
    gy = gy < 0 ? gy + twoN : gy;
    gx = gx < 0 ? gx + twoN : gx;
    goff[u] = (gy % twoN) * twoN + gx % twoN;
  }
  f4v va[kGatherStage];
  const f4v* B = Bg + (long)jp0 * twoN * twoN;
#pragma unroll
  for (int u = 0; u < kGatherStage; ++u) va[u] = B[goff[u]];
  for (int jp = jp0; jp < jp1; ++jp) {
    __syncthreads();  // the previous pair's interpolation has read the tile
#pragma unroll
    for (int u = 0; u < kGatherStage; ++u) lds4[threadIdx.x + u * kWorkMax] = va[u];
    __syncthreads();
    if (jp + 1 < jp1) {
      B += (long)twoN * twoN;
#pragma unroll
      for (int u = 0; u < kGatherStage; ++u) va[u] = B[goff[u]];
    }
    if (sid < 0) continue;
    const f4v* rp = lds4 + off;
    f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k1 = 0; k1 < kW; ++k1) {
      f4v r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k0 = 0; k0 < kW; ++k0) r += wx[k0 / 4][k0 % 4] * rp[k1 * kGE + k0];
      acc += wy[k1 / 4][k1 % 4] * r;
      __builtin_amdgcn_sched_barrier(0);  // one row's reads in flight per wave: no spills
    }
    G[(long)jp * ns + sid] = acc;
  }
}

// centred inverse 1D DFT of each (angle, slice) line of gathered samples,
// fftshift1c signs folded into index rotations, detector crop; zq slices of
// one angle per workgroup (lines padded to N+1 in LDS)
__global__ __launch_bounds__(256) void k_line_idft(float2* __restrict__ g, const float2* __restrict__ G,
                            const float2* __restrict__ tw, LinePlan plan, float oscale, int n,
                            int ntheta, int pz, int zq) {
  extern __shared__ float2 lds[];
  const int N = plan.N, th = blockIdx.x, z0 = blockIdx.y * zq;
  const int nzl = min(zq, pz - z0);
  float2* lb = lds + zq * (N + 1);
  float2* twl = lb + zq * (N + 1);
  for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = tw[i];
  for (int i = threadIdx.x; i < zq * N; i += blockDim.x) {
    const int zz = i / N, k = i - zz * N;
    int a = k - N / 2;  // kappa -> kappa mod N
    if (a < 0) a += N;
    lds[zz * (N + 1) + a] =
        zz < nzl ? G[(((long)((z0 + zz) >> 1) * ntheta + th) * N + k) * 2 + ((z0 + zz) & 1)]
                 : make_float2(0.f, 0.f);
  }
  __syncthreads();
  const float2* res = lds_fft_pp<1>(lds, lb, N + 1, zq, plan, twl, threadIdx.x, blockDim.x);
  for (int i = threadIdx.x; i < nzl * n; i += blockDim.x) {
    const int zz = i / n, j = i - zz * n;
    int b = j - n / 2;
    if (b < 0) b += N;
    g[((long)th * pz + z0 + zz) * n + j] = cscale(res[zz * (N + 1) + b], oscale);
  }
}

// ------------------------------------------------------------------ adjoint line: pad + 1D DFT
// ZQ slices of one angle per workgroup; output Q[sample][z] (z fastest, pzs =
// pz rounded up to 8 slices, the rest zeros) for the owner-computes scatter.
constexpr int kZQ = 8;
__global__ __launch_bounds__(256) void k_adj_line(float2* __restrict__ Q, const float2* __restrict__ g,
                           const float2* __restrict__ tw, const float* __restrict__ filt,
                           LinePlan plan, float oscale, int n, int ntheta, int pz, int pzs,
                           int zq) {
  extern __shared__ float2 lds[];
  const int N = plan.N, th = blockIdx.x, z0 = blockIdx.y * zq;
  const int nzl = min(zq, pz - z0);
  const int o = N / 6;
  float2* lb = lds + zq * (N + 1);
  float2* twl = lb + zq * (N + 1);
  for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = tw[i];
  for (int i = threadIdx.x; i < zq * N; i += blockDim.x) {
    const int zz = i / N, sidx = i - zz * N;
    float2 v = make_float2(0.f, 0.f);
    if (zz < nzl) {
      const int j = min(max(sidx - o, 0), n - 1);  // pad (kernels.cuh:189-206)
      v = g[((long)th * pz + z0 + zz) * n + j];
    }
    int a = sidx + N / 2;
    if (a >= N) a -= N;
    lds[zz * (N + 1) + a] = v;
  }
  __syncthreads();
  const float2* res = lds_fft_pp<-1>(lds, lb, N + 1, zq, plan, twl, threadIdx.x, blockDim.x);
  for (int t = threadIdx.x; t < zq * N; t += blockDim.x) {
    const int i = t / zq, zz = t - i * zq;
    if (z0 + zz >= pzs) continue;
    int b = i - N / 2;  // kappa
    if (b < 0) b += N;
    const float w = filt ? oscale * filt[i] : oscale;
    Q[((long)th * N + i) * pzs + z0 + zz] = cscale(res[zz * (N + 1) + b], w);
  }
}

// ------------------------------------------------------------------ scatter (owner computes)
// Adjoint gridding (kernels.cuh:128-158 transposed, wrapadj folded in by the
// periodic entry offsets) onto the 2n x 2n grid -- the n object points are
// oversampled by 2 -- as a matrix product per grid tile of 8 x 8 points:
//   G[(z, part)][point] = sum_entries Q_e[(z, part)] * (wx_e wy_e)[point],
// K = the tile's entries (samples whose 8 x 8 footprint covers part of the
// tile, in list order), on FP32 matrix cores: one 16x16x4 MFMA takes 4
// entries, 8 slices (16 rows: slice, re/im) and 16 points (8 columns x 2
// rows).  A wavefront takes one tile entry chunk and 8 ZB slices, i.e. 4 ZB
// MFMAs per 4 entries; the A operand is read straight from the samples
// (16 adjacent lanes: 64 contiguous bytes), the B operand is the product of a
// column and a row weight.  Per 32 entries, lane l stages the column (l < 32)
// or row weights of entry l % 32, clipped to the tile, in LDS; the weights of
// the next 32 entries and the index of the ones after are loaded meanwhile.
// MFMA 16x16x4 f32 operand layout (lane l): A[i][k]: i = l%16, k = l/16;
// B[k][j]: j = l%16, k = l/16; D[i][j]: j = l%16, i = 4*(l/16) + r, so a lane
// ends with one point of one slice pair: a 16-byte store, 8 adjacent points.
// Bound: matrix cores.  A footprint meets (15/8)^2 = 3.5 tiles, so 450
// multiply-adds per sample and slice (0.22 ms at 256^3, 384 angles); tiles of
// 16 x 8 points would take 690.  Measured there: 0.45 ms per launch, 1.39 ms with
// 15 x 15 Gaussian footprints on the 3n x 3n grid (whose column pass took 0.39
// ms and row pass 0.12, now 0.19 and 0.11).
constexpr int kTS = 8;    // scatter tile edge
constexpr int kSE = 32;   // entries per staged chunk
typedef float f4m __attribute__((ext_vector_type(4)));
template <int ZB>
__global__ __launch_bounds__(64) void k_scatter_own(f4m* __restrict__ Bg, f4m* __restrict__ part,
                                                    const float* __restrict__ Q,
                                                    const f4m* __restrict__ wts,
                                                    const int2* __restrict__ ent,
                                                    const int* __restrict__ wi_tile,
                                                    const int2* __restrict__ wi_range,
                                                    const int* __restrict__ wi_slot, int ntx,
                                                    int pzs) {
  __shared__ float wl[2][kSE][kTS + 1];  // column, row weights on the tile
  __shared__ int sl[kSE];                // samples
  // XCD-contiguous order: adjacent tiles share the samples of their entries
  const int lw = xcd_contig(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int zb = lw / gridDim.x;
  const int wi = lw - zb * gridDim.x, z0 = zb * 8 * ZB;
  const int nzb = min(ZB, (pzs - z0) / 8);  // blocks of 8 slices
  const int lane = threadIdx.x, j16 = lane & 15, kq = lane >> 4;
  const int el = lane & (kSE - 1), ax = lane / kSE;
  const int tile = wi_tile[wi];
  const int2 rg = wi_range[wi];
  f4m acc[ZB][4];
#pragma unroll
  for (int t = 0; t < ZB; ++t)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[t][b] = f4m{0.f, 0.f, 0.f, 0.f};
  // entry (sample, offsets) of this lane; past the end: sample -1
  auto fetch_ent = [&](int c0) { return c0 + el < rg.y ? ent[c0 + el] : make_int2(-1, 0); };
  int2 ec = fetch_ent(rg.x), en = fetch_ent(rg.x + kSE);
  const f4m* wp = wts + (long)max(ec.x, 0) * 4 + 2 * ax;
  f4m w0 = wp[0], w1 = wp[1];
  const float* Qz = Q + 2 * (long)z0 + j16;
  for (int c0 = rg.x; c0 < rg.y; c0 += kSE) {
    __syncthreads();  // the previous chunk's weights are read
    {
      const int o = ax ? ec.y >> 8 : (ec.y & 255) - 8;  // footprint origin - tile
      float* row = wl[ax][el];
#pragma unroll
      for (int k = 0; k < kTS; ++k) row[k] = 0.f;
      if (ec.x >= 0) {
#pragma unroll
        for (int k = 0; k < kW; ++k) {
          const int x = k + o;
          if (x >= 0 && x < kTS) row[x] = k < 4 ? w0[k] : w1[k - 4];
        }
      }
      if (!ax) sl[el] = max(ec.x, 0);  // a sample of zero weight past the end
    }
    __syncthreads();
    const int ng = (min(kSE, rg.y - c0) + 3) / 4;
    // all samples of the chunk in flight
    float q[kSE / 4][ZB];
#pragma unroll
    for (int g = 0; g < kSE / 4; ++g) {
      const float* qp = Qz + (long)sl[4 * g + kq] * (2 * pzs);
#pragma unroll
      for (int t = 0; t < ZB; ++t) q[g][t] = (g < ng && t < nzb) ? qp[16 * t] : 0.f;
    }
    ec = en;
    wp = wts + (long)max(ec.x, 0) * 4 + 2 * ax;
    w0 = wp[0];
    w1 = wp[1];
    en = fetch_ent(c0 + 2 * kSE);
#pragma unroll
    for (int g = 0; g < kSE / 4; ++g) {
      if (g < ng) {
        const int e = 4 * g + kq;
        const float wx = wl[0][e][j16 & 7];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float w = wx * wl[1][e][2 * b + (j16 >> 3)];
#pragma unroll
          for (int t = 0; t < ZB; ++t)
            acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[g][t], w, acc[t][b], 0, 0, 0);
        }
      }
    }
  }
  const int slot = wi_slot[wi], G = kTS * ntx, npair = pzs / 2;
  const int x = j16 & 7, y = j16 >> 3;
#pragma unroll
  for (int t = 0; t < ZB; ++t) {
    if (t >= nzb) break;
    const long pr = z0 / 2 + 4 * t + kq;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (slot < 0)
        Bg[(pr * G + (tile / ntx) * kTS + 2 * b + y) * G + (tile % ntx) * kTS + x] = acc[t][b];
      else
        part[(slot * (long)npair + pr) * (kTS * kTS) + (2 * b + y) * kTS + x] = acc[t][b];
    }
  }
}

// tiles whose entry list spans several chunks: sum the chunk partials in order
__global__ __launch_bounds__(kTS * kTS) void k_scatter_fix(f4m* __restrict__ Bg,
                                                           const f4m* __restrict__ part,
                                                           const int4* __restrict__ fix, int ntx,
                                                           int npair) {
  const int4 f = fix[blockIdx.x];  // (tile, first slot, nslots, -)
  const int pr = blockIdx.y, p = threadIdx.x, G = kTS * ntx;
  f4m s = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < f.z; ++k) s += part[((f.y + k) * (long)npair + pr) * (kTS * kTS) + p];
  Bg[((long)pr * G + (f.x / ntx) * kTS + p / kTS) * G + (f.x % ntx) * kTS + p % kTS] = s;
}

// ------------------------------------------------------------------ adjoint column pass
// C = 2^lc of the 4n columns (kx, slice) of slice pair z per workgroup: centred
// inverse 2n-point DFT along ky evaluated at the n object rows, as the even
// and the odd n-point inverse DFTs run one after the other in the same C LDS
// lines (ping-pong pair); the even half waits in registers.
// Bg[z][2n][2n][2] -> A[z][n][2n][2].
__global__ __launch_bounds__(256) void k_col_adj(float2* __restrict__ A, const float2* __restrict__ Bg,
                          const float2* __restrict__ tw, const float2* __restrict__ twist,
                          LinePlan plan, int lc) {
  extern __shared__ float2 lds[];
  const int n = plan.N, W = 4 * n, S = n + 1, C = 1 << lc;
  const int gx = (W + C - 1) >> lc;
  const int L = xcd_contig(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int z = L / gx, k0 = (L - z * gx) << lc;
  float2* la = lds;
  float2* lb = la + C * S;
  float2* twl = lb + C * S;
  for (int i = threadIdx.x; i < n; i += blockDim.x) twl[i] = tw[i];
  const int nv = (n * C + 255) >> 8;  // n * C <= 256 * kColVpt since 3n/2 * C is
  const float2* Bz = Bg + (long)z * (2 * n) * W + k0;
  float2* Az = A + (long)z * n * W + k0;
  // lines of parity par of the C columns -> LDS, inverse FFT
  auto phase = [&](int par) -> const float2* {
    for (int i = threadIdx.x; i < n * C; i += blockDim.x) {
      const int r = i >> lc, cc = i & (C - 1);
      const int m = r - n / 2;  // ky - n = 2m + par
      const int b = m < 0 ? m + n : m;
      const bool in =
          k0 + cc < W && abs(2 * m + par) <= disc_rows(((k0 + cc) >> 1) - n, n);
      la[cc * S + b] = in ? Bz[(long)(2 * m + par + n) * W + cc] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    return lds_fft_pp<1>(la, lb, S, C, plan, twl, threadIdx.x, blockDim.x);
  };
  float2 ev[kColVpt];
  const float2* res = phase(0);
#pragma unroll
  for (int v = 0; v < kColVpt; ++v) {
    const int i = threadIdx.x + v * 256;
    const int q = i >> lc, cc = i & (C - 1);
    int a = q - n / 2;
    if (a < 0) a += n;
    if (v < nv && q < n) ev[v] = res[cc * S + a];
  }
  __syncthreads();
  res = phase(1);
#pragma unroll
  for (int v = 0; v < kColVpt; ++v) {
    const int i = threadIdx.x + v * 256;
    const int q = i >> lc, cc = i & (C - 1);
    if (v < nv && q < n && k0 + cc < W) {
      int a = q - n / 2;
      if (a < 0) a += n;
      Az[(long)q * W + cc] = cadd(ev[v], cmulc(res[cc * S + a], twist[q]));
    }
  }
}

// ------------------------------------------------------------------ adjoint row pass
// A workgroup takes `rows` of the pair's 2 n (row, slice) lines; unpaddivphi +
// circ + crop while storing.
__global__ __launch_bounds__(256) void k_row_adj(float2* __restrict__ f, const float2* __restrict__ A,
                          const float2* __restrict__ tw, const float2* __restrict__ twist,
                          const float* __restrict__ dphi, const int2* __restrict__ mrange,
                          LinePlan plan, int rows, float scale, int pz) {
  extern __shared__ float2 lds[];
  const int n = plan.N, r0 = blockIdx.x * rows, pr = blockIdx.y;
  const int o = n / 4;  // (3n/2) / 6
  const int nl = 2 * rows;
  float2* lb = lds + nl * (n + 1);
  float2* twl = lb + nl * (n + 1);
  for (int i = threadIdx.x; i < n; i += blockDim.x) twl[i] = tw[i];
  for (int i = threadIdx.x; i < 2 * n * rows; i += blockDim.x) {
    const int rl = i / (2 * n), kx = i - rl * 2 * n;
    const int r = r0 + rl;
    float2 val = make_float2(0.f, 0.f);
    if (r < 2 * n) val = A[(((long)pr * n + (r >> 1)) * (2 * n) + kx) * 2 + (r & 1)];
    const int kp = kx - n;
    const int par = kp & 1;
    const int m = (kp - par) / 2;
    const int b = m < 0 ? m + n : m;
    lds[(2 * rl + par) * (n + 1) + b] = val;
  }
  __syncthreads();
  const float2* res = lds_fft_pp<1>(lds, lb, n + 1, nl, plan, twl, threadIdx.x, blockDim.x);
  for (int i = threadIdx.x; i < n * rows; i += blockDim.x) {
    const int rl = i / n, p = i - rl * n;
    const int r = r0 + rl, q = r >> 1, z = 2 * pr + (r & 1);
    if (q >= n || z >= pz) continue;
    int a = p - n / 2;
    if (a < 0) a += n;
    const float2 e = res[(2 * rl) * (n + 1) + a];
    const float2 od = res[(2 * rl + 1) * (n + 1) + a];
    const float2 v = cadd(e, cmulc(od, twist[p]));
    const int2 mr = mrange[q + o];
    const float w = (p + o >= mr.x && p + o < mr.y) ? dphi[q] * dphi[p] * scale : 0.f;
    f[((long)z * n + q) * n + p] = cscale(v, w);
  }
}

// ------------------------------------------------------------------ register line FFT passes
// The six line passes above on the register line FFT (LineReg) for n = 64, 96,
// 128, 192, 256, 512: every lane holds P points of one line, the passes' index
// arithmetic is compile-time, and LDS is used only for the exchanges between
// Stockham passes.  Lines of N = 3n/2 points (the forward's grid passes and the
// detector lines) take P = 24; lines of n points (the adjoint's grid passes)
// P = 16 for powers of two, else 24.  A workgroup of NT = nt_of<N, P>() lanes
// holds NT / T lines (T = N / P), each with one LDS row; the twiddle table
// follows them.  Each kernel computes the same quantities as its generic
// counterpart (same index maps; FP32 sums in a different order).
//
// The centred index maps become register rotations: the rotated FFT position
// a = t + T m of an input at centred index c = a + N/2 (mod N) is
// c = t + T ((m + P/2) mod P), and output position b = t + T m is centred
// frequency b (m < P/2) or b - N (m >= P/2).  Of the N points of a detector
// line, the n = 2N/3 pixels are m in [2P/3, P) and [0, P/3) in the rotated order.
constexpr int kNT = kLineThreads;
// lanes of a workgroup: 2 T C with C, the columns of a column tile, the
// largest power of two that fits kNT (T = 16: 256 lanes; T = 6, 12: 192)
template <int N, int P = kLineP>
constexpr int nt_of() {
  constexpr int T = LineReg<N, P>::T;
  int c = 1;
  while (4 * T * c <= kNT) c *= 2;
  return 2 * T * c;
}
// points per lane of the adjoint's n-point lines
template <int n>
constexpr int pa_of() { return n % 3 == 0 ? 24 : 16; }
template <int N>
__device__ __forceinline__ void stage_twiddles(float2* twl, const float2* __restrict__ tw) {
  for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = tw[i];
}
template <int N, int P = kLineP>
constexpr size_t reg_lds_bytes() {
  return sizeof(float2) * ((size_t)(nt_of<N, P>() / LineReg<N, P>::T) * (N + 1) + N);
}

// forward row pass: rows q of slice pair z, lines (r, parity, slice); lane =
// slice + 2 (par + 2 (t + T r))
template <int N>
__global__ __launch_bounds__(kNT) void k_row_fwd_r(float2* __restrict__ A,
                                                   const float2* __restrict__ u,
                                                   const float2* __restrict__ tw,
                                                   const float2* __restrict__ twist,
                                                   const float* __restrict__ dphi,
                                                   const int2* __restrict__ mrange, int n,
                                                   int pz) {
  constexpr int P = kLineP, H = P / 2, T = LineReg<N>::T, NL = nt_of<N>() / T, ROWS = NL / 4,
                o = N / 6;
  extern __shared__ float2 lds[];
  float2* twl = lds + NL * (N + 1);
  stage_twiddles<N>(twl, tw);
  const int tid = threadIdx.x, zz = tid & 1, par = (tid >> 1) & 1, t = (tid >> 2) % T,
            r = tid / (4 * T);
  const int z = min(2 * (int)blockIdx.y + zz, pz - 1), q = blockIdx.x * ROWS + r;
  const bool rowok = q < N;
  const int2 mr = rowok ? mrange[q] : make_int2(0, 0);
  const float dq = rowok ? dphi[q] : 0.f;
  const float2* ur = u + ((long)z * n + min(max(q - o, 0), n - 1)) * n;
  // all P loads unconditional (clamped indices) and in flight together; the
  // circ mask and the parity select afterwards
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    v[m] = ur[min(max(t + T * ((m + H) % P) - o, 0), n - 1)];
  });
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int c = t + T * ((m + H) % P);
    const float2 x = cscale(v[m], dq * dphi[c]);
    const float2 xt = cmul(x, twist[c]);
    v[m] = (c >= mr.x && c < mr.y) ? (par ? xt : x) : make_float2(0.f, 0.f);
  });
  __syncthreads();
  line_reg_fft<N, -1>(v, lds + (4 * r + 2 * zz + par) * (N + 1), twl, t);
  if (!rowok) return;
  float2* Ar = A + ((long)blockIdx.y * N + q) * (4 * N) + 2 * par + zz;
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int b = t + T * m;
    Ar[2 * (m < H ? 2 * b + N : 2 * b - N)] = v[m];
  });
}

// forward column pass: C = NT / (2T) of the 4N columns (kx, slice) of slice
// pair z, lines (par C + cc); lane = cc + C (par + 2 t)
template <int N>
__global__ __launch_bounds__(kNT) void k_col_fwd_r(float2* __restrict__ Bg,
                                                   const float2* __restrict__ A,
                                                   const float2* __restrict__ tw,
                                                   const float2* __restrict__ twist) {
  constexpr int P = kLineP, H = P / 2, T = LineReg<N>::T, C = nt_of<N>() / (2 * T), W = 4 * N,
                gx = W / C;
  static_assert(W % C == 0, "column tiles");
  extern __shared__ float2 lds[];
  float2* twl = lds + 2 * C * (N + 1);
  stage_twiddles<N>(twl, tw);
  const int tid = threadIdx.x, cc = tid % C, par = (tid / C) & 1, t = tid / (2 * C);
  const int L = xcd_contig(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int z = L / gx, k0 = (L - z * gx) * C;
  const float2* Az = A + (long)z * N * W + k0 + cc;
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    v[m] = Az[(long)(t + T * ((m + H) % P)) * W];
  });
  if (par) {
    static_for<0, P>([&](auto mc) {
      constexpr int m = decltype(mc)::value;
      v[m] = cmul(v[m], twist[t + T * ((m + H) % P)]);
    });
  }
  __syncthreads();
  line_reg_fft<N, -1>(v, lds + (par * C + cc) * (N + 1), twl, t);
  float2* Bz = Bg + (long)z * (2 * N) * W + k0 + cc;
  const int ym = disc_rows(((k0 + cc) >> 1) - N, N);
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int b = t + T * m, ky = (m < H ? 2 * b : 2 * b - 2 * N) + par;
    if (m < H ? ky <= ym : -ky <= ym) Bz[(long)(ky + N) * W] = v[m];
  });
}

// forward detector lines: ZQ = NT / T slices of angle th; lane = zz%2 + 2 (t + T (zz/2))
template <int N>
__global__ __launch_bounds__(kNT) void k_line_idft_r(float2* __restrict__ g,
                                                     const float2* __restrict__ G,
                                                     const float2* __restrict__ tw, float oscale,
                                                     int ntheta, int pz) {
  constexpr int P = kLineP, H = P / 2, P3 = P / 3, T = LineReg<N>::T, ZQ = nt_of<N>() / T,
                n = 2 * N / 3;
  extern __shared__ float2 lds[];
  float2* twl = lds + ZQ * (N + 1);
  stage_twiddles<N>(twl, tw);
  const int tid = threadIdx.x, t = (tid >> 1) % T, zz = 2 * (tid / (2 * T)) + (tid & 1);
  const int th = blockIdx.x, z = blockIdx.y * ZQ + zz, zc = min(z, pz - 1);
  const bool ok = z < pz;
  const float2* Gl = G + (((long)(zc >> 1) * ntheta + th) * N) * 2 + (zc & 1);
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    v[m] = Gl[2 * (t + T * ((m + H) % P))];  // row clamped: a lane past pz transforms a copy
  });
  __syncthreads();
  line_reg_fft<N, 1>(v, lds + zz * (N + 1), twl, t);
  if (!ok) return;
  // detector pixel j: position j - n/2 (mod N); m in [P/3, 2P/3) lies outside
  float2* gl = g + ((long)th * pz + z) * n;
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    if constexpr (m < P3) gl[t + T * (m + P3)] = cscale(v[m], oscale);
    else if constexpr (m >= 2 * P3) gl[t + T * (m - 2 * P3)] = cscale(v[m], oscale);
  });
}

// adjoint detector lines: ZQ slices of angle th; lane = zz + ZQ t (z fastest
// for the Q[sample][z] stores)
template <int N>
__global__ __launch_bounds__(kNT) void k_adj_line_r(float2* __restrict__ Q,
                                                    const float2* __restrict__ g,
                                                    const float2* __restrict__ tw,
                                                    const float* __restrict__ filt, float oscale,
                                                    int ntheta, int pz, int pzs) {
  constexpr int P = kLineP, H = P / 2, T = LineReg<N>::T, ZQ = nt_of<N>() / T, n = 2 * N / 3,
                o = N / 6;
  extern __shared__ float2 lds[];
  float2* twl = lds + ZQ * (N + 1);
  stage_twiddles<N>(twl, tw);
  const int tid = threadIdx.x, zz = tid % ZQ, t = tid / ZQ;
  const int th = blockIdx.x, z = blockIdx.y * ZQ + zz;
  const bool ok = z < pz;
  const float2* gl = g + ((long)th * pz + min(z, pz - 1)) * n;
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int s = t + T * ((m + H) % P);  // padded detector index (kernels.cuh:189-206)
    v[m] = gl[min(max(s - o, 0), n - 1)];  // row clamped: a lane past pz transforms a copy
  });
  __syncthreads();
  line_reg_fft<N, -1>(v, lds + zz * (N + 1), twl, t);
  if (z >= pzs) return;
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int i = t + T * ((m + H) % P);  // sample index along the line
    const float w = filt ? oscale * filt[i] : oscale;
    Q[((long)th * N + i) * pzs + z] = cscale(v[m], ok ? w : 0.f);
  });
}

// Parity halves of an adjoint 2n-point line: the even (par 0) and odd (par 1)
// inverse DFTs of one output line sit in partner lanes (lane ^ pm).  Output
// positions m in [0, P/2) are finished by the par 0 lane, the others by the
// par 1 lane; each lane sends the P/2 values its partner needs.
template <int P>
__device__ __forceinline__ void parity_swap(const float2 (&v)[P], int par, int pm,
                                            float2 (&E)[P / 2], float2 (&O)[P / 2]) {
  static_for<0, P / 2>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    const float2 s = par ? v[k] : v[P / 2 + k];
    float2 r;
    r.x = __shfl_xor(s.x, pm, 64);
    r.y = __shfl_xor(s.y, pm, 64);
    E[k] = par ? r : v[k];
    O[k] = par ? v[P / 2 + k] : r;
  });
}

// adjoint column pass: C of the 4n columns (kx, slice) of slice pair z, lines
// (par C + cc); lane = cc + C (par + 2 t)
template <int n>
__global__ __launch_bounds__(kNT) void k_col_adj_r(float2* __restrict__ A,
                                                   const float2* __restrict__ Bg,
                                                   const float2* __restrict__ tw,
                                                   const float2* __restrict__ twist) {
  constexpr int P = pa_of<n>(), H = P / 2, T = LineReg<n, P>::T, C = nt_of<n, P>() / (2 * T),
                W = 4 * n, gx = W / C;
  static_assert(W % C == 0, "column tiles");
  static_assert(C <= 32 && (C & (C - 1)) == 0, "parity partner lane ^ C in the same wavefront");
  extern __shared__ float2 lds[];
  float2* twl = lds + 2 * C * (n + 1);
  stage_twiddles<n>(twl, tw);
  const int tid = threadIdx.x, cc = tid % C, par = (tid / C) & 1, t = tid / (2 * C);
  const int L = xcd_contig(blockIdx.x + gx * blockIdx.y, gx * gridDim.y);
  const int z = L / gx, k0 = (L - z * gx) * C;
  const float2* Bz = Bg + (long)z * (2 * n) * W + k0 + cc;
  const int ym = disc_rows(((k0 + cc) >> 1) - n, n);
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int b = t + T * m, ky = (m < H ? 2 * b : 2 * b - 2 * n) + par;
    const bool in = m < H ? ky <= ym : -ky <= ym;
    v[m] = Bz[(long)(in ? ky + n : n) * W];  // outside: a point of the centre row
    if (!in) v[m] = make_float2(0.f, 0.f);
  });
  __syncthreads();
  line_reg_fft<n, 1>(v, lds + (par * C + cc) * (n + 1), twl, t);
  float2 E[H], O[H];
  parity_swap<P>(v, par, C, E, O);
  float2* Az = A + (long)z * n * W + k0 + cc;
  static_for<0, H>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    const int q = t + T * (par ? k : k + H);  // object row: rotated position q - n/2
    Az[(long)q * W] = cadd(E[k], cmulc(O[k], twist[q]));
  });
}

// adjoint row pass: object rows q of slice pair z, lines (r, slice, parity);
// lane = slice + 2 (par + 2 (t + T r))
template <int n>
__global__ __launch_bounds__(kNT) void k_row_adj_r(float2* __restrict__ f,
                                                   const float2* __restrict__ A,
                                                   const float2* __restrict__ tw,
                                                   const float2* __restrict__ twist,
                                                   const float* __restrict__ dphi,
                                                   const int2* __restrict__ mrange, float scale,
                                                   int pz) {
  constexpr int P = pa_of<n>(), H = P / 2, T = LineReg<n, P>::T, NL = nt_of<n, P>() / T,
                ROWS = NL / 4, o = n / 4;
  static_assert(n % ROWS == 0, "whole row tiles");
  extern __shared__ float2 lds[];
  float2* twl = lds + NL * (n + 1);
  stage_twiddles<n>(twl, tw);
  const int tid = threadIdx.x, zz = tid & 1, par = (tid >> 1) & 1, t = (tid >> 2) % T,
            r = tid / (4 * T);
  const int q = blockIdx.x * ROWS + r, z = 2 * blockIdx.y + zz;
  const float2* Ar = A + ((long)blockIdx.y * n + q) * (4 * n) + 2 * par + zz;
  float2 v[P];
  static_for<0, P>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    const int b = t + T * m;
    v[m] = Ar[2 * (m < H ? 2 * b + n : 2 * b - n)];
  });
  __syncthreads();
  line_reg_fft<n, 1>(v, lds + (4 * r + 2 * zz + par) * (n + 1), twl, t);
  float2 E[H], O[H];
  parity_swap<P>(v, par, 2, E, O);
  if (z >= pz) return;
  const int2 mr = mrange[q + o];
  const float dq = dphi[q];
  float2* fr = f + ((long)z * n + q) * n;
  static_for<0, H>([&](auto kc) {
    constexpr int k = decltype(kc)::value;
    const int p = t + T * (par ? k : k + H);  // object column: rotated position p - n/2
    const float w = (p + o >= mr.x && p + o < mr.y) ? dq * dphi[p] * scale : 0.f;
    fr[p] = cscale(cadd(E[k], cmulc(O[k], twist[p])), w);
  });
}

// ------------------------------------------------------------------ host helpers
// LDS of a line kernel: nl padded lines, their ping-pong partners and the
// twiddle table
size_t line_lds_bytes(int N, int nl) { return sizeof(float2) * (2 * (size_t)nl * (N + 1) + N); }
// LDS of a column kernel: C padded lines, their partners and the twiddle table
size_t col_lds_bytes(int N, int C) { return sizeof(float2) * (2 * (size_t)C * (N + 1) + N); }
constexpr size_t kLdsCap = 64 * 1024;

int lines_fit(const LinePlan& p, int maxlines, size_t lds_cap) {
  int best = 1;
  for (int l = 1; l <= maxlines; ++l) {
    if (line_lds_bytes(p.N, l) > lds_cap) break;
    best = l;
  }
  return best;
}

// C columns per workgroup of the column passes: a power of two whose tile
// fits the per-thread registers and the LDS
bool col_fits(const LinePlan& p, int C) {
  if (C < 1 || (C & (C - 1))) return false;
  return (long)p.N * C <= 256L * kColVpt && col_lds_bytes(p.N, C) <= kLdsCap;
}
int ilog2(int c) {
  int l = 0;
  while ((1 << l) < c) ++l;
  return l;
}

// the register line passes serve N = 96, 144, 192, 288, 384, 768 (n = 64, 96, 128, 192,
// 256, 512)
bool reg_lines(const pt_tomo* h) {
  const int N = h->N;
  return h->line_kind == PT_LINES_AUTO && (N == 96 || N == 144 || N == 192 || N == 288 ||
                                           N == 384 || N == 768);
}
template <class F>
int with_reg_n(int N, F&& fn) {
  switch (N) {
    case 96: return fn(ic<96>{});
    case 144: return fn(ic<144>{});
    case 192: return fn(ic<192>{});
    case 288: return fn(ic<288>{});
    case 384: return fn(ic<384>{});
    default: return fn(ic<768>{});
  }
}

template <int N>
int fwd_grid_r(pt_tomo* h, const float2* f, hipStream_t st) {
  constexpr int T = LineReg<N>::T, ROWS = nt_of<N>() / (4 * T), C = nt_of<N>() / (2 * T);
  constexpr size_t lds = reg_lds_bytes<N>();
  const int npair = (h->pz + 1) / 2;
  {
    ProfScope prof("tomo_row_fwd", st);
    hipLaunchKernelGGL(k_row_fwd_r<N>, dim3((N + ROWS - 1) / ROWS, npair), dim3(nt_of<N>()), lds,
                       st, h->A, f, h->tw, h->twist, h->dphi, h->mrange, h->n, h->pz);
    PT_LAUNCH_CHECK();
  }
  {
    ProfScope prof("tomo_col_fwd", st);
    hipLaunchKernelGGL(k_col_fwd_r<N>, dim3(4 * N / C, npair), dim3(nt_of<N>()), lds, st, h->Bg, h->A,
                       h->tw, h->twist);
    PT_LAUNCH_CHECK();
  }
  return PT_OK;
}

template <int N>
int fwd_lines_r(pt_tomo* h, float2* g, float oscale, hipStream_t st) {
  constexpr int ZQ = nt_of<N>() / LineReg<N>::T;
  ProfScope prof("tomo_line_idft", st);
  hipLaunchKernelGGL(k_line_idft_r<N>, dim3(h->ntheta, (h->pz + ZQ - 1) / ZQ), dim3(nt_of<N>()),
                     reg_lds_bytes<N>(), st, g, h->Q, h->tw, oscale, h->ntheta, h->pz);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

template <int N>
int adj_lines_r(pt_tomo* h, const float2* g, float oscale, hipStream_t st) {
  constexpr int ZQ = nt_of<N>() / LineReg<N>::T;
  ProfScope prof("tomo_adj_line", st);
  hipLaunchKernelGGL(k_adj_line_r<N>, dim3(h->ntheta, (h->pzs + ZQ - 1) / ZQ), dim3(nt_of<N>()),
                     reg_lds_bytes<N>(), st, h->Q, g, h->tw, h->filt, oscale, h->ntheta, h->pz,
                     h->pzs);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

template <int N>
int adj_grid_r(pt_tomo* h, float2* f, float scale, hipStream_t st) {
  constexpr int n = 2 * N / 3, P = pa_of<n>(), T = LineReg<n, P>::T, NT = nt_of<n, P>(),
                ROWS = NT / (4 * T), C = NT / (2 * T);
  constexpr size_t lds = reg_lds_bytes<n, P>();
  const int npair = (h->pz + 1) / 2;
  {
    ProfScope prof("tomo_col_adj", st);
    hipLaunchKernelGGL(k_col_adj_r<n>, dim3(4 * n / C, npair), dim3(NT), lds, st, h->A, h->Bg,
                       h->twn, h->twistn);
    PT_LAUNCH_CHECK();
  }
  {
    ProfScope prof("tomo_row_adj", st);
    hipLaunchKernelGGL(k_row_adj_r<n>, dim3(n / ROWS, npair), dim3(NT), lds, st, f, h->A, h->twn,
                       h->twistn, h->dphia, h->mrange, scale, h->pz);
    PT_LAUNCH_CHECK();
  }
  return PT_OK;
}

template <int ZB>
int scatter(pt_tomo* h, hipStream_t st) {
  ProfScope prof("tomo_scatter", st);
  hipLaunchKernelGGL(k_scatter_own<ZB>, dim3(h->nswi, (h->pzs / 8 + ZB - 1) / ZB), dim3(64), 0, st,
                     (f4m*)h->Bg, (f4m*)h->spart, (const float*)h->Q, (const f4m*)h->wadj, h->ent,
                     h->swi_tile, h->swi_range, h->swi_slot, h->nts, h->pzs);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

int run_fwd(pt_tomo* h, float2* g, const float2* f, float scale, hipStream_t st) {
  const int N = h->N, npair = (h->pz + 1) / 2;
  const int nthr = 256;
  const bool rl = reg_lines(h);
  if (rl) {
    const int rc = with_reg_n(N, [&](auto nc) { return fwd_grid_r<decltype(nc)::value>(h, f, st); });
    if (rc) return rc;
  }
  if (!rl) {
    const int rows = h->rows_per_wg;
    dim3 grid((2 * N + rows - 1) / rows, npair);
    size_t lds = line_lds_bytes(N, 2 * rows);
    ProfScope prof("tomo_row_fwd", st);
    hipLaunchKernelGGL(k_row_fwd, grid, dim3(nthr), lds, st, h->A, f, h->tw, h->twist, h->dphi,
                       h->mrange, h->plan, h->n, rows, h->pz);
    PT_LAUNCH_CHECK();
  }
  if (!rl) {
    const int cols = h->cols_per_wg;
    dim3 grid((4 * N + cols - 1) / cols, npair);
    ProfScope prof("tomo_col_fwd", st);
    hipLaunchKernelGGL(k_col_fwd, grid, dim3(nthr), col_lds_bytes(N, cols), st, h->Bg, h->A, h->tw,
                       h->twist, h->plan, ilog2(cols));
    PT_LAUNCH_CHECK();
  }
  {
    // slice pairs per workgroup: up to 8, so that the next pair's loads overlap
    // the interpolation, but fewer where that leaves under 2048 workgroups
    // (8 per CU)
    int zper = 8;
    while (zper > 1 && (long)h->nwi * ((npair + zper - 1) / zper) < 2048) zper /= 2;
    dim3 grid(h->nwi, (npair + zper - 1) / zper);
    ProfScope prof("tomo_gather", st);
    hipLaunchKernelGGL(k_gather_tile, grid, dim3(kWorkMax), 0, st, (f4v*)h->Q, (const f4v*)h->Bg,
                       (const f4v*)h->wfwd, h->sfloor, h->wi_tile, h->wi_range, h->bin_sample, N,
                       h->ntile1, h->ntheta * N, npair, zper);
    PT_LAUNCH_CHECK();
  }
  {
    const double sgn = ((N / 2) % 2) ? -1.0 : 1.0;
    const float oscale = (float)(sgn / (double)N * (double)scale);
    if (rl) return with_reg_n(N, [&](auto nc) { return fwd_lines_r<decltype(nc)::value>(h, g, oscale, st); });
    const int zq = h->adj_lines;    // detector lines per workgroup (fits the LDS FFT)
    dim3 grid(h->ntheta, (h->pz + zq - 1) / zq);
    ProfScope prof("tomo_line_idft", st);
    hipLaunchKernelGGL(k_line_idft, grid, dim3(256), line_lds_bytes(N, zq), st, g, h->Q,
                       h->tw, h->plan, oscale, h->n, h->ntheta, h->pz, zq);
    PT_LAUNCH_CHECK();
  }
  return PT_OK;
}

int run_adj(pt_tomo* h, float2* f, const float2* g, float scale, hipStream_t st) {
  const int N = h->N, npair = (h->pz + 1) / 2;
  const bool rl = reg_lines(h);
  const double sgn = ((N / 2) % 2) ? -1.0 : 1.0;
  const float oscale = (float)(sgn / (double)N);
  if (rl) {
    const int rc = with_reg_n(N, [&](auto nc) { return adj_lines_r<decltype(nc)::value>(h, g, oscale, st); });
    if (rc) return rc;
  } else {
    const int zq = h->adj_lines;
    dim3 grid(h->ntheta, (h->pzs + zq - 1) / zq);
    ProfScope prof("tomo_adj_line", st);
    hipLaunchKernelGGL(k_adj_line, grid, dim3(256), line_lds_bytes(N, zq), st, h->Q, g, h->tw,
                       h->filt, h->plan, oscale, h->n, h->ntheta, h->pz, h->pzs, zq);
    PT_LAUNCH_CHECK();
  }
  {
    const int rc = h->szb == 4 ? scatter<4>(h, st) : h->szb == 2 ? scatter<2>(h, st)
                                                                  : scatter<1>(h, st);
    if (rc) return rc;
    if (h->nfix) {
      ProfScope prof("tomo_scatter_fix", st);
      hipLaunchKernelGGL(k_scatter_fix, dim3(h->nfix, npair), dim3(kTS * kTS), 0, st,
                         (f4m*)h->Bg, (const f4m*)h->spart, h->sfix, h->nts, h->pzs / 2);
      PT_LAUNCH_CHECK();
    }
  }
  if (rl) return with_reg_n(N, [&](auto nc) { return adj_grid_r<decltype(nc)::value>(h, f, scale, st); });
  {
    const int cols = h->cols_per_wg;
    dim3 grid((4 * h->n + cols - 1) / cols, npair);
    ProfScope prof("tomo_col_adj", st);
    hipLaunchKernelGGL(k_col_adj, grid, dim3(256), col_lds_bytes(h->n, cols), st, h->A, h->Bg,
                       h->twn, h->twistn, h->plann, ilog2(cols));
    PT_LAUNCH_CHECK();
  }
  {
    const int rows = h->rows_per_wg;
    dim3 grid((2 * h->n + rows - 1) / rows, npair);
    ProfScope prof("tomo_row_adj", st);
    hipLaunchKernelGGL(k_row_adj, grid, dim3(256), line_lds_bytes(h->n, 2 * rows), st, f, h->A,
                       h->twn, h->twistn, h->dphia, h->mrange, h->plann, rows, scale, h->pz);
    PT_LAUNCH_CHECK();
  }
  return PT_OK;
}

}  // namespace

bool make_line_plan(int N, LinePlan* p) {
  p->N = N;
  p->npass = 0;
  int rem = N;
  // prefer radix 8, then 4, then 2; odd radices 3 and 5
  const int order[] = {8, 4, 2, 3, 5};
  // take odd factors first so that power-of-two passes come last
  for (int r : {3, 5}) {
    while (rem % r == 0) {
      if (p->npass >= 12) return false;
      p->radix[p->npass++] = r;
      rem /= r;
    }
  }
  (void)order;
  while (rem > 1) {
    int r = (rem % 8 == 0 && rem != 16) ? 8 : (rem % 4 == 0 ? 4 : (rem % 2 == 0 ? 2 : 0));
    if (!r || p->npass >= 12) return false;
    p->radix[p->npass++] = r;
    rem /= r;
  }
  int Ns = 1;
  for (int i = 0; i < p->npass; ++i) {
    p->dnb[i] = make_divc((unsigned)(N / p->radix[i]));
    p->dns[i] = make_divc((unsigned)Ns);
    Ns *= p->radix[i];
  }
  return true;
}

}  // namespace pt

using namespace pt;

extern "C" int pt_tomo_create(int ntheta, int pnz, int n, pt_tomo** out) {
  PT_REQUIRE(out, PT_ERR_ARG, "pt_tomo_create: null output handle");
  *out = nullptr;
  PT_REQUIRE(ntheta > 0 && pnz > 0 && n > 0, PT_ERR_SIZE, "pt_tomo_create: sizes must be positive");
  PT_REQUIRE(n % 4 == 0, PT_ERR_SIZE, "pt_tomo_create: n must be a multiple of 4");
  const int N = n * 3 / 2;
  LinePlan plan;
  PT_REQUIRE(make_line_plan(N, &plan), PT_ERR_SIZE,
             "pt_tomo_create: 3n/2 must factor into radices 2, 3, 4, 5, 8");
  PT_REQUIRE(line_lds_bytes(N, 2) <= kLdsCap && col_fits(plan, 1), PT_ERR_SIZE,
             "pt_tomo_create: n too large");
  pt_tomo* h = new pt_tomo();
  h->ntheta = ntheta; h->pz = pnz; h->pzs = (pnz + 7) / 8 * 8; h->n = n; h->N = N;
  h->plan = plan;
  make_line_plan(n, &h->plann);  // n = 2/3 N factors as N does
  // LDS lines per workgroup of the row and detector-line passes (<= 48 KB);
  // columns per workgroup of the column passes (up to 16: whole cache lines)
  const size_t cap = 48 * 1024;
  int lines = lines_fit(plan, 16, cap);
  h->rows_per_wg = std::max(1, lines / 2);
  int cols = 16;
  while (cols > 1 && !col_fits(plan, cols)) cols /= 2;
  h->cols_per_wg = cols;
  h->adj_lines = lines_fit(plan, kZQ, cap);
  // host tables
  auto line_tables = [](int L, std::vector<float2>& tw, std::vector<float2>& twist,
                        std::vector<float>& dphi) {
    tw.resize(L); twist.resize(L); dphi.resize(L);
    for (int m = 0; m < L; ++m) {
      const int j = m - L / 2;
      const double a = -2.0 * kPi * m / L, b = -kPi * j / L;
      tw[m] = make_float2((float)std::cos(a), (float)std::sin(a));
      twist[m] = make_float2((float)std::cos(b), (float)std::sin(b));
      dphi[m] = (float)kb_inverse_ft((double)j / (2.0 * L));
    }
  };
  std::vector<float2> tw, twist, twn, twistn;
  std::vector<float> dphi, dphia;
  std::vector<int2> mr(N);
  line_tables(N, tw, twist, dphi);
  line_tables(n, twn, twistn, dphia);
  // circ mask (kernels.cuh:160-172), float32 arithmetic without contraction
  for (int q = 0; q < N; ++q) {
    volatile float y = (float)(q - N / 2) / (float)N;
    volatile float yy = 4.0f * y;
    yy = yy * y;
    volatile float thr = 1.0f - 1.0f / (float)N;
    int lo = N, hi = 0;
    for (int c = 0; c < N; ++c) {
      volatile float x = (float)(c - N / 2) / (float)N;
      volatile float xx = 4.0f * x;
      xx = xx * x;
      volatile float v = xx + yy;
      if (v < thr) {
        lo = std::min(lo, c);
        hi = std::max(hi, c + 1);
      }
    }
    if (lo >= hi) lo = hi = 0;
    mr[q] = make_int2(lo, hi);
  }
  auto fail = [&](hipError_t e, const char* what) {
    set_error(std::string("pt_tomo_create: ") + what + ": " + hipGetErrorString(e));
    pt_tomo_destroy(h);
    return PT_ERR_HIP;
  };
  hipError_t e;
  const size_t ns = (size_t)ntheta * N;
  if ((e = hipMalloc(&h->tw, sizeof(float2) * N))) return fail(e, "tables");
  if ((e = hipMalloc(&h->twist, sizeof(float2) * N))) return fail(e, "tables");
  if ((e = hipMalloc(&h->twn, sizeof(float2) * n))) return fail(e, "tables");
  if ((e = hipMalloc(&h->twistn, sizeof(float2) * n))) return fail(e, "tables");
  if ((e = hipMalloc(&h->dphi, sizeof(float) * N))) return fail(e, "tables");
  if ((e = hipMalloc(&h->dphia, sizeof(float) * n))) return fail(e, "tables");
  if ((e = hipMalloc(&h->mrange, sizeof(int2) * N))) return fail(e, "tables");
  if ((e = hipMalloc(&h->spos, sizeof(float2) * ns))) return fail(e, "positions");
  if ((e = hipMalloc(&h->sfloor, sizeof(int2) * ns))) return fail(e, "positions");
  if ((e = hipMalloc(&h->bin_sample, sizeof(int) * ns))) return fail(e, "bins");
  if ((e = hipMalloc(&h->wfwd, sizeof(float) * 2 * kW * ns))) return fail(e, "weights");
  if ((e = hipMalloc(&h->wadj, sizeof(float) * 2 * kW * ns))) return fail(e, "weights");
  // the adjoint's 2n x 2n grid in blocks of 8 slices, the forward's 2N x 2N in pairs
  const size_t pzp = (size_t)(pnz + 1) / 2 * 2, pzs = h->pzs;
  if ((e = hipMalloc(&h->A, sizeof(float2) * pzp * N * 2 * N))) return fail(e, "row buffer");
  if ((e = hipMalloc(&h->Bg, sizeof(float2) * std::max(pzp * 4 * N * N, pzs * 4 * n * n))))
    return fail(e, "grid");
  if ((e = hipMalloc(&h->Q, sizeof(float2) * pzs * ns))) return fail(e, "samples");
  if ((e = hipMemcpy(h->tw, tw.data(), sizeof(float2) * N, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->twist, twist.data(), sizeof(float2) * N, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->twn, twn.data(), sizeof(float2) * n, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->twistn, twistn.data(), sizeof(float2) * n, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->dphi, dphi.data(), sizeof(float) * N, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->dphia, dphia.data(), sizeof(float) * n, hipMemcpyHostToDevice))) return fail(e, "copy");
  if ((e = hipMemcpy(h->mrange, mr.data(), sizeof(int2) * N, hipMemcpyHostToDevice))) return fail(e, "copy");
  *out = h;
  return PT_OK;
}

static void free_bins(pt_tomo* h) {
  void** ptrs[] = {(void**)&h->wi_tile, (void**)&h->wi_range, (void**)&h->ent,
                   (void**)&h->swi_tile, (void**)&h->swi_range,
                   (void**)&h->swi_slot, (void**)&h->sfix, (void**)&h->spart};
  for (void** p : ptrs) {
    if (*p) (void)hipFree(*p);
    *p = nullptr;
  }
  h->nwi = h->nswi = h->nfix = 0;
}

template <typename T>
static int upload(T** dst, const std::vector<T>& v, hipStream_t st) {
  PT_HIP(hipMalloc(dst, sizeof(T) * std::max<size_t>(v.size(), 1)));
  if (!v.empty()) PT_HIP(hipMemcpyAsync(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice, st));
  return PT_OK;
}

extern "C" int pt_tomo_destroy(pt_tomo* h) {
  if (!h) return PT_OK;
  void* ptrs[] = {h->tw, h->twist, h->twn, h->twistn, h->dphi, h->dphia, h->filt, h->mrange,
                  h->spos, h->sfloor, h->wfwd, h->wadj, h->A, h->Bg, h->Q};
  for (void* p : ptrs) (void)hipFree(p);
  (void)hipFree(h->bin_sample);
  free_bins(h);
  delete h;
  return PT_OK;
}

extern "C" int pt_tomo_set_theta(pt_tomo* h, const float* theta, pt_stream stream) {
  PT_REQUIRE(h && theta, PT_ERR_ARG, "pt_tomo_set_theta: null argument");
  hipStream_t st = (hipStream_t)stream;
  const int N = h->N, nt = h->ntheta;
  std::vector<float> th(nt);
  PT_HIP(hipMemcpyAsync(th.data(), theta, sizeof(float) * nt, hipMemcpyDeviceToHost, st));
  PT_HIP(hipStreamSynchronize(st));
  // takexy (kernels.cuh:84-95): FP64 then float32, clamp at 0.5
  const long ns = (long)nt * N;
  std::vector<float2> pos(ns);
  std::vector<int2> ff(ns);  // exact floors, as the weights' (k_kb_weights)
  const float lim = (float)(0.5 - 1e-5);
  for (int t = 0; t < nt; ++t) {
    const double c = std::cos((double)th[t]), s = std::sin((double)th[t]);
    for (int i = 0; i < N; ++i) {
      const double k = (double)(i - N / 2);
      float x = (float)(k / N * c);
      float y = (float)(-k / N * s);
      if (x >= 0.5f) x = lim;
      if (y >= 0.5f) y = lim;
      pos[(long)t * N + i] = make_float2(x, y);
      ff[(long)t * N + i] =
          make_int2((int)std::floor(2.0 * N * x), (int)std::floor(2.0 * N * y));
    }
  }
  for (long q = 0; q < ns; ++q) {
    if (ff[q].x < -N || ff[q].x >= N || ff[q].y < -N || ff[q].y >= N) {
      set_error("pt_tomo_set_theta: sample outside the gridding domain");
      return PT_ERR_ARG;
    }
  }
  const int twoNi = 2 * N;
  // gather bins: samples by kTile x kTile tile of their floor position,
  // chunks of at most kWorkMax samples
  const int nt1 = (twoNi + kTile - 1) / kTile;
  const long ntiles = (long)nt1 * nt1;
  std::vector<int> cnt(ntiles + 1, 0);
  for (long q = 0; q < ns; ++q)
    cnt[(long)((ff[q].y + N) / kTile) * nt1 + (ff[q].x + N) / kTile + 1]++;
  for (long i = 0; i < ntiles; ++i) cnt[i + 1] += cnt[i];
  std::vector<int> fillp(cnt.begin(), cnt.end() - 1), list(ns);
  for (long q = 0; q < ns; ++q)
    list[fillp[(long)((ff[q].y + N) / kTile) * nt1 + (ff[q].x + N) / kTile]++] = (int)q;
  // within a bin, samples in row-major order of their floor position: the
  // lanes of a wavefront then read neighbouring LDS words for each tap (few
  // bank conflicts); each lane still computes its own sample, so the order
  // does not change any result
  for (long tI = 0; tI < ntiles; ++tI)
    std::sort(list.begin() + cnt[tI], list.begin() + cnt[tI + 1], [&](int a, int b) {
      if (ff[a].y != ff[b].y) return ff[a].y < ff[b].y;
      if (ff[a].x != ff[b].x) return ff[a].x < ff[b].x;
      return a < b;
    });
  std::vector<int> wtile;
  std::vector<int2> wrange;
  // Within each work item, samples dealt round-robin over the 16 classes of
  // their footprint origin's LDS address mod 16 float4 (64 banks of 4 B).
  // Every tap reads at the same offset from each lane's origin, so 16
  // consecutive lanes then fall on distinct banks for all taps (8 consecutive
  // lanes on distinct 32-bank sets).  Row-major order put neighbouring lanes a
  // few float4 apart, i.e. on overlapping banks.  Each lane still computes its
  // own samples, so the order changes no result.
  std::vector<int> bucket[16];
  for (long tI = 0; tI < ntiles; ++tI)
    for (int s0 = cnt[tI]; s0 < cnt[tI + 1]; s0 += kWorkMax) {
      const int s1 = std::min(s0 + kWorkMax, cnt[tI + 1]);
      const int ty0 = (int)(tI / nt1) * kTile - N, tx0 = (int)(tI % nt1) * kTile - N;
      for (auto& b : bucket) b.clear();
      for (int i = s0; i < s1; ++i) {
        const int2 f = ff[list[i]];
        bucket[((f.y - ty0) * kGE + (f.x - tx0)) & 15].push_back(list[i]);
      }
      int at = s0;
      for (size_t r = 0; at < s1; ++r)
        for (auto& b : bucket)
          if (r < b.size()) list[at++] = b[r];
      wtile.push_back((int)tI);
      wrange.push_back(make_int2(s0, s1));
    }
  // scatter lists: for every 8 x 8 tile of the 2n x 2n grid, the samples whose
  // 8 x 8 footprint (periodic) covers part of it, in sample order, with the
  // footprint's origin relative to the tile in [-7, 7]; along each axis a
  // footprint meets the tile of its origin and, unless aligned, the next one
  const int n = h->n, nts = 2 * n / kTS;
  const long ntl = (long)nts * nts;
  auto tiles_of = [&](float x, int* tl, int* off) {
    int org = n + (int)std::floor(2.0 * n * x) - kWLo;
    org = org < 0 ? org + 2 * n : org >= 2 * n ? org - 2 * n : org;
    tl[0] = org / kTS;
    off[0] = org - tl[0] * kTS;
    tl[1] = tl[0] + 1 == nts ? 0 : tl[0] + 1;
    off[1] = off[0] - kTS;
    return off[0] ? 2 : 1;
  };
  std::vector<int> ecnt(ntl + 1, 0);
  int tx[2], ox[2], ty[2], oy[2];
  for (long q = 0; q < ns; ++q) {
    const int nx = tiles_of(pos[q].x, tx, ox), ny = tiles_of(pos[q].y, ty, oy);
    for (int a = 0; a < ny; ++a)
      for (int b = 0; b < nx; ++b) ecnt[(long)ty[a] * nts + tx[b] + 1]++;
  }
  for (long i = 0; i < ntl; ++i) ecnt[i + 1] += ecnt[i];
  std::vector<int> efill(ecnt.begin(), ecnt.end() - 1);
  std::vector<int2> ents(ecnt[ntl]);
  for (long q = 0; q < ns; ++q) {
    const int nx = tiles_of(pos[q].x, tx, ox), ny = tiles_of(pos[q].y, ty, oy);
    for (int a = 0; a < ny; ++a)
      for (int b = 0; b < nx; ++b)
        ents[efill[(long)ty[a] * nts + tx[b]]++] =
            make_int2((int)q, (ox[b] + kTS) | (int)((unsigned)oy[a] << 8));
  }
  // Slices per work item (8 szb): as many as leave 4096 wavefronts (4 per SIMD),
  // since each staged weight and sample index then serves more products.
  // Entries per work item: at most 512, fewer in small problems, where the
  // dense tiles around the grid's centre would outlast the others; each chunk
  // beyond a tile's first is a partial to write and add.  The share of 2048 work
  // items is a compromise between the two: with 4096 the adjoint at 180^2 x 21
  // slices, 201 angles takes 88 us instead of 94 and cg_tomo at 128^3 2175 instead of
  // 2070, with 8192 that 2477, with 1024 the adjoint 104 and cg_tomo 2114.
  int szb = 4;
  while (szb > 1 && ntl * ((h->pzs / 8 + szb - 1) / szb) < 4096) szb /= 2;
  const long share = (long)ecnt[ntl] * ((h->pzs / 8 + szb - 1) / szb) / 2048;
  const int chunk = (int)std::min(512L, std::max(64L, share / kSE * kSE));
  std::vector<int> stile, sslot;
  std::vector<int2> srange;
  std::vector<int4> sfix;
  int nslots = 0;
  for (long tI = 0; tI < ntl; ++tI) {
    const int e0 = ecnt[tI], e1 = ecnt[tI + 1];
    // an empty tile wholly beyond the rows that the column pass reads
    const int tx = (int)(tI % nts) * kTS - n, ty = (int)(tI / nts) * kTS - n;
    const int dx = std::max({tx, -(tx + kTS - 1), 0}), dy = std::max({ty, -(ty + kTS - 1), 0});
    if (e0 == e1 && dy > disc_rows(dx, n)) continue;
    const int nch = std::max(1, (e1 - e0 + chunk - 1) / chunk);
    if (nch > 1) sfix.push_back(make_int4((int)tI, nslots, nch, 0));
    for (int c = 0; c < nch; ++c) {
      stile.push_back((int)tI);
      srange.push_back(make_int2(std::min(e0 + c * chunk, e1), std::min(e0 + (c + 1) * chunk, e1)));
      sslot.push_back(nch > 1 ? nslots + c : -1);
    }
    if (nch > 1) nslots += nch;
  }
  free_bins(h);
  h->ready = false;
  int rc;
  if ((rc = upload(&h->wi_tile, wtile, st)) || (rc = upload(&h->wi_range, wrange, st)) ||
      (rc = upload(&h->ent, ents, st)) || (rc = upload(&h->swi_tile, stile, st)) || (rc = upload(&h->swi_range, srange, st)) ||
      (rc = upload(&h->swi_slot, sslot, st)) || (rc = upload(&h->sfix, sfix, st)))
    return rc;
  PT_HIP(hipMalloc(&h->spart,
                   sizeof(float2) * (size_t)std::max(nslots, 1) * h->pzs * kTS * kTS));
  PT_HIP(hipMemcpyAsync(h->spos, pos.data(), sizeof(float2) * ns, hipMemcpyHostToDevice, st));
  PT_HIP(hipMemcpyAsync(h->sfloor, ff.data(), sizeof(int2) * ns, hipMemcpyHostToDevice, st));
  PT_HIP(hipMemcpyAsync(h->bin_sample, list.data(), sizeof(int) * ns, hipMemcpyHostToDevice, st));
  for (int dir = 0; dir < 2; ++dir) {
    hipLaunchKernelGGL(k_kb_weights, dim3((unsigned)((ns * 2 * kW + 255) / 256)), dim3(256), 0, st,
                       dir ? h->wadj : h->wfwd, h->spos, ns, dir ? 2 * n : 2 * N,
                       bessel_i0(kBeta));
    PT_LAUNCH_CHECK();
  }
  PT_HIP(hipStreamSynchronize(st));
  h->ntile1 = nt1;
  h->nwi = (int)wtile.size();
  h->nts = nts;
  h->szb = szb;
  h->nswi = (int)stile.size();
  h->nfix = (int)sfix.size();
  h->ready = true;
  return PT_OK;
}

static int tomo_fwd_impl(pt_tomo* h, void* g, const void* f, float scale, pt_stream stream) {
  PT_REQUIRE(h && g && f, PT_ERR_ARG, "pt_tomo_fwd: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_tomo_fwd: set_theta not called");
  return run_fwd(h, (float2*)g, (const float2*)f, scale, (hipStream_t)stream);
}
static int tomo_adj_impl(pt_tomo* h, void* f, const void* g, float scale, pt_stream stream) {
  PT_REQUIRE(h && g && f, PT_ERR_ARG, "pt_tomo_adj: null argument");
  PT_REQUIRE(h->ready, PT_ERR_STATE, "pt_tomo_adj: set_theta not called");
  return run_adj(h, (float2*)f, (const float2*)g, scale, (hipStream_t)stream);
}

extern "C" int pt_tomo_get_tuning(pt_tomo* h, int* rows, int* cols, int* adj_lines) {
  PT_REQUIRE(h && rows && cols && adj_lines, PT_ERR_ARG, "pt_tomo_get_tuning: null argument");
  *rows = h->rows_per_wg;
  *cols = h->cols_per_wg;
  *adj_lines = h->adj_lines;
  return PT_OK;
}

extern "C" int pt_tomo_set_tuning(pt_tomo* h, int rows, int cols, int adj_lines) {
  PT_REQUIRE(h, PT_ERR_ARG, "pt_tomo_set_tuning: null handle");
  const int N = h->N;
  auto ok = [&](int lines) {
    return lines >= 1 && line_lds_bytes(N, lines) <= kLdsCap;
  };
  PT_REQUIRE(ok(2 * rows), PT_ERR_SIZE, "pt_tomo_set_tuning: rows per workgroup do not fit");
  PT_REQUIRE(col_fits(h->plan, cols), PT_ERR_SIZE,
             "pt_tomo_set_tuning: columns per workgroup must be a power of two whose tile fits");
  PT_REQUIRE(ok(adj_lines) && adj_lines <= kZQ, PT_ERR_SIZE,
             "pt_tomo_set_tuning: adjoint lines per workgroup do not fit");
  h->rows_per_wg = rows;
  h->cols_per_wg = cols;
  h->adj_lines = adj_lines;
  return PT_OK;
}

extern "C" int pt_tomo_set_line_kernels(pt_tomo* h, int kind) {
  PT_REQUIRE(h, PT_ERR_ARG, "pt_tomo_set_line_kernels: null handle");
  PT_REQUIRE(kind == PT_LINES_AUTO || kind == PT_LINES_GENERIC, PT_ERR_ARG,
             "pt_tomo_set_line_kernels: unknown kind");
  h->line_kind = kind;
  return PT_OK;
}

extern "C" int pt_tomo_get_line_kernels(pt_tomo* h, int* reg) {
  PT_REQUIRE(h && reg, PT_ERR_ARG, "pt_tomo_get_line_kernels: null argument");
  *reg = reg_lines(h) ? 1 : 0;
  return PT_OK;
}

extern "C" int pt_tomo_set_filter(pt_tomo* h, int kind) {
  PT_REQUIRE(h, PT_ERR_ARG, "pt_tomo_set_filter: null handle");
  PT_REQUIRE(kind == PT_FILTER_NONE || kind == PT_FILTER_RAMP, PT_ERR_ARG,
             "pt_tomo_set_filter: unknown filter kind");
  if (kind == PT_FILTER_NONE) {
    if (h->filt) PT_HIP(hipFree(h->filt));
    h->filt = nullptr;
    return PT_OK;
  }
  // applyfilter (kernels.cuh:174-187): w = |rho| N 4 sin(rho)/rho, rho =
  // (i - N/2)/N, w = 0 at rho = 0; evaluated in FP32 as there
  const int N = h->N;
  std::vector<float> w(N);
  for (int i = 0; i < N; ++i) {
    const float rho = (float)(i - N / 2) / (float)N;
    w[i] = rho == 0.f ? 0.f : std::fabs(rho) * (float)N * 4.f * std::sin(rho) / rho;
  }
  if (!h->filt) PT_HIP(hipMalloc(&h->filt, sizeof(float) * N));
  PT_HIP(hipMemcpy(h->filt, w.data(), sizeof(float) * N, hipMemcpyHostToDevice));
  return PT_OK;
}

extern "C" int pt_tomo_fwd(pt_tomo* h, void* g, const void* f, pt_stream stream) {
  return tomo_fwd_impl(h, g, f, 1.0f, stream);
}
extern "C" int pt_tomo_adj(pt_tomo* h, void* f, const void* g, pt_stream stream) {
  return tomo_adj_impl(h, f, g, 1.0f, stream);
}
extern "C" int pt_tomo_fwd_scaled(pt_tomo* h, void* g, const void* f, float scale, pt_stream stream) {
  return tomo_fwd_impl(h, g, f, scale, stream);
}
extern "C" int pt_tomo_adj_scaled(pt_tomo* h, void* f, const void* g, float scale, pt_stream stream) {
  return tomo_adj_impl(h, f, g, scale, stream);
}
