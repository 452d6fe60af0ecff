// Shared device/host helpers for the ptychotomo HIP library (gfx950).
//
//  * status codes and a per-thread last-error string for the C ABI
//  * complex helpers on float2
//  * compile-time trig (twiddle constants) and an in-register FFT whose
//    length is a template parameter (detector frames: 8..64 points per lane)
//  * an LDS Stockham FFT with a run-time mixed-radix plan (2,3,4,5,8) for the
//    tomography lines (N = 3n/2 points)
//  * FP64 wavefront / workgroup reductions
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <type_traits>
#include <utility>

#include "../../include/ptychotomo_hip.h"

namespace pt {

// ---------------------------------------------------------------- errors
void set_error(const std::string& msg);

#define PT_HIP(call)                                                          \
  do {                                                                        \
    hipError_t e_ = (call);                                                   \
    if (e_ != hipSuccess) {                                                   \
      ::pt::set_error(std::string(#call) + ": " + hipGetErrorString(e_));     \
      return PT_ERR_HIP;                                                      \
    }                                                                         \
  } while (0)

#define PT_REQUIRE(cond, code, msg)                                           \
  do {                                                                        \
    if (!(cond)) {                                                            \
      ::pt::set_error(msg);                                                   \
      return code;                                                            \
    }                                                                         \
  } while (0)

#define PT_LAUNCH_CHECK()                                                     \
  do {                                                                        \
    hipError_t e_ = hipGetLastError();                                        \
    if (e_ != hipSuccess) {                                                   \
      ::pt::set_error(std::string("kernel launch: ") + hipGetErrorString(e_)); \
      return PT_ERR_HIP;                                                      \
    }                                                                         \
  } while (0)

// ---------------------------------------------------------------- complex
__host__ __device__ inline float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__host__ __device__ inline float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__host__ __device__ inline float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__host__ __device__ inline float2 cmulc(float2 a, float2 b) {  // a * conj(b)
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__host__ __device__ inline float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
__host__ __device__ inline float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
__host__ __device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__host__ __device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// complex value of the same type as C from two reals
__host__ __device__ inline float2 cmake(float2, float x, float y) { return make_float2(x, y); }
__host__ __device__ inline double2 cmake(double2, double x, double y) { return make_double2(x, y); }
// multiply by SIGN*i  (SIGN = -1: -i, SIGN = +1: +i)
template <int SIGN, typename C>
__host__ __device__ inline C mul_i(C a) {
  return SIGN < 0 ? cmake(a, a.y, -a.x) : cmake(a, -a.y, a.x);
}

// ---------------------------------------------------------------- compile-time helpers
template <int I>
using ic = std::integral_constant<int, I>;

template <int B, int E, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(ic<B>{});
    static_for<B + 1, E>(static_cast<F&&>(f));
  }
}

constexpr double kPi = 3.14159265358979323846;

// sin/cos of 2*pi*num/den evaluated exactly enough at compile time (Taylor
// series after octant reduction; |error| < 1e-16).
constexpr double ct_sin_small(double x) {
  double term = x, sum = x;
  for (int k = 1; k < 14; ++k) {
    term *= -x * x / ((2 * k) * (2 * k + 1));
    sum += term;
  }
  return sum;
}
constexpr double ct_cos_small(double x) {
  double term = 1.0, sum = 1.0;
  for (int k = 1; k < 14; ++k) {
    term *= -x * x / ((2 * k - 1) * (2 * k));
    sum += term;
  }
  return sum;
}
// cos/sin of 2*pi*m/L for integer m, L (m reduced mod L)
constexpr double ct_cos2pi(long m, long L) {
  long r = ((m % L) + L) % L;
  // reduce to first quadrant using symmetry on 8*r/L
  double x = 2.0 * kPi * (double)r / (double)L;
  if (x > kPi) x -= 2.0 * kPi;                 // (-pi, pi]
  double ax = x < 0 ? -x : x;                  // [0, pi]
  double c;
  if (ax <= kPi / 4) c = ct_cos_small(ax);
  else if (ax <= 3 * kPi / 4) c = ct_sin_small(kPi / 2 - ax);
  else c = -ct_cos_small(kPi - ax);
  return c;
}
constexpr double ct_sin2pi(long m, long L) {
  long r = ((m % L) + L) % L;
  double x = 2.0 * kPi * (double)r / (double)L;
  if (x > kPi) x -= 2.0 * kPi;
  double ax = x < 0 ? -x : x;
  double s;
  if (ax <= kPi / 4) s = ct_sin_small(ax);
  else if (ax <= 3 * kPi / 4) s = ct_cos_small(kPi / 2 - ax);
  else s = ct_sin_small(kPi - ax);
  return x < 0 ? -s : s;
}

// W_L^(SIGN*m) = exp(SIGN * 2 pi i m / L), rounded to float (re, im) and
// to double (re64, im64)
template <int L, int M, int SIGN>
struct Tw {
  static constexpr long mm = ((long)M % L + L) % L;
  static constexpr double re64 = ct_cos2pi(mm, L);
  static constexpr double im64 = SIGN * ct_sin2pi(mm, L);
  static constexpr float re = (float)re64;
  static constexpr float im = (float)im64;
  static constexpr bool one = (mm == 0);
  static constexpr bool minus_one = (2 * mm == L);
  static constexpr bool plus_i = (4 * mm == L && SIGN > 0) || (4 * mm == 3 * L && SIGN < 0);
  static constexpr bool minus_i = (4 * mm == L && SIGN < 0) || (4 * mm == 3 * L && SIGN > 0);
};

// a * W_L^(SIGN*M) for float2 (float constants) or double2 (double constants)
template <int L, int M, int SIGN, typename C>
__host__ __device__ __forceinline__ C twiddle_ct(C a) {
  using T = Tw<L, M, SIGN>;
  using R = decltype(a.x);
  constexpr R re = std::is_same<R, double>::value ? (R)T::re64 : (R)T::re;
  constexpr R im = std::is_same<R, double>::value ? (R)T::im64 : (R)T::im;
  if constexpr (T::one) return a;
  else if constexpr (T::minus_one) return cmake(a, -a.x, -a.y);
  else if constexpr (T::plus_i) return cmake(a, -a.y, a.x);
  else if constexpr (T::minus_i) return cmake(a, a.y, -a.x);
  else return cmake(a, a.x * re - a.y * im, a.x * im + a.y * re);
}

// ---------------------------------------------------------------- small DFTs (compile-time)
template <int SIGN, typename C>
__host__ __device__ __forceinline__ void dft2(C& a0, C& a1) {
  C t = a0;
  a0 = cadd(t, a1);
  a1 = csub(t, a1);
}

template <int SIGN, typename C>
__host__ __device__ __forceinline__ void dft4(C& a0, C& a1, C& a2, C& a3) {
  C t0 = cadd(a0, a2), t1 = csub(a0, a2);
  C t2 = cadd(a1, a3), t3 = mul_i<SIGN>(csub(a1, a3));
  a0 = cadd(t0, t2);
  a2 = csub(t0, t2);
  a1 = cadd(t1, t3);
  a3 = csub(t1, t3);
}

template <int SIGN, typename C>
__host__ __device__ __forceinline__ void dft8(C* a) {
  C e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6];
  C o0 = a[1], o1 = a[3], o2 = a[5], o3 = a[7];
  dft4<SIGN>(e0, e1, e2, e3);
  dft4<SIGN>(o0, o1, o2, o3);
  o1 = twiddle_ct<8, 1, SIGN>(o1);
  o2 = twiddle_ct<8, 2, SIGN>(o2);
  o3 = twiddle_ct<8, 3, SIGN>(o3);
  a[0] = cadd(e0, o0); a[4] = csub(e0, o0);
  a[1] = cadd(e1, o1); a[5] = csub(e1, o1);
  a[2] = cadd(e2, o2); a[6] = csub(e2, o2);
  a[3] = cadd(e3, o3); a[7] = csub(e3, o3);
}

template <int R, int SIGN, typename C>
__host__ __device__ __forceinline__ void dft_ct(C* a) {
  if constexpr (R == 2) dft2<SIGN>(a[0], a[1]);
  else if constexpr (R == 4) dft4<SIGN>(a[0], a[1], a[2], a[3]);
  else if constexpr (R == 8) dft8<SIGN>(a);
  else static_assert(R == 2, "radix");
}

// ---------------------------------------------------------------- in-register FFT
// Unnormalised DFT of L points held by one lane, natural order in and out:
//   X[k] = sum_j x[j] exp(SIGN * 2 pi i j k / L).
// Stockham passes with compile-time radices; all indices are constants so
// the data stay in VGPRs.
template <int L>
struct RegPlan {
  // first radix used at stage with Ns already done
  static constexpr int radix(int rem) { return rem == 16 ? 4 : (rem % 8 == 0 ? 8 : (rem % 4 == 0 ? 4 : 2)); }
};

template <int L, int Ns, int SIGN, typename C>
__host__ __device__ __forceinline__ void reg_fft_pass(C (&v)[L]) {
  if constexpr (Ns < L) {
    constexpr int R = RegPlan<L>::radix(L / Ns);
    C out[L];
    static_for<0, L / R>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      constexpr int k = j % Ns;
      C a[R];
      static_for<0, R>([&](auto icc) {
        constexpr int i = decltype(icc)::value;
        a[i] = twiddle_ct<Ns * R, i * k, SIGN>(v[j + i * (L / R)]);
      });
      dft_ct<R, SIGN>(a);
      constexpr int idxD = (j / Ns) * Ns * R + k;
      static_for<0, R>([&](auto icc) {
        constexpr int i = decltype(icc)::value;
        out[idxD + i * Ns] = a[i];
      });
    });
    static_for<0, L>([&](auto icc) { v[decltype(icc)::value] = out[decltype(icc)::value]; });
    reg_fft_pass<L, Ns * R, SIGN>(v);
  }
}

// C = float2 (FP32 arithmetic) or double2 (FP64 arithmetic, double twiddles)
template <int L, int SIGN, typename C>
__host__ __device__ __forceinline__ void reg_fft(C (&v)[L]) {
  if constexpr (L > 1) reg_fft_pass<L, 1, SIGN>(v);
}

// ---------------------------------------------------------------- LDS mixed-radix FFT
// Division by a run-time invariant d (Granlund & Montgomery, "Division by
// invariant integers using multiplication", 1994, round-up variant):
// x / d == (umulhi(x, m) + x) >> s for 0 <= x < 2^31, with
// s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1.
struct DivC {
  unsigned m, s;
};
inline DivC make_divc(unsigned d) {
  unsigned s = 0;
  while ((1u << s) < d) ++s;
  const unsigned long long m = ((1ull << 32) * ((1ull << s) - d)) / d + 1;
  return DivC{(unsigned)m, s};
}
__device__ __forceinline__ int fdiv(int x, DivC c) {
  return (int)((__umulhi((unsigned)x, c.m) + (unsigned)x) >> c.s);
}

// Run-time plan for one line length N = prod(radix[i]), with the division
// constants of each pass: by its butterfly count N / radix[i] and by its
// input stride Ns = radix[0] * ... * radix[i-1].  Twiddle table
// tw[m] = exp(-2 pi i m / N) (FP64-rounded) in global memory or staged in LDS.
struct LinePlan {
  int N;
  int npass;
  int radix[12];
  DivC dnb[12], dns[12];
};

template <int SIGN>
__device__ __forceinline__ void dft3(float2* a) {
  constexpr float s3 = 0.86602540378443864676f * (float)SIGN;
  const float2 t1 = cadd(a[1], a[2]);
  const float2 t2 = make_float2(a[0].x - 0.5f * t1.x, a[0].y - 0.5f * t1.y);
  const float2 d = csub(a[1], a[2]);
  const float2 t3 = make_float2(-s3 * d.y, s3 * d.x);  // SIGN*i*sqrt(3)/2*(a1-a2)
  a[0] = cadd(a[0], t1);
  a[1] = cadd(t2, t3);
  a[2] = csub(t2, t3);
}

template <int SIGN>
__device__ __forceinline__ void dft5(float2* a) {
  constexpr float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
  constexpr float s1 = 0.95105651629515357212f * (float)SIGN;
  constexpr float s2 = 0.58778525229247312917f * (float)SIGN;
  const float2 b1 = cadd(a[1], a[4]), b4 = csub(a[1], a[4]);
  const float2 b2 = cadd(a[2], a[3]), b3 = csub(a[2], a[3]);
  const float2 x0 = a[0];
  const float2 r1 = make_float2(x0.x + c1 * b1.x + c2 * b2.x, x0.y + c1 * b1.y + c2 * b2.y);
  const float2 r2 = make_float2(x0.x + c2 * b1.x + c1 * b2.x, x0.y + c2 * b1.y + c1 * b2.y);
  const float2 q1 = make_float2(-(s1 * b4.y + s2 * b3.y), s1 * b4.x + s2 * b3.x);
  const float2 q2 = make_float2(-(s2 * b4.y - s1 * b3.y), s2 * b4.x - s1 * b3.x);
  a[0] = make_float2(x0.x + b1.x + b2.x, x0.y + b1.y + b2.y);
  a[1] = cadd(r1, q1);
  a[4] = csub(r1, q1);
  a[2] = cadd(r2, q2);
  a[3] = csub(r2, q2);
}

template <int R, int SIGN>
__device__ __forceinline__ void dft_small(float2* a) {
  if constexpr (R == 3) dft3<SIGN>(a);
  else if constexpr (R == 5) dft5<SIGN>(a);
  else dft_ct<R, SIGN>(a);
}

// One out-of-place Stockham pass of radix R over `nlines` lines (src and
// dst at line * stride): each thread takes butterflies b = t, t + nthr, ...
// one at a time (R values live), so the pass needs no register budget and
// one barrier.  Twiddle W_{Ns R}^{i k} = tw[i k N/(Ns R)] (conjugated for
// SIGN=+1); tw[0] = 1 exactly, so the k = 0 products are exact.
template <int R, int SIGN>
__device__ __forceinline__ void pp_pass(const float2* __restrict__ src, float2* __restrict__ dst,
                                        int stride, int nlines, int N, int Ns, DivC dnb, DivC dns,
                                        const float2* __restrict__ tw, int t, int nthr) {
  const int nb = N / R;
  const int total = nb * nlines;
  const int step = nb / Ns;
  for (int b = t; b < total; b += nthr) {
    const int line = fdiv(b, dnb), j = b - line * nb;
    const int jq = fdiv(j, dns), k = j - jq * Ns;
    const float2* s = src + line * stride + j;
    float2 v[R];
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = s[i * nb];
#pragma unroll
    for (int i = 1; i < R; ++i) {
      float2 w = tw[i * k * step];
      if (SIGN > 0) w.y = -w.y;
      v[i] = cmul(v[i], w);
    }
    dft_small<R, SIGN>(v);
    float2* d = dst + line * stride + jq * Ns * R + k;
#pragma unroll
    for (int i = 0; i < R; ++i) d[i * Ns] = v[i];
  }
}

// FFT of `nlines` lines of length plan.N held in LDS at a + line*stride,
// ping-ponging with b (same shape), by `nthr` threads (index t) that all
// call it together; begins with the caller's barrier already passed and
// ends with one.  Returns the buffer that holds the result (a or b).
// sign -1 forward, +1 inverse (unnormalised).
template <int SIGN>
__device__ inline float2* lds_fft_pp(float2* a, float2* b, int stride, int nlines,
                                     const LinePlan& plan, const float2* __restrict__ tw, int t,
                                     int nthr) {
  int Ns = 1;
  for (int p = 0; p < plan.npass; ++p) {
    const DivC dnb = plan.dnb[p], dns = plan.dns[p];
    switch (plan.radix[p]) {
      case 2: pp_pass<2, SIGN>(a, b, stride, nlines, plan.N, Ns, dnb, dns, tw, t, nthr); break;
      case 3: pp_pass<3, SIGN>(a, b, stride, nlines, plan.N, Ns, dnb, dns, tw, t, nthr); break;
      case 4: pp_pass<4, SIGN>(a, b, stride, nlines, plan.N, Ns, dnb, dns, tw, t, nthr); break;
      case 5: pp_pass<5, SIGN>(a, b, stride, nlines, plan.N, Ns, dnb, dns, tw, t, nthr); break;
      default: pp_pass<8, SIGN>(a, b, stride, nlines, plan.N, Ns, dnb, dns, tw, t, nthr); break;
    }
    __syncthreads();
    Ns *= plan.radix[p];
    float2* c = a;
    a = b;
    b = c;
  }
  return a;
}

// ---------------------------------------------------------------- register line FFT
// Unnormalised DFT of R points in registers, R = 2^a (a <= 4) or 3 x 2^a (a <= 3):
// 2, 4, 8 (dft_ct), 16 (reg_fft), 3 (dft3), 6, 12, 24 as decimation in time R = 3 x B:
//   X[k1 + 3 k2] = sum_n2 W_B^(n2 k2) W_R^(n2 k1) sum_n1 x[B n1 + n2] W_3^(n1 k1).
template <int R, int SIGN>
__device__ __forceinline__ void dft_r(float2* a);

template <int B, int SIGN>
__device__ __forceinline__ void dft_3b(float2* a) {
  constexpr int R = 3 * B;
  float2 y[B][3];
  static_for<0, B>([&](auto n2c) {
    constexpr int n2 = decltype(n2c)::value;
    float2 s[3] = {a[n2], a[B + n2], a[2 * B + n2]};
    dft3<SIGN>(s);
    static_for<0, 3>([&](auto k1c) {
      constexpr int k1 = decltype(k1c)::value;
      y[n2][k1] = twiddle_ct<R, n2 * k1, SIGN>(s[k1]);
    });
  });
  static_for<0, 3>([&](auto k1c) {
    constexpr int k1 = decltype(k1c)::value;
    float2 s[B];
    static_for<0, B>([&](auto n2c) { s[decltype(n2c)::value] = y[decltype(n2c)::value][k1]; });
    dft_r<B, SIGN>(s);
    static_for<0, B>([&](auto k2c) {
      constexpr int k2 = decltype(k2c)::value;
      a[k1 + 3 * k2] = s[k2];
    });
  });
}

template <int R, int SIGN>
__device__ __forceinline__ void dft_r(float2* a) {
  if constexpr (R == 1) {
  } else if constexpr (R == 3) {
    dft3<SIGN>(a);
  } else if constexpr (R == 2 || R == 4 || R == 8) {
    dft_ct<R, SIGN>(a);
  } else if constexpr (R == 16) {
    float2 v[16];
    static_for<0, 16>([&](auto c) { v[decltype(c)::value] = a[decltype(c)::value]; });
    reg_fft<16, SIGN>(v);
    static_for<0, 16>([&](auto c) { a[decltype(c)::value] = v[decltype(c)::value]; });
  } else {
    static_assert(R == 6 || R == 12 || R == 24, "radix");
    dft_3b<R / 3, SIGN>(a);
  }
}

constexpr int ilog2_ct(int v) {
  int e = 0;
  while (v > 1) {
    v >>= 1;
    ++e;
  }
  return e;
}

// Points per lane of the register line FFT for lines of 3n/2 points and the
// workgroup size of its kernels; lines of n = 2^e points take 16 per lane.
constexpr int kLineP = 24;
constexpr int kLineThreads = 6144 / kLineP;

// Compile-time plan of an N-point line FFT held P points per lane by
// T = N / P lanes: lane t holds the points at positions t + T m, m < P, in
// registers.  Stockham passes of radices that divide P (24 = 3 x 2^3, or 16;
// each lane then does P / R whole butterflies per pass and reads its inputs
// from the positions it holds): the factors 3 one per pass from the first, a
// factors 2 per pass from the last, the rest of the 2s in the first pass; with
// P = 24: N = 384: 6, 8, 8; 768: 12, 8, 8; 192: 3, 8, 8; 96: 12, 8; with
// P = 16: N = 64: 4, 16; 128: 8, 16; 256: 16, 16; 512: 2, 16, 16.
template <int N, int P_ = kLineP>
struct LineReg {
  static constexpr int P = P_;
  static_assert(P == 24 || P == 16, "register line FFT: 24 or 16 points per lane");
  static_assert(N % P == 0 && N % 27 != 0, "register line FFT: N = P T with at most 3^2");
  static constexpr int T = N / P;
  static constexpr int amax = P == 16 ? 4 : 3;
  static constexpr int n3 = (N % 9 == 0) ? 2 : (N % 3 == 0) ? 1 : 0;
  static constexpr int m3 = n3 == 2 ? 9 : n3 == 1 ? 3 : 1;
  static constexpr int e = ilog2_ct(N / m3);
  static_assert((N / m3) == (1 << e), "register line FFT: N = 3^b 2^e");
  static constexpr int np = n3 > (e + amax - 1) / amax ? n3 : (e + amax - 1) / amax;
  static constexpr int radix(int p) {
    return (p < n3 ? 3 : 1) << (p == 0 ? e - amax * (np - 1) : amax);
  }
  static constexpr int ns(int p) {
    int s = 1;
    for (int q = 0; q < p; ++q) s *= radix(q);
    return s;
  }
};

// Pass p for lane t of one line (LDS row ln, N values; tw[m] = exp(-2 pi i
// m/N)).  Butterfly j = t + T b (b < P/R) takes the points j + (N/R) i =
// registers b + (P/R) i, applies W_{Ns R}^(i k), k = j mod Ns, and the
// radix-R DFT.  An inner pass stores its outputs at Stockham positions
// (j div Ns) Ns R + k + Ns i in ln; the last pass (Ns R = N) puts output i
// back at position j + (N/R) i, i.e. in place in the registers.
template <int N, int SIGN, int p, int P>
__device__ __forceinline__ void line_reg_pass(float2 (&v)[P], float2* __restrict__ ln,
                                              const float2* __restrict__ tw, int t) {
  using L = LineReg<N, P>;
  constexpr int R = L::radix(p), Ns = L::ns(p), B = L::P / R, T = L::T;
  static_for<0, B>([&](auto bc) {
    constexpr int b = decltype(bc)::value;
    const int j = t + T * b;
    const int k = Ns == 1 ? 0 : j % Ns;
    float2 a[R];
    static_for<0, R>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      a[i] = v[b + B * i];
      if constexpr (i > 0 && Ns > 1) {
        float2 w = tw[i * k * (N / (Ns * R))];
        if constexpr (SIGN > 0) w.y = -w.y;
        a[i] = cmul(a[i], w);
      }
    });
    dft_r<R, SIGN>(a);
    if constexpr (p == L::np - 1) {
      static_for<0, R>([&](auto ic) { v[b + B * decltype(ic)::value] = a[decltype(ic)::value]; });
    } else {
      const int base = (j / Ns) * Ns * R + k;
      static_for<0, R>([&](auto ic) { ln[base + Ns * decltype(ic)::value] = a[decltype(ic)::value]; });
    }
  });
}

// The whole line FFT, registers in and out (positions t + T m both ways).
// Every lane of the workgroup calls it together: the LDS exchanges between
// passes end with a barrier each, and the caller's LDS writes before the
// call (e.g. the twiddle table) must be behind a barrier already.
template <int N, int SIGN, int P>
__device__ __forceinline__ void line_reg_fft(float2 (&v)[P], float2* __restrict__ ln,
                                             const float2* __restrict__ tw, int t) {
  using L = LineReg<N, P>;
  static_for<0, L::np>([&](auto pc) {
    constexpr int p = decltype(pc)::value;
    line_reg_pass<N, SIGN, p, P>(v, ln, tw, t);
    if constexpr (p < L::np - 1) {
      __syncthreads();
      static_for<0, L::P>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        v[m] = ln[t + L::T * m];
      });
      __syncthreads();
    }
  });
}

// ---------------------------------------------------------------- reductions
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Sum of `NV` doubles over the workgroup; result valid in thread 0.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* smem /* >= NV*16 */) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
  __syncthreads();
  if (lane == 0)
    for (int i = 0; i < NV; ++i) smem[i * 16 + wid] = v[i];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 0; i < NV; ++i) {
      double s = 0;
      for (int w = 0; w < nw; ++w) s += smem[i * 16 + w];
      v[i] = s;
    }
  }
}

// host: factor N into the supported radices; returns false if impossible
bool make_line_plan(int N, LinePlan* p);

// Launch profiler: when enabled for a kernel tag, HIP events are recorded on
// the launch stream right before and after every launch of that kernel.
struct ProfScope {
  bool active;
  int slot;
  hipStream_t st;
  ProfScope(const char* tag, hipStream_t stream);
  ~ProfScope();
};

// Workgroups are dispatched round-robin over the 8 XCDs (linear id w runs on
// XCD w % 8), each with its own L2.  xcd_contig renumbers linear ids so that
// every XCD runs one contiguous range of logical ids (the first total % 8
// XCDs one id more than the rest), in dispatch order: work items that read
// overlapping regions share one L2.  A bijection on [0, total); results do
// not depend on it.
__device__ __forceinline__ int xcd_contig(int w, int total) {
  const int q = total >> 3, r = total & 7, x = w & 7;
  return x * q + min(x, r) + (w >> 3);
}

// ---------------------------------------------------------------- line search
// One sweep's decision of a segment (solver.py:171-177): f_j = f1[j] + f2[j] already
// weighted, candidates cand[j] (j = 0: gamma = 0).  Accepts the first candidate
// that is not a strict ascent or is <= 1e-12 (then 0): step = {gamma, 0}, state =
// {gamma, 1}; otherwise the next sweep (cand_next) continues from half the last
// candidate, or, with `last`, the search ends at 0.  FP64, no contraction: the
// host restatement of the rule gives the same bits.
template <class F>
__device__ inline void ls_decide(double* state, double* step, const double* cand,
                                 double* cand_next, int ngam, int ngam_next, int last, F f) {
#pragma clang fp contract(off)
  const double fz = f(0);
  for (int j = 1; j < ngam; ++j) {
    const double g = cand[j];
    if (fz - f(j) < 0.0 && g > 1e-12) continue;
    const double out = g <= 1e-12 ? 0.0 : g;
    step[0] = out;
    step[1] = 0.0;
    state[0] = out;
    state[1] = 1.0;
    return;
  }
  if (last) {
    step[0] = step[1] = 0.0;
    state[0] = 0.0;
    state[1] = 1.0;
    return;
  }
  const double cur = cand[ngam - 1] * 0.5;
  state[0] = cur;
  cand_next[0] = 0.0;
  for (int j = 1; j < ngam_next; ++j) cand_next[j] = cur * ldexp(1.0, -(j - 1));
}

// Sums over pixels of the rho term's change at ngam candidates per segment, left
// as partials [seg][block][8] in the stream's reduction scratch (pt_k_rho_minf
// without its second pass): *part, *nblk.
int rho_minf_partials(double** part, int* nblk, const void* h, const void* psi, const void* lamd,
                      const void* d, double rho, const double* rho_dev, const double* gammas,
                      int ngam, long len, int nseg, const double* skip, hipStream_t st);

}  // namespace pt
