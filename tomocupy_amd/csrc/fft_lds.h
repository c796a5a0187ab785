// LDS-resident Stockham autosort FFT for sizes N <= 16384 whose prime factors
// are at most kFftMaxPrime (per transform), executed cooperatively by a
// workgroup on 2^lgH interleaved transforms held in LDS.
//
// Pass with radix R and current sub-transform length Ns (1, R1, R1*R2, ...):
//   for j in [0, N/R):  k = j mod Ns
//     a_r = x[j + r N/R] * W^(r k N/(Ns R))         (r = 0..R-1)
//     b   = DFT_R(a)
//     y[(j/Ns) Ns R + k + q Ns] = b_q
// which leaves the output in natural order.  Every thread stages all of its
// butterflies in registers before the barrier, so one LDS buffer suffices.
// Twiddles come from a per-size table W_N^k = exp(-2 pi i k/N) computed on the
// host in FP64; the inverse transform uses their conjugates.  Unnormalised in
// both directions.
//
// Two forms: sizes 2^k 3^a 5^b of with_static_size() have everything constant
// at compile time (lds_fft_c); any other size runs passes of radix 2..18, 20
// and larger primes chosen at plan time (lds_fft).
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"

namespace tomo {

constexpr int kFftMaxRadices = 16;
constexpr int kFftEPT = 16;  // complex elements staged per thread per pass (compiled sizes)
constexpr int kFftMaxPrime = 127;  // largest prime factor of a transform length
constexpr int kFftRegPrime = 17;   // larger primes run wave-uniform (rt_pass_prime)
constexpr int kFftRtVals = 20;     // values a thread holds in a run-time pass of small radix

// A run-time plan: the passes in order and the tables they read.
struct FftDesc {
  int N;
  int nr;
  int r[kFftMaxRadices];
  const float2 *tw;    // device, N entries
  const void *pm[3];  // cosine/sine matrices of the primes above kFftRegPrime, in pass order
                      // (float pairs; FftPlan::init by_rule: columns of double)
};

// The radix sequence of the compiled sizes; for every size the sequence by
// which widths are accepted (fft_threads).
struct FftRule {
  int N;
  int nr;
  int r[kFftMaxRadices];
};

// Host-side plan: radix sequence + device tables.
struct FftPlan {
  FftDesc d{};
  FftRule rule{};
  DevBuf tw, pm;
  // N <= 16384, prime factors <= kFftMaxPrime; by_rule: d has the rule's radices
  int init(int N, bool by_rule = false);
  // the rule's radix sequence alone (no device memory, no HIP call)
  static int radices(int N, FftRule &r);
  void release() {
    tw.release();
    pm.release();
  }
};

// The cheapest passes of a run-time plan for 2^lgH interleaved transforms of
// length N (no HIP call, the tables stay); their cost, without the prime passes,
// or d.nr = 0 where there are none.
double fft_rt_radices(int N, FftDesc &d, int lgH = 0);

template <int DIR>
__device__ __forceinline__ float2 mul_i(float2 a) {
  // multiply by (-i) for the forward transform, (+i) for the inverse
  return DIR < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

template <int R, int DIR>
__device__ __forceinline__ void butterfly(float2 *a) {
  if constexpr (R == 2) {
    float2 t = a[0];
    a[0] = cadd(t, a[1]);
    a[1] = csub(t, a[1]);
  } else if constexpr (R == 3) {
    const float s3 = 0.86602540378443864676f;  // sqrt(3)/2
    float2 t1 = cadd(a[1], a[2]);
    float2 t2 = csub(a[1], a[2]);
    float2 m = make_float2(a[0].x - 0.5f * t1.x, a[0].y - 0.5f * t1.y);
    float2 r = cscale(mul_i<DIR>(t2), s3);
    a[0] = cadd(a[0], t1);
    a[1] = cadd(m, r);
    a[2] = csub(m, r);
  } else if constexpr (R == 5) {
    // y_k = sum_j a_j W^(jk), W = exp(-+2 pi i/5): pairs a_j +- a_(5-j) with
    // c_m = cos(2 pi m/5), s_m = sin(2 pi m/5)
    const float c1 = 0.30901699437494745f, c2 = -0.80901699437494734f;
    const float s1 = 0.95105651629515353f, s2 = 0.58778525229247320f;
    const float2 t1 = cadd(a[1], a[4]), t2 = cadd(a[2], a[3]);
    const float2 t3 = csub(a[1], a[4]), t4 = csub(a[2], a[3]);
    const float2 b1 = make_float2(a[0].x + c1 * t1.x + c2 * t2.x, a[0].y + c1 * t1.y + c2 * t2.y);
    const float2 b2 = make_float2(a[0].x + c2 * t1.x + c1 * t2.x, a[0].y + c2 * t1.y + c1 * t2.y);
    const float2 d1 = mul_i<DIR>(make_float2(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y));
    const float2 d2 = mul_i<DIR>(make_float2(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y));
    a[0] = cadd(a[0], cadd(t1, t2));
    a[1] = cadd(b1, d1);
    a[4] = csub(b1, d1);
    a[2] = cadd(b2, d2);
    a[3] = csub(b2, d2);
  } else if constexpr (R == 7) {
    // pairs a_j +- a_(7-j), j = 1..3; y_m = a0 + sum_j cos(2 pi jm/7) t_j
    // -+ i sum_j sin(2 pi jm/7) u_j, y_(7-m) its conjugate combination
    const float C[4] = {1.f, 0.62348980185873353f, -0.22252093395631440f,
                        -0.90096886790241913f};
    const float S[4] = {0.f, 0.78183148246802981f, 0.97492791218182361f,
                        0.43388373911755812f};
    float2 t[4], u[4];
#pragma unroll
    for (int j = 1; j <= 3; ++j) {
      t[j] = cadd(a[j], a[7 - j]);
      u[j] = csub(a[j], a[7 - j]);
    }
    float2 y[7];
    y[0] = cadd(a[0], cadd(t[1], cadd(t[2], t[3])));
#pragma unroll
    for (int m = 1; m <= 3; ++m) {
      float2 b = a[0], d = make_float2(0.f, 0.f);
#pragma unroll
      for (int j = 1; j <= 3; ++j) {
        const int q = (j * m) % 7;  // cos(2 pi q/7) = C[min(q, 7-q)], sin = +-S[min(q, 7-q)]
        const float c = C[q <= 3 ? q : 7 - q];
        const float sg = q <= 3 ? S[q] : -S[7 - q];
        b = make_float2(b.x + c * t[j].x, b.y + c * t[j].y);
        d = make_float2(d.x + sg * u[j].x, d.y + sg * u[j].y);
      }
      const float2 di = mul_i<DIR>(d);
      y[m] = cadd(b, di);
      y[7 - m] = csub(b, di);
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) a[k] = y[k];
  } else if constexpr (R == 4) {
    float2 t0 = cadd(a[0], a[2]);
    float2 t1 = csub(a[0], a[2]);
    float2 t2 = cadd(a[1], a[3]);
    float2 t3 = mul_i<DIR>(csub(a[1], a[3]));
    a[0] = cadd(t0, t2);
    a[2] = csub(t0, t2);
    a[1] = cadd(t1, t3);
    a[3] = csub(t1, t3);
  } else if constexpr (R == 8) {
    float2 e[4] = {a[0], a[2], a[4], a[6]};
    float2 o[4] = {a[1], a[3], a[5], a[7]};
    butterfly<4, DIR>(e);
    butterfly<4, DIR>(o);
    const float h = 0.70710678118654752440f;
    // w8^q for q = 1,2,3 with w8 = exp(DIR * i pi/4)
    float2 o1 = make_float2(h * (o[1].x - DIR * o[1].y), h * (o[1].y + DIR * o[1].x));
    float2 o2 = mul_i<DIR>(o[2]);
    float2 o3 = make_float2(h * (-o[3].x - DIR * o[3].y), h * (-o[3].y + DIR * o[3].x));
    a[0] = cadd(e[0], o[0]);
    a[4] = csub(e[0], o[0]);
    a[1] = cadd(e[1], o1);
    a[5] = csub(e[1], o1);
    a[2] = cadd(e[2], o2);
    a[6] = csub(e[2], o2);
    a[3] = cadd(e[3], o3);
    a[7] = csub(e[3], o3);
  } else if constexpr (R == 16) {
    // 16 = 4 x 4 in place: radix-4 over r2 for each r1 (results q2 back in
    // slots r1 + 4 q2), internal twiddles w16^(r1 q2), radix-4 over r1 for each
    // q2 (results q1 in slots 4 q2 + q1).  Output q = q2 + 4 q1 therefore sits
    // in slot out_slot<16>(q) = 4 (q & 3) + (q >> 2).
#pragma unroll
    for (int r1 = 0; r1 < 4; ++r1) {
      float2 t[4] = {a[r1], a[r1 + 4], a[r1 + 8], a[r1 + 12]};
      butterfly<4, DIR>(t);
      a[r1] = t[0];
      a[r1 + 4] = t[1];
      a[r1 + 8] = t[2];
      a[r1 + 12] = t[3];
    }
    // w16^m = exp(DIR * 2 pi i m / 16), m = r1*q2 in {1,2,3,4,6,9}
    const float c1 = 0.92387953251128675613f, s1 = 0.38268343236508977173f;
    const float h = 0.70710678118654752440f;
    const float2 w1 = make_float2(c1, DIR * s1), w2 = make_float2(h, DIR * h);
    const float2 w3 = make_float2(s1, DIR * c1);
    const float2 w6 = make_float2(-h, DIR * h), w9 = make_float2(-c1, -DIR * s1);
    a[1 + 4 * 1] = cmul(a[1 + 4 * 1], w1);
    a[1 + 4 * 2] = cmul(a[1 + 4 * 2], w2);
    a[1 + 4 * 3] = cmul(a[1 + 4 * 3], w3);
    a[2 + 4 * 1] = cmul(a[2 + 4 * 1], w2);
    a[2 + 4 * 2] = mul_i<DIR>(a[2 + 4 * 2]);  // w16^4 = exp(DIR i pi/2) = DIR * i
    a[2 + 4 * 3] = cmul(a[2 + 4 * 3], w6);
    a[3 + 4 * 1] = cmul(a[3 + 4 * 1], w3);
    a[3 + 4 * 2] = cmul(a[3 + 4 * 2], w6);
    a[3 + 4 * 3] = cmul(a[3 + 4 * 3], w9);
#pragma unroll
    for (int q2 = 0; q2 < 4; ++q2) butterfly<4, DIR>(a + 4 * q2);
  }
}

// Register slot holding output q of butterfly<R>: the identity except for the
// in-place radix-16 butterfly.
template <int R>
__device__ __forceinline__ constexpr int out_slot(int q) {
  return R == 16 ? 4 * (q & 3) + (q >> 2) : q;
}

// LDS index of element i of a transform: one pad slot per 16 elements, which
// breaks the power-of-two strides of the early Stockham passes across banks.
__device__ __forceinline__ int lds_pad(int i) { return i + (i >> 4); }
// LDS elements needed for a padded transform of length N.
__host__ __device__ inline int lds_padded_len(int N) { return N + (N >> 4); }

// LDS index of element i of a transform: compiled size (NS > 0) or run-time
// size (NS = 0).
template <int NS>
__device__ __forceinline__ int lidx(int i) {
  return NS > 0 ? lds_pad(i) : i;
}

// a[r] *= w^r for r = 1..R-1 with w = W_N^base (conjugated for the inverse).
// Powers of two of w come from the FP64-built table; the others are products
// of at most three of them (relative error a few float32 ulps).
template <int R, int DIR>
__device__ __forceinline__ void twiddle(float2 *a, const float2 *__restrict__ tw, unsigned base) {
  auto ld = [&](unsigned m) {
    float2 w = tw[base * m];
    if (DIR > 0) w.y = -w.y;
    return w;
  };
  if constexpr (R == 2) {
    a[1] = cmul(a[1], ld(1));
  } else if constexpr (R == 3) {
    a[1] = cmul(a[1], ld(1));
    a[2] = cmul(a[2], ld(2));
  } else if constexpr (R == 5) {
    const float2 w1 = ld(1), w2 = ld(2), w4 = ld(4);
    a[1] = cmul(a[1], w1);
    a[2] = cmul(a[2], w2);
    a[3] = cmul(a[3], cmul(w2, w1));
    a[4] = cmul(a[4], w4);
  } else if constexpr (R == 4) {
    const float2 w1 = ld(1), w2 = ld(2);
    a[1] = cmul(a[1], w1);
    a[2] = cmul(a[2], w2);
    a[3] = cmul(a[3], cmul(w2, w1));
  } else {
    float2 w[R];
    w[1] = ld(1);
    w[2] = ld(2);
    w[4] = ld(4);
    w[3] = cmul(w[2], w[1]);
    w[5] = cmul(w[4], w[1]);
    w[6] = cmul(w[4], w[2]);
    w[7] = cmul(w[4], w[3]);
    if constexpr (R == 16) {
      w[8] = ld(8);
#pragma unroll
      for (int r = 9; r < 16; ++r) w[r] = cmul(w[8], w[r - 8]);
    }
#pragma unroll
    for (int r = 1; r < R; ++r) a[r] = cmul(a[r], w[r]);
  }
}

// ---- transforms of a run-time size -------------------------------------------
// What bounds them: vector instructions, so the passes are few (radices up to
// 20: three for the 2n of a detector) and their index arithmetic small: one
// index split per butterfly, inputs at a uniform stride, no bank padding (an
// odd radix goes first where there is one; its writes, R apart, then fall on
// different banks).  Each pass sits behind a call, so a kernel's register
// demand is its largest pass's; pointers carry their address space (a generic
// one would turn every table read into a FLAT access).  The call's convention
// spends 87 registers on the 64 a pass needs (5 waves per SIMD); inlined, the
// switch spilled.  n = 2448 (2n = 17 18 16), 8 slices x 1500 angles, us, row
// pass / column pass / filter and spectrum: 378 / 528 / 283, against 1211 /
// 1123 / 1065 with radices 16, 2, 3, 3, 17 and per-element index arithmetic (of the
// filter's 1065, 349 were left by the plans, the rest went with its transforms of
// 2n points).

typedef float f2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f2v *LdsPtr;
typedef const __attribute__((address_space(1))) f2v *TabPtr;
typedef const __attribute__((address_space(4))) float *ScalarPtr;
typedef const __attribute__((address_space(4))) double *ScalarPtr64;

__device__ __forceinline__ float2 ldf2(LdsPtr p) {
  const f2v v = *p;
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ float2 ldf2(TabPtr p) {
  const f2v v = *p;
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ void stf2(LdsPtr p, float2 v) { *p = f2v{v.x, v.y}; }

// cos and sin(2 pi m / R) at compile time (Taylor series on [-pi, pi]).
constexpr double cx_angle(int m, int R) {
  const int q = ((m % R) + R) % R;
  return 2.0 * 3.14159265358979323846 * (2 * q > R ? q - R : q) / R;
}
constexpr double cx_cos(int m, int R) {
  const double x = cx_angle(m, R);
  double t = 1.0, s = 1.0;
  for (int i = 2; i < 40; i += 2) {
    t *= -x * x / ((i - 1) * i);
    s += t;
  }
  return s;
}
constexpr double cx_sin(int m, int R) {
  const double x = cx_angle(m, R);
  double t = x, s = x;
  for (int i = 3; i < 40; i += 2) {
    t *= -x * x / ((i - 1) * i);
    s += t;
  }
  return s;
}
template <int M, int R>
struct Root {
  static constexpr float c = (float)cx_cos(M, R), s = (float)cx_sin(M, R);
};

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f) {
  (f(std::integral_constant<int, I>()), ...);
}
// f(integral_constant<int, i>) for i = 0..N-1
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(std::make_integer_sequence<int, N>(), f);
}

// v * exp(DIR 2 pi i M / R)
template <int M, int R, int DIR>
__device__ __forceinline__ float2 rotate(float2 v) {
  constexpr int m = M % R;
  if constexpr (m == 0)
    return v;
  else if constexpr (2 * m == R)
    return make_float2(-v.x, -v.y);
  else if constexpr (4 * m == R)
    return mul_i<DIR>(v);
  else if constexpr (4 * m == 3 * R)
    return mul_i<-DIR>(v);
  else
    return cmul(v, make_float2(Root<m, R>::c, DIR * Root<m, R>::s));
}

// First factor of the split R = A * B of a composite radix.
constexpr int dft_split(int R) {
  return R == 12 || R == 32 ? 4 : R == 20 ? 5 : R == 15 || R == 9 ? 3 : R == 18 ? 9 : 2;
}

// a <- DFT_R(a) in natural order, in registers, every constant a literal.
template <int R, int DIR>
__device__ __forceinline__ void dft(float2 *a) {
  if constexpr (R <= 5 || R == 7 || R == 8) {
    butterfly<R, DIR>(a);
  } else if constexpr (R == 16) {
    butterfly<16, DIR>(a);
    float2 t[16];
    static_for<16>([&](auto q) { t[q] = a[4 * (q & 3) + (q >> 2)]; });
    static_for<16>([&](auto q) { a[q] = t[q]; });
  } else if constexpr (R == 11 || R == 13 || R == 17) {
    // cosine and sine pairs a_j +- a_(R-j)
    constexpr int h = (R - 1) / 2;
    float2 P[h + 1], M[h + 1];
    const float2 a0 = a[0];
    static_for<h>([&](auto i) {
      constexpr int j = i + 1;
      P[j] = cadd(a[j], a[R - j]);
      M[j] = csub(a[j], a[R - j]);
      a[0] = cadd(a[0], P[j]);
    });
    // (all real-coefficient sums, then all imaginary ones: P is dead before the
    // second half, which keeps the registers of radix 17 at 80)
    float2 re[h];
    static_for<h>([&](auto i) {
      constexpr int q = i + 1;
      re[i] = a0;
      static_for<h>([&](auto l) {
        constexpr int j = l + 1, m = (j * q) % R;
        re[i].x = fmaf(Root<m, R>::c, P[j].x, re[i].x);
        re[i].y = fmaf(Root<m, R>::c, P[j].y, re[i].y);
      });
    });
    static_for<h>([&](auto i) {
      constexpr int q = i + 1;
      float2 im = make_float2(0.f, 0.f);
      static_for<h>([&](auto l) {
        constexpr int j = l + 1, m = (j * q) % R;
        im.x = fmaf(Root<m, R>::s, M[j].x, im.x);
        im.y = fmaf(Root<m, R>::s, M[j].y, im.y);
      });
      const float2 mi = mul_i<DIR>(im);
      a[q] = cadd(re[i], mi);
      a[R - q] = csub(re[i], mi);
    });
  } else {
    // n = B i1 + i2, k = k1 + A k2:
    //   X[k] = sum_i2 W_B^(i2 k2) W_R^(i2 k1) sum_i1 W_A^(i1 k1) a[n]
    constexpr int A = dft_split(R), B = R / A;
    float2 c[R];
    static_for<B>([&](auto i2) {
      float2 t[A];
      static_for<A>([&](auto i1) { t[i1] = a[B * i1 + i2]; });
      dft<A, DIR>(t);
      static_for<A>([&](auto k1) {
        c[k1 * B + i2] = rotate<decltype(i2)::value * decltype(k1)::value, R, DIR>(t[k1]);
      });
    });
    static_for<A>([&](auto k1) {
      float2 t[B];
      static_for<B>([&](auto i2) { t[i2] = c[k1 * B + i2]; });
      dft<B, DIR>(t);
      static_for<B>([&](auto k2) { a[k1 + A * k2] = t[k2]; });
    });
  }
}

// a[r] *= w^r, w = W_N^base (conjugated for the inverse): w, w^2 and every
// fourth power from the table, the others products of two or three of them,
// four at a time (few registers).
template <int R, int DIR>
__device__ __forceinline__ void rt_twiddle(float2 *a, TabPtr tw, unsigned base) {
  auto ld = [&](unsigned r) {
    float2 w = ldf2(tw + base * r);
    if (DIR > 0) w.y = -w.y;
    return w;
  };
  float2 w[4];
  w[1] = ld(1);
  if constexpr (R > 2) w[2] = ld(2);
  if constexpr (R > 3) w[3] = cmul(w[2], w[1]);
  static_for<(R + 3) / 4>([&](auto blk) {
    constexpr int r0 = 4 * blk;
    float2 wb = make_float2(1.f, 0.f);
    if constexpr (r0 > 0) {
      wb = ld(r0);
      a[r0] = cmul(a[r0], wb);
    }
    static_for<3>([&](auto i) {
      constexpr int c = i + 1;
      if constexpr (r0 + c < R) a[r0 + c] = cmul(a[r0 + c], r0 > 0 ? cmul(wb, w[c]) : w[c]);
    });
  });
}

// Butterflies of radix R a thread takes in a pass (ten of radix 2 would cost a
// wave per SIMD: 98 registers).
constexpr int rt_maxb(int R) { return R == 2 ? 8 : R <= kFftRtVals / 2 ? kFftRtVals / R : 1; }

// One pass of radix R over 2^lgH interleaved transforms of length N (element
// i of transform t at buf[(i << lgH) + t]); ends with a barrier.  PAD (lgH = 0):
// 1 a first pass of radix 2, 4, 8 or 16 that writes element i at lds_pad(i), 2
// the pass after it.
template <int R, int DIR, int PAD = 0>
__device__ __noinline__ void rt_pass(LdsPtr buf, int N_, int Ns_, TabPtr tw, int lgH_, int tid,
                                     int nt_) {
  constexpr int MAXB = rt_maxb(R);
  const int N = __builtin_amdgcn_readfirstlane(N_), Ns = __builtin_amdgcn_readfirstlane(Ns_);
  const int lgH = __builtin_amdgcn_readfirstlane(lgH_), nt = __builtin_amdgcn_readfirstlane(nt_);
  const int S = (N / R) << lgH;  // butterflies; distance between a butterfly's inputs
  const int twstep = N / R / Ns;
  const float invNs = 1.0f / (float)Ns;
  float2 v[MAXB][R];
  int o[MAXB];
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < S) {
      LdsPtr p = buf + g;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = ldf2(PAD == 2 ? buf + lds_pad(g + r * S) : p + r * S);
      const int j = g >> lgH;
      // j / Ns and j mod Ns: float quotient, corrected
      int jq = (int)((float)j * invNs), k = j - jq * Ns;
      if (k < 0) jq -= 1, k += Ns;
      if (k >= Ns) jq += 1, k -= Ns;
      o[q] = ((jq * Ns * R + k) << lgH) + (g - (j << lgH));
      if constexpr (PAD == 1) o[q] = lds_pad(g * R);
      if (Ns > 1) rt_twiddle<R, DIR>(v[q], tw, (unsigned)(k * twstep));
      dft<R, DIR>(v[q]);
    }
  }
  __syncthreads();
  const int W = Ns << lgH;
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    if (tid + q * nt < S) {
      LdsPtr p = buf + o[q];
#pragma unroll
      for (int r = 0; r < R; ++r) stf2(p + r * W, v[q][r]);
    }
  }
  __syncthreads();
}

// Columns of a prime's cosine/sine matrix: whole groups of 8, 12 or 16 pairs.
constexpr int rt_prime_cols(int p) { return ((p - 1) / 2 + 47) / 48 * 48; }

// Waves a pass of a prime p above kFftRegPrime needs with G output pairs per
// wave, and the G it runs with.
constexpr int rt_prime_waves(int nb, int p, int G) {
  return ((nb + 63) / 64) * (((p - 1) / 2 + G - 1) / G);
}
constexpr int rt_prime_pairs(int nb, int p) {
  return rt_prime_waves(nb, p, 8) <= 16 ? 8 : rt_prime_waves(nb, p, 12) <= 16 ? 12 : 16;
}

// Pass of a prime radix p > kFftRegPrime.  With P_j = a_j + a_(p-j) and
// M_j = a_j - a_(p-j) (formed in place first, twiddles included),
//   b_q, b_(p-q) = a_0 + sum_j cos(2 pi j q/p) P_j -/+ i sum_j sin(2 pi j q/p) M_j.
// A wave takes 64 butterflies (one per lane) and G of the (p-1)/2 output
// pairs, so the cosines and sines are the same for the whole wave: scalar
// loads from the (p-1)/2 x hp matrix `pm` of (cos, sin), and an output pair
// costs four multiply-adds per j instead of eight with two table reads.
template <int G, int DIR>
__device__ __noinline__ void rt_pass_prime(LdsPtr buf, int N_, int Ns_, int p_, TabPtr tw,
                                           const float *pm_, int lgH_, int tid, int nt_) {
  const int N = __builtin_amdgcn_readfirstlane(N_), Ns = __builtin_amdgcn_readfirstlane(Ns_);
  const int p = __builtin_amdgcn_readfirstlane(p_), nt = __builtin_amdgcn_readfirstlane(nt_);
  const int lgH = __builtin_amdgcn_readfirstlane(lgH_);
  const uintptr_t pa = (uintptr_t)pm_;
  const unsigned plo = __builtin_amdgcn_readfirstlane((unsigned)pa);
  const unsigned phi = __builtin_amdgcn_readfirstlane((unsigned)(pa >> 32));
  const ScalarPtr pm = (ScalarPtr)(((uintptr_t)phi << 32) | plo);
  const int h = (p - 1) / 2, hp = rt_prime_cols(p);
  const int nb = (N / p) << lgH, twstep = N / p / Ns;
  for (int e = tid; e < nb * h; e += nt) {
    const int jj = e / nb, g = e - jj * nb;
    const LdsPtr x = buf + g + (jj + 1) * nb, y = buf + g + (p - 1 - jj) * nb;
    float2 u = ldf2(x), v = ldf2(y);
    if (Ns > 1) {
      const int kt = ((g >> lgH) % Ns) * twstep;
      float2 wu = ldf2(tw + kt * (jj + 1)), wv = ldf2(tw + kt * (p - 1 - jj));
      if (DIR > 0) wu.y = -wu.y, wv.y = -wv.y;
      u = cmul(u, wu);
      v = cmul(v, wv);
    }
    stf2(x, cadd(u, v));
    stf2(y, csub(u, v));
  }
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nblk = (nb + 63) / 64, grp = w / nblk;
  const int g = (w - grp * nblk) * 64 + lane;
  const bool live = grp * G < h && g < nb;
  float2 A[G], B[G], a0 = make_float2(0.f, 0.f), y0 = a0;
#pragma unroll
  for (int u = 0; u < G; ++u) A[u] = B[u] = make_float2(0.f, 0.f);
  if (live) {
    a0 = y0 = ldf2(buf + g);
#pragma unroll 1
    for (int j = 0; j < h; ++j) {
      const float2 P = ldf2(buf + g + (j + 1) * nb), M = ldf2(buf + g + (p - 1 - j) * nb);
      const ScalarPtr m = pm + 2 * (j * hp + grp * G);
      y0 = cadd(y0, P);
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const float c = m[2 * u], s = m[2 * u + 1];
        A[u].x = fmaf(c, P.x, A[u].x);
        A[u].y = fmaf(c, P.y, A[u].y);
        B[u].x = fmaf(s, M.x, B[u].x);
        B[u].y = fmaf(s, M.y, B[u].y);
      }
    }
  }
  __syncthreads();
  if (live) {
    const int j = g >> lgH, jq = j / Ns, k = j - jq * Ns;
    LdsPtr o = buf + (((jq * Ns * p + k) << lgH) + (g - (j << lgH)));
    const int W = Ns << lgH;
    if (grp == 0) stf2(o, y0);
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int q = grp * G + u + 1;
      if (q > h) break;
      const float2 re = cadd(a0, A[u]), mi = mul_i<DIR>(B[u]);
      stf2(o + q * W, cadd(re, mi));
      stf2(o + (p - q) * W, csub(re, mi));
    }
  }
  __syncthreads();
}

// The same in 64 bits between the LDS reads and writes, for one transform: P_j and
// M_j are rounded once, the sums too, and the cosines and sines are doubles (`pm`:
// row j has hp cosines, then hp sines).  Roundings of each step, and of the (p-1)/2
// constants, whose error all terms share, show where the result is what is left of
// much larger inputs, the high frequencies of a smooth row: noisy sinogram rows of
// ellipses, ramp, ne = 2840 (71), 2.7e-6 with floats, 2.4e-6 as one sum with the
// length's table, 2.15e-6 now.  What bounds it is the multiply-adds, at the rate of
// float ones; the cosine sums are finished before the sine sums begin (a third fewer
// registers).  8 x 720 rows of ne = 2840: 175 us with floats, 998 as one sum, 212 now.
template <int G, int DIR>
__device__ __noinline__ void rt_pass_prime64(LdsPtr buf, int N_, int Ns_, int p_, TabPtr tw,
                                             const double *pm_, int tid, int nt_) {
  const int N = __builtin_amdgcn_readfirstlane(N_), Ns = __builtin_amdgcn_readfirstlane(Ns_);
  const int p = __builtin_amdgcn_readfirstlane(p_), nt = __builtin_amdgcn_readfirstlane(nt_);
  const uintptr_t pa = (uintptr_t)pm_;
  const unsigned plo = __builtin_amdgcn_readfirstlane((unsigned)pa);
  const unsigned phi = __builtin_amdgcn_readfirstlane((unsigned)(pa >> 32));
  const ScalarPtr64 pm = (ScalarPtr64)(((uintptr_t)phi << 32) | plo);
  const int h = (p - 1) / 2, hp = rt_prime_cols(p);
  const int nb = N / p, twstep = nb / Ns;
  for (int e = tid; e < nb * h; e += nt) {
    const int jj = e / nb, g = e - jj * nb, kt = g % Ns * twstep;
    const LdsPtr x = buf + g + (jj + 1) * nb, y = buf + g + (p - 1 - jj) * nb;
    const float2 u = ldf2(x), v = ldf2(y);
    float2 wu = ldf2(tw + kt * (jj + 1)), wv = ldf2(tw + kt * (p - 1 - jj));
    if (DIR > 0) wu.y = -wu.y, wv.y = -wv.y;
    const double ux = (double)u.x * wu.x - (double)u.y * wu.y;
    const double uy = (double)u.x * wu.y + (double)u.y * wu.x;
    const double vx = (double)v.x * wv.x - (double)v.y * wv.y;
    const double vy = (double)v.x * wv.y + (double)v.y * wv.x;
    stf2(x, make_float2((float)(ux + vx), (float)(uy + vy)));
    stf2(y, make_float2((float)(ux - vx), (float)(uy - vy)));
  }
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nblk = (nb + 63) / 64, grp = w / nblk;
  const int g = (w - grp * nblk) * 64 + lane;
  const bool live = grp * G < h && g < nb;
  float2 re[G], y0;
  double Sx[G], Sy[G];
  if (live) {
    const float2 a0 = ldf2(buf + g);
    double y0x = a0.x, y0y = a0.y;
#pragma unroll
    for (int u = 0; u < G; ++u) Sx[u] = a0.x, Sy[u] = a0.y;
#pragma unroll 1
    for (int j = 0; j < h; ++j) {
      const float2 P = ldf2(buf + g + (j + 1) * nb);
      const double px = P.x, py = P.y;
      const ScalarPtr64 m = pm + 2 * j * hp + grp * G;
      y0x += px;
      y0y += py;
#pragma unroll
      for (int u = 0; u < G; ++u) {
        Sx[u] = fma(m[u], px, Sx[u]);
        Sy[u] = fma(m[u], py, Sy[u]);
      }
    }
    y0 = make_float2((float)y0x, (float)y0y);
#pragma unroll
    for (int u = 0; u < G; ++u) {
      re[u] = make_float2((float)Sx[u], (float)Sy[u]);
      Sx[u] = Sy[u] = 0.0;
    }
#pragma unroll 1
    for (int j = 0; j < h; ++j) {
      const float2 M = ldf2(buf + g + (p - 1 - j) * nb);
      const double mx = M.x, my = M.y;
      const ScalarPtr64 m = pm + (2 * j + 1) * hp + grp * G;
#pragma unroll
      for (int u = 0; u < G; ++u) {
        Sx[u] = fma(m[u], mx, Sx[u]);
        Sy[u] = fma(m[u], my, Sy[u]);
      }
    }
  }
  __syncthreads();
  if (live) {
    const int jq = g / Ns, k = g - jq * Ns;
    LdsPtr o = buf + jq * Ns * p + k;
    if (grp == 0) stf2(o, y0);
#pragma unroll
    for (int u = 0; u < G; ++u) {
      const int q = grp * G + u + 1;
      if (q > h) break;
      const float2 mi = mul_i<DIR>(make_float2((float)Sx[u], (float)Sy[u]));
      stf2(o + q * Ns, cadd(re[u], mi));
      stf2(o + (p - q) * Ns, csub(re[u], mi));
    }
  }
  __syncthreads();
}

// The prime passes with the output pairs a wave takes.
template <int DIR, bool WIDE>
__device__ __forceinline__ void rt_prime(LdsPtr buf, int N, int Ns, int R, TabPtr tw,
                                         const void *pm, int lgH, int tid, int nt) {
  const int G = rt_prime_pairs((N / R) << lgH, R);
  if (WIDE && G == 16)
    rt_pass_prime<16, DIR>(buf, N, Ns, R, tw, (const float *)pm, lgH, tid, nt);
  else if (G == 12)
    rt_pass_prime<12, DIR>(buf, N, Ns, R, tw, (const float *)pm, lgH, tid, nt);
  else
    rt_pass_prime<8, DIR>(buf, N, Ns, R, tw, (const float *)pm, lgH, tid, nt);
}

template <int DIR, bool WIDE>
__device__ __forceinline__ void rt_prime64(LdsPtr buf, int N, int Ns, int R, TabPtr tw,
                                           const void *pm, int tid, int nt) {
  const int G = rt_prime_pairs(N / R, R);
  if (WIDE && G == 16)
    rt_pass_prime64<16, DIR>(buf, N, Ns, R, tw, (const double *)pm, tid, nt);
  else if (WIDE && G == 12)
    rt_pass_prime64<12, DIR>(buf, N, Ns, R, tw, (const double *)pm, tid, nt);
  else
    rt_pass_prime64<8, DIR>(buf, N, Ns, R, tw, (const double *)pm, tid, nt);
}

// In-place transform of 2^lgH interleaved sequences of length d.N held in LDS
// at buf[(i << lgH) + t], with a run-time plan and fft_rt_threads() threads.
// The caller must __syncthreads() after filling buf; the function ends with a
// barrier.  WIDE: also the prime passes of 16 pairs a wave, which a few
// lengths above 13000 need (their registers would cost every other length a
// fifth of the waves: row pass at n = 2448 378 us against 478).
template <int DIR, bool WIDE = false>
__device__ void lds_fft(float2 *buf_, const FftDesc &d, int lgH, int tid, int nt) {
  const LdsPtr buf = (LdsPtr)buf_;
  const TabPtr tw = (TabPtr)d.tw;
  const int N = d.N;
  int Ns = 1, np = 0;
  for (int s = 0; s < d.nr; ++s) {
    const int R = d.r[s];
    switch (R) {
#define TOMO_RT_PASS(r) \
  case r: rt_pass<r, DIR>(buf, N, Ns, tw, lgH, tid, nt); break;
      TOMO_RT_PASS(2) TOMO_RT_PASS(3) TOMO_RT_PASS(4) TOMO_RT_PASS(5) TOMO_RT_PASS(6)
      TOMO_RT_PASS(7) TOMO_RT_PASS(8) TOMO_RT_PASS(9) TOMO_RT_PASS(10) TOMO_RT_PASS(11)
      TOMO_RT_PASS(12) TOMO_RT_PASS(13) TOMO_RT_PASS(14) TOMO_RT_PASS(15) TOMO_RT_PASS(16)
      TOMO_RT_PASS(17) TOMO_RT_PASS(18) TOMO_RT_PASS(20)
#undef TOMO_RT_PASS
      default: rt_prime<DIR, WIDE>(buf, N, Ns, R, tw, d.pm[np++], lgH, tid, nt);
    }
    Ns *= R;
  }
}

// The same for one transform with a plan of the rule's radices (FftPlan::init
// by_rule), in LDS of lds_padded_len(N) elements.  Its error is the smaller one
// where a row is smooth and the result is its high frequencies: the powers of
// two come first, whose differences of near-equal values are exact, and no
// radix is a product with factors between.  What is left of the row's mean
// then sits in one of their outputs.  (Relative error of a ramp-filtered row of
// ellipses without noise, ne = 1016: 1.5e-5 with fft_rt_radices' order, 127 first,
// against 7.6e-6, 6.6e-6 with its pass in 64 bits; 9792 6.6e-5 against 6.0e-5; white
// rows, ne = 4000: 2.1e-7 against 1.8e-7.)  A first pass of a power of two writes
// with a pad slot per 16 elements: its writes, R apart, would meet the same banks.
// WIDE: also the prime passes of 12 and 16 pairs a wave (120 registers against 85).
template <int DIR, bool WIDE>
__device__ void lds_fft_rule(float2 *buf_, const FftDesc &d, int tid, int nt) {
  const LdsPtr buf = (LdsPtr)buf_;
  const TabPtr tw = (TabPtr)d.tw;
  const int N = d.N;
  int Ns = 1, np = 0, s = 0;
  if (d.nr > 1 && d.r[1] <= kFftRegPrime && N % 2 == 0) {
    switch (d.r[0]) {
      case 2: rt_pass<2, DIR, 1>(buf, N, 1, tw, 0, tid, nt); break;
      case 4: rt_pass<4, DIR, 1>(buf, N, 1, tw, 0, tid, nt); break;
      case 8: rt_pass<8, DIR, 1>(buf, N, 1, tw, 0, tid, nt); break;
      case 16: rt_pass<16, DIR, 1>(buf, N, 1, tw, 0, tid, nt); break;
    }
    Ns = d.r[0];
    switch (d.r[1]) {
#define TOMO_RT_PASS(r) \
  case r: rt_pass<r, DIR, 2>(buf, N, Ns, tw, 0, tid, nt); break;
      TOMO_RT_PASS(2) TOMO_RT_PASS(3) TOMO_RT_PASS(4) TOMO_RT_PASS(5) TOMO_RT_PASS(7)
      TOMO_RT_PASS(8) TOMO_RT_PASS(11) TOMO_RT_PASS(13) TOMO_RT_PASS(16) TOMO_RT_PASS(17)
#undef TOMO_RT_PASS
    }
    Ns *= d.r[1];
    s = 2;
  }
  for (; s < d.nr; ++s) {
    const int R = d.r[s];
    switch (R) {
#define TOMO_RT_PASS(r) \
  case r: rt_pass<r, DIR>(buf, N, Ns, tw, 0, tid, nt); break;
      TOMO_RT_PASS(2) TOMO_RT_PASS(3) TOMO_RT_PASS(4) TOMO_RT_PASS(5) TOMO_RT_PASS(7)
      TOMO_RT_PASS(8) TOMO_RT_PASS(11) TOMO_RT_PASS(13) TOMO_RT_PASS(16) TOMO_RT_PASS(17)
#undef TOMO_RT_PASS
      default: rt_prime64<DIR, WIDE>(buf, N, Ns, R, tw, d.pm[np++], tid, nt);
    }
    Ns *= R;
  }
}

// Threads of a workgroup transforming 2^lgH interleaved sequences with a
// run-time plan: as few as hold the passes' butterflies (more resident
// workgroups; N = 2000, row pass, us: 52 with 128 threads, 68 with 256), but
// for lengths up to 1024, whose launches are short, one butterfly per thread;
// -1 if more than 1024 would be needed.
inline int fft_rt_threads(const FftDesc &d, int lgH, bool one_each = true) {
  int64_t t = 64, one = 64;
  for (int i = 0; i < d.nr; ++i) {
    const int R = d.r[i];
    const int64_t nb = (int64_t)(d.N / R) << lgH;
    if (R > kFftRtVals || R == 19)
      t = std::max<int64_t>(t, 64 * rt_prime_waves((int)nb, R, rt_prime_pairs((int)nb, R)));
    else
      t = std::max<int64_t>(t, (nb + rt_maxb(R) - 1) / rt_maxb(R));
    if (R <= kFftRtVals && R != 19) one = std::max(one, nb);
  }
  if (one_each && d.N <= 1024 && one <= 512) t = std::max(t, one);
  t = (t + 63) / 64 * 64;
  return t > 1024 ? -1 : (int)t;
}

// True if the plan has a prime pass of `pairs` pairs a wave or more: 16 for lds_fft's
// WIDE, 12 for lds_fft_rule's.
inline bool fft_rt_wide(const FftDesc &d, int lgH, int pairs = 16) {
  bool wide = false;
  for (int i = 0; i < d.nr; ++i) {
    const int R = d.r[i];
    wide |= (R > kFftRtVals || R == 19) && rt_prime_pairs((d.N / R) << lgH, R) >= pairs;
  }
  return wide;
}

// ---- transforms of a compile-time size ---------------------------------------
// The same Stockham passes with N, the radix sequence, the sub-transform
// lengths, the twiddle steps and the interleave 2^LGH all constants, for
// N = 2^k 3^a 5^b with 2^k >= 256.  The radices are those FftPlan::radices
// picks: radix 16 passes, one radix 8/4/2 pass for the remaining power of
// two, then the radix-3 and radix-5 passes, so every sub-transform length Ns
// is 1 or a multiple of 16 (its index splits are divisions by constants).  With one
// pad slot per 16 elements, the R reads of a butterfly (stride N/R, a multiple of
// 16) and its R writes (stride Ns, a multiple of 16, or consecutive when Ns = 1) sit
// at constant offsets from one base address, so a pass costs one address
// computation per butterfly instead of one per element.
constexpr int ilog2c(int x) { return x <= 1 ? 0 : 1 + ilog2c(x / 2); }

constexpr int count_factor(int x, int p) { return x % p == 0 ? 1 + count_factor(x / p, p) : 0; }
constexpr int ipow(int b, int e) { return e == 0 ? 1 : b * ipow(b, e - 1); }

template <int N>
struct StaticPlan {
  static constexpr int n3 = count_factor(N, 3), n5 = count_factor(N, 5);
  static constexpr int P2 = N / (ipow(3, n3) * ipow(5, n5));
  static_assert(P2 >= 256 && (P2 & (P2 - 1)) == 0, "2^k 3^a 5^b with 2^k >= 256");
  static constexpr int n16 = ilog2c(P2) / 4;
  static constexpr int rest = 1 << (ilog2c(P2) % 4);
  static constexpr int n2p = n16 + (rest > 1 ? 1 : 0);  // passes of the power of two
  static constexpr int passes = n2p + n3 + n5;
  static constexpr int radix(int s) {
    return s < n16 ? 16 : s < n2p ? rest : s < n2p + n3 ? 3 : 5;
  }
};

// (ODD: of the transform at odd frequencies, see chain_first)
template <int R, int Ns, int N, int DIR, int EPT, int LGH, bool ODD = false>
__device__ __forceinline__ void fft_pass_c(float2 *buf, const float2 *__restrict__ tw, int tid,
                                           int nt) {
  constexpr int MAXB = EPT / R;
  constexpr int H = 1 << LGH;
  constexpr int nbPer = N / R;
  constexpr int nb = nbPer << LGH;
  constexpr int twstep = N / (Ns * R);
  static_assert(MAXB >= 1, "EPT must cover the radix");
  static_assert(nbPer % 16 == 0 && (Ns == 1 || Ns % 16 == 0), "constant-offset layout");
  constexpr int rstride = (nbPer + nbPer / 16) << LGH;
  constexpr int wstride = Ns == 1 ? H : (Ns + Ns / 16) << LGH;
  float2 v[MAXB][R];
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int t = g & (H - 1), j = g >> LGH;
      const int base = (lds_pad(j) << LGH) + t;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = buf[base + r * rstride];
      if constexpr (Ns > 1)
        twiddle<R, DIR>(v[q], tw, (unsigned)((ODD ? 2 * (j % Ns) + 1 : j % Ns) * twstep));
      butterfly<R, DIR>(v[q]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int t = g & (H - 1), j = g >> LGH;
      const int k = j % Ns;
      const int base = (lds_pad((j - k) * R + k) << LGH) + t;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[base + r * wstride] = v[q][out_slot<R>(r)];
    }
  }
  __syncthreads();
}

// In-place transform of 2^LGH interleaved sequences of a compile-time length N
// (StaticPlan) held in LDS, element i of sequence t at
// buf[lds_pad(i) * 2^LGH + t]; `tw` is the twiddle table of size N.  Needs
// fft_threads() threads; the caller must __syncthreads() after filling buf,
// and the function ends with a barrier.
// Passes S .. SEnd-1 only (Ns: the sub-transform length entering pass S).
template <int N, int DIR, int EPT, int LGH, int S = 0, int Ns = 1,
          int SEnd = StaticPlan<N>::passes, bool ODD = false>
__device__ __forceinline__ void lds_fft_c(float2 *buf, const float2 *__restrict__ tw, int tid,
                                          int nt) {
  if constexpr (S < SEnd) {
    constexpr int R = StaticPlan<N>::radix(S);
    fft_pass_c<R, Ns, N, DIR, EPT, LGH, ODD>(buf, tw, tid, nt);
    lds_fft_c<N, DIR, EPT, LGH, S + 1, Ns * R, SEnd, ODD>(buf, tw, tid, nt);
  }
}

// ---- compile-time transforms with global input and output --------------
// fft_c_global runs the transform of lds_fft_c, but its first pass takes its
// inputs from ld(i, t) (element i of interleaved sequence t, straight into
// registers) and its last pass hands each output to st(i, t, value) instead
// of writing it to LDS: two LDS sweeps and four barriers fewer than staging
// the input in LDS and reading the result back.  The caller must not use
// `buf` concurrently (it is written without a barrier first) and gets no
// barrier at the end.  Requires at least two passes.

// Pass 0 (Ns = 1, no twiddles) from ld into LDS.
template <int R, int N, int DIR, int EPT, int LGH, typename Ld>
__device__ __forceinline__ void fft_pass_c_first(float2 *buf, int tid, int nt, Ld ld) {
  constexpr int MAXB = EPT / R;
  constexpr int H = 1 << LGH;
  constexpr int nbPer = N / R;
  constexpr int nb = nbPer << LGH;
  static_assert(MAXB >= 1 && nbPer % 16 == 0, "layout");
  float2 v[MAXB][R];
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int t = g & (H - 1), j = g >> LGH;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = ld(j + r * nbPer, t);
    }
  }
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int t = g & (H - 1), j = g >> LGH;
      butterfly<R, DIR>(v[q]);
      const int base = (lds_pad(j * R) << LGH) + t;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[base + r * H] = v[q][out_slot<R>(r)];
    }
  }
}

// The last pass (sub-transform length Ns) from LDS to st.  Outputs outside
// [LO, HI) are dropped, and not computed where all of a register's are outside.
template <int R, int Ns, int N, int DIR, int EPT, int LGH, int LO = 0, int HI = N, typename St>
__device__ __forceinline__ void fft_pass_c_last(const float2 *buf, const float2 *__restrict__ tw,
                                                int tid, int nt, St st) {
  constexpr int MAXB = EPT / R;
  constexpr int H = 1 << LGH;
  constexpr int nbPer = N / R;
  constexpr int nb = nbPer << LGH;
  constexpr int twstep = N / (Ns * R);
  static_assert(MAXB >= 1 && nbPer % 16 == 0 && Ns > 1 && Ns % 16 == 0, "layout");
  constexpr int rstride = (nbPer + nbPer / 16) << LGH;
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int t = g & (H - 1), j = g >> LGH;
      const int base = (lds_pad(j) << LGH) + t;
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = buf[base + r * rstride];
      const int k = j % Ns;
      twiddle<R, DIR>(v, tw, (unsigned)(k * twstep));
      butterfly<R, DIR>(v);
      // (Ns = N / R: k = j, output r is element k + r Ns)
      __builtin_assume(k >= 0 && k < Ns);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if ((r + 1) * Ns <= LO || r * Ns >= HI) continue;
        const int o = k + r * Ns;
        if (o >= LO && o < HI) st(o, t, v[out_slot<R>(r)]);
      }
    }
  }
}

// First pass from ld, the rest in LDS (ends with a barrier, result in buf).
template <int N, int DIR, int EPT, int LGH, typename Ld>
__device__ __forceinline__ void fft_c_from_global(float2 *buf, const float2 *__restrict__ tw,
                                                  int tid, int nt, Ld ld) {
  constexpr int R0 = StaticPlan<N>::radix(0);
  fft_pass_c_first<R0, N, DIR, EPT, LGH>(buf, tid, nt, ld);
  __syncthreads();
  lds_fft_c<N, DIR, EPT, LGH, 1, R0>(buf, tw, tid, nt);
}

template <int N, int DIR, int EPT, int LGH, int LO = 0, int HI = N, typename Ld, typename St>
__device__ __forceinline__ void fft_c_global(float2 *buf, const float2 *__restrict__ tw, int tid,
                                             int nt, Ld ld, St st) {
  using SP = StaticPlan<N>;
  static_assert(SP::passes >= 2, "two passes at least");
  constexpr int R0 = SP::radix(0);
  constexpr int RL = SP::radix(SP::passes - 1);
  fft_pass_c_first<R0, N, DIR, EPT, LGH>(buf, tid, nt, ld);
  __syncthreads();
  lds_fft_c<N, DIR, EPT, LGH, 1, R0, SP::passes - 1>(buf, tw, tid, nt);
  fft_pass_c_last<RL, N / RL, N, DIR, EPT, LGH, LO, HI>(buf, tw, tid, nt, st);
}

// ---- pieces of chained compile-time transforms ------------------------------
// A chain of transforms through one LDS buffer: chain_first takes a thread's
// inputs from ld (which may read the buffer: a barrier separates the reads
// from the writes), lds_fft_c runs the passes between, chain_last leaves the
// outputs in registers.
//
// ODD: the N values of X[m] = sum_j x[j] W_2N^(j (2m + 1)), the transform of
// length 2N of a zero-padded sequence at the odd frequencies.  Splitting j as
// the passes do gives the same butterflies with the twiddles W_(2 Ns R)^((2k + 1) r)
// for W_(Ns R)^(k r) (table index (2k + 1) N / (Ns R) of the table of size 2N),
// in the first pass the constants W_2R^r.

// Pass 0 of N points.  ld(i, s) gives element i; of a power of two length s is
// the thread's element count, i = (tid >> LGH) + s N / EPT.
template <int R, int N, int DIR, int EPT, int LGH, bool ODD, typename Ld>
__device__ __forceinline__ void chain_first(float2 *buf, int tid, int nt, Ld ld) {
  constexpr int MAXB = EPT / R, H = 1 << LGH, nbPer = N / R, nb = nbPer << LGH;
  static_assert(MAXB >= 1 && nbPer % 16 == 0, "layout");
  float2 v[MAXB][R];
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = ld((g >> LGH) + r * nbPer, q + r * MAXB);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      if constexpr (ODD)
        static_for<R>([&](auto r) { v[q][r] = rotate<decltype(r)::value, 2 * R, DIR>(v[q][r]); });
      butterfly<R, DIR>(v[q]);
      const int base = (lds_pad((g >> LGH) * R) << LGH) + (g & (H - 1));
#pragma unroll
      for (int r = 0; r < R; ++r) buf[base + r * H] = v[q][out_slot<R>(r)];
    }
  }
  __syncthreads();
}

// a[r] *= w^(2r + 1), w = exp(DIR pi i k / N): the twiddles W_N^(k r) of a last
// pass and the common factor W_2N^k.  tw2: the table of size 2N.
template <int R, int DIR>
__device__ __forceinline__ void twiddle_mod(float2 *a, const float2 *__restrict__ tw2, int k) {
  auto ld = [&](int m) {
    float2 w = tw2[(unsigned)(k * m)];
    if (DIR > 0) w.y = -w.y;
    return w;
  };
  float2 p[R];
  p[0] = ld(1);
#pragma unroll
  for (int h = 1; h < R; h *= 2) {
    const float2 b = ld(2 * h);
#pragma unroll
    for (int r = h; r < 2 * h && r < R; ++r) p[r] = cmul(p[r - h], b);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) a[r] = cmul(a[r], p[r]);
}

// The last pass; output (k, r) = element k + r N / R of butterfly q goes to
// out[q * R + r].  MOD: times exp(DIR pi i element / N) (tw: the table of size 2N).
template <int R, int N, int DIR, int EPT, int LGH, bool MOD>
__device__ __forceinline__ void chain_last(const float2 *buf, const float2 *__restrict__ tw,
                                           int tid, int nt, float2 *out) {
  constexpr int MAXB = EPT / R, H = 1 << LGH, Ns = N / R, nb = Ns << LGH;
  static_assert(MAXB >= 1 && Ns % 16 == 0, "layout");
  constexpr int rstride = (Ns + Ns / 16) << LGH;
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      const int k = g >> LGH;
      const int base = (lds_pad(k) << LGH) + (g & (H - 1));
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = buf[base + r * rstride];
      if constexpr (MOD)
        twiddle_mod<R, DIR>(v, tw, k);
      else
        twiddle<R, DIR>(v, tw, (unsigned)k);
      butterfly<R, DIR>(v);
      static_for<R>([&](auto r) {
        constexpr int M = decltype(r)::value;
        out[q * R + M] = rotate<MOD ? M : 0, 2 * R, DIR>(v[out_slot<R>(M)]);
      });
    }
  }
}

// ---- compile-time transforms exchanged one component at a time ----------
// fft_c_split is fft_c_global with kFftSplitEPT values per thread kept in
// registers through the whole transform: between passes the real parts go
// through LDS, then the imaginary parts, so the buffer holds 4 bytes per
// element and a workgroup takes twice the sequences.  For the column passes,
// whose sequences are columns, that doubles the bytes a workgroup uses of each
// cache line (a line is read once per workgroup that needs a part of it).
// Outputs outside [LO, HI) are dropped, and not computed where a whole
// register of the last pass is outside.
constexpr int kFftSplitEPT = 32;

// log2 of the sequences a split workgroup takes: as many as 1024 threads hold,
// at most 16 (30 of a thread's values in the radix-3 and 5 passes).
constexpr int split_lg(int N) {
  return ilog2c(1024 * kFftSplitEPT / N) > 4 ? 4 : ilog2c(1024 * kFftSplitEPT / N);
}

// Its radices: those of StaticPlan, but a left-over factor 2 joins the first
// pass (radix 32, without twiddles).
template <int N>
struct SplitPlan {
  using SP = StaticPlan<N>;
  static constexpr bool r32 = SP::rest == 2;
  static constexpr int passes = SP::passes - (r32 ? 1 : 0);
  static constexpr int radix(int s) {
    return !r32 ? SP::radix(s) : s == 0 ? 32 : s < SP::n16 ? 16 : SP::radix(s + 1);
  }
};

// a <- DFT_R(a), outputs in slots out_slot<R>(q).
template <int R, int DIR>
__device__ __forceinline__ void split_butterfly(float2 *a) {
  if constexpr (R == 32)
    dft<32, DIR>(a);
  else
    butterfly<R, DIR>(a);
}

template <int R, int Ns, int N, int DIR, int LGH>
__device__ __forceinline__ void split_butterflies(float2 *v, const float2 *__restrict__ tw,
                                                  int tid, int nt) {
  constexpr int MAXB = kFftSplitEPT / R, nb = (N / R) << LGH;
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
      if constexpr (Ns > 1)
        twiddle<R, DIR>(v + q * R, tw, (unsigned)(((g >> LGH) % Ns) * (N / (Ns * R))));
      split_butterfly<R, DIR>(v + q * R);
    }
  }
}

// Outputs of a radix-R pass (length Ns before it) to the inputs of the next,
// radix R2: v is replaced.
template <int R, int Ns, int R2, int N, int LGH>
__device__ __forceinline__ void split_exchange(float2 *v, float *buf, int tid, int nt) {
  constexpr int MAXB = kFftSplitEPT / R, nb = (N / R) << LGH, H = 1 << LGH;
  constexpr int MAXB2 = kFftSplitEPT / R2, nb2 = (N / R2) << LGH;
  static_assert((N / R) % 16 == 0 && (N / R2) % 16 == 0 && (Ns == 1 || Ns % 16 == 0), "layout");
  // (output r of the first pass is element j R + r: a pad slot after 16)
  constexpr int wstride = Ns == 1 ? H : (Ns + Ns / 16) << LGH;
  constexpr int wpad = Ns == 1 ? H : 0;
  constexpr int rstride = (N / R2 + N / R2 / 16) << LGH;
  float x[kFftSplitEPT];
  auto write = [&](auto part) {
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
      const int g = tid + q * nt;
      if (g < nb) {
        const int t = g & (H - 1), j = g >> LGH, k = j % Ns;
        float *o = buf + (lds_pad((j - k) * R + k) << LGH) + t;
#pragma unroll
        for (int r = 0; r < R; ++r)
          o[r * wstride + (r >> 4) * wpad] = part(v[q * R + out_slot<R>(r)]);
      }
    }
  };
  auto read = [&](auto put) {
#pragma unroll
    for (int q = 0; q < MAXB2; ++q) {
      const int g = tid + q * nt;
      if (g < nb2) {
        const int t = g & (H - 1), j = g >> LGH;
        const float *i = buf + (lds_pad(j) << LGH) + t;
#pragma unroll
        for (int r = 0; r < R2; ++r) put(q * R2 + r, i[r * rstride]);
      }
    }
  };
  write([](float2 a) { return a.x; });
  __syncthreads();
  read([&](int i, float a) { x[i] = a; });
  __syncthreads();
  write([](float2 a) { return a.y; });
  __syncthreads();
  read([&](int i, float a) { v[i] = make_float2(x[i], a); });
}

template <int N, int DIR, int LGH, int LO, int HI, int S, int Ns, typename St>
__device__ __forceinline__ void split_rest(float2 *v, float *buf, const float2 *__restrict__ tw,
                                           int tid, int nt, St st) {
  using SP = SplitPlan<N>;
  constexpr int R = SP::radix(S);
  split_butterflies<R, Ns, N, DIR, LGH>(v, tw, tid, nt);
  if constexpr (S + 1 < SP::passes) {
    if constexpr (S > 0) __syncthreads();  // the last exchange's reads
    split_exchange<R, Ns, SP::radix(S + 1), N, LGH>(v, buf, tid, nt);
    split_rest<N, DIR, LGH, LO, HI, S + 1, Ns * R>(v, buf, tw, tid, nt, st);
  } else {
    constexpr int MAXB = kFftSplitEPT / R, nb = (N / R) << LGH, H = 1 << LGH;
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
      const int g = tid + q * nt;
      if (g < nb) {
        const int t = g & (H - 1), j = g >> LGH;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if ((r + 1) * Ns <= LO || r * Ns >= HI) continue;
          const int o = j + r * Ns;
          if (o >= LO && o < HI) st(o, t, v[q * R + out_slot<R>(r)]);
        }
      }
    }
  }
}

// The passes S .. of a transform whose values stay in registers (v: the inputs
// of pass S, then the outputs of the last pass in its order).
template <int N, int DIR, int LGH, int S, int Ns>
__device__ __forceinline__ void split_regs(float2 *v, float *buf, const float2 *__restrict__ tw,
                                           int tid, int nt) {
  using SP = SplitPlan<N>;
  constexpr int R = SP::radix(S);
  // (a pass computes its own addresses: kept from one for the next, they and
  // the 64 registers of v would not fit 128)
  asm volatile("" : "+v"(tid));
  split_butterflies<R, Ns, N, DIR, LGH>(v, tw, tid, nt);
  if constexpr (S + 1 < SP::passes) {
    __syncthreads();  // the last exchange's reads, of this transform or the one before
    split_exchange<R, Ns, SP::radix(S + 1), N, LGH>(v, buf, tid, nt);
    split_regs<N, DIR, LGH, S + 1, Ns * R>(v, buf, tw, tid, nt);
  }
}

// Threads of fft_split_regs: every one holds kFftSplitEPT values.
constexpr int split_threads(int N, int LGH) { return (N << LGH) / kFftSplitEPT; }

// Transform of 2^LGH interleaved sequences of a power of two length N in
// registers, thread tid of split_threads(N, LGH) holding elements
// (tid >> LGH) + s N / 32 of sequence tid mod 2^LGH in a[s], before and after.
// buf: lds_padded_len(N) << LGH floats (a barrier precedes its first use).
template <int N, int DIR, int LGH>
__device__ __forceinline__ void fft_split_regs(float2 *a, float *buf,
                                               const float2 *__restrict__ tw, int tid) {
  using SP = SplitPlan<N>;
  static_assert((N & (N - 1)) == 0, "every butterfly of every pass has a thread");
  constexpr int E = kFftSplitEPT, R0 = SP::radix(0), RL = SP::radix(SP::passes - 1);
  float2 v[E];
#pragma unroll
  for (int q = 0; q < E / R0; ++q)
#pragma unroll
    for (int r = 0; r < R0; ++r) v[q * R0 + r] = a[q + r * (E / R0)];
  split_regs<N, DIR, LGH, 0, 1>(v, buf, tw, tid, split_threads(N, LGH));
#pragma unroll
  for (int q = 0; q < E / RL; ++q)
#pragma unroll
    for (int r = 0; r < RL; ++r) a[q + r * (E / RL)] = v[q * RL + out_slot<RL>(r)];
}

// buf: lds_padded_len(N) << LGH floats.
template <int N, int DIR, int LGH, int LO, int HI, typename Ld, typename St>
__device__ __forceinline__ void fft_c_split(float *buf, const float2 *__restrict__ tw, int tid,
                                            int nt, Ld ld, St st) {
  constexpr int R = SplitPlan<N>::radix(0);
  constexpr int MAXB = kFftSplitEPT / R, nb = (N / R) << LGH, H = 1 << LGH;
  float2 v[kFftSplitEPT];
#pragma unroll
  for (int q = 0; q < MAXB; ++q) {
    const int g = tid + q * nt;
    if (g < nb) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[q * R + r] = ld((g >> LGH) + r * (N / R), g & (H - 1));
    }
  }
  split_rest<N, DIR, LGH, LO, HI, 0, 1>(v, buf, tw, tid, nt, st);
}

// Calls f(std::integral_constant<int, N>) for the sizes with a compiled
// specialisation (2^k; 3, 9, 5 and 15 times a power of two: the detector
// widths 2^k, 3 2^k, 1152/2304, 1280/2560 and 1920), f(std::integral_constant
// <int, 0>) otherwise.
template <typename F>
inline void with_static_size(int N, F &&f) {
  switch (N) {
    case 256: f(std::integral_constant<int, 256>()); break;
    case 512: f(std::integral_constant<int, 512>()); break;
    case 768: f(std::integral_constant<int, 768>()); break;
    case 1280: f(std::integral_constant<int, 1280>()); break;
    case 1536: f(std::integral_constant<int, 1536>()); break;
    case 2304: f(std::integral_constant<int, 2304>()); break;
    case 2560: f(std::integral_constant<int, 2560>()); break;
    case 3072: f(std::integral_constant<int, 3072>()); break;
    case 3840: f(std::integral_constant<int, 3840>()); break;
    case 4608: f(std::integral_constant<int, 4608>()); break;
    case 5120: f(std::integral_constant<int, 5120>()); break;
    case 6144: f(std::integral_constant<int, 6144>()); break;
    case 1024: f(std::integral_constant<int, 1024>()); break;
    case 2048: f(std::integral_constant<int, 2048>()); break;
    case 4096: f(std::integral_constant<int, 4096>()); break;
    case 8192: f(std::integral_constant<int, 8192>()); break;
    default: f(std::integral_constant<int, 0>()); break;
  }
}

// True if N has a compiled specialisation.
inline bool static_fft_size(int N) {
  bool ok = false;
  with_static_size(N, [&](auto ns) { ok = decltype(ns)::value > 0; });
  return ok;
}

// Maps a flattened workgroup id to a logical one such that the workgroups the
// dispatcher sends to one XCD (round robin over 8 XCDs) receive consecutive
// logical ids: neighbouring tiles then share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int id, int total) {
  const int q = total / 8, r = total % 8;
  const int x = id % 8, i = id / 8;
  return x * q + min(x, r) + i;
}

// Copies `count` items into LDS with U global loads of each thread in flight
// at once (all loads of a round are issued before the first LDS store, so
// the round costs one memory latency rather than U): item i is produced by
// ld(i) and written by st(i, value).
template <int U, typename T, typename Ld, typename St>
__device__ __forceinline__ void stage_lds(int count, int tid, int nt, Ld ld, St st) {
  for (int base = tid; base < count; base += U * nt) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u * nt;
      if (i < count) v[u] = ld(i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = base + u * nt;
      if (i < count) st(i, v[u]);
    }
  }
}

// Workgroup size for transforming `elems` complex values (all interleaved
// sequences) of a compiled size, and the size by which a width is accepted:
// 16 values per thread for radices 2/4/8/16, fewer with a radix-3, 5, 7, 11 or
// 13 pass (15, 15, 14, 11, 13: whole butterflies); at least 256 and a multiple
// of 64.  Returns -1 if more than 1024 threads would be needed.
inline int fft_threads(const FftRule &d, int64_t elems, int ept = kFftEPT) {
  int64_t per = ept;  // values a thread covers in every pass: whole butterflies
  for (int i = 0; i < d.nr; ++i) {
    const int R = d.r[i];
    if (R <= 8 || R == 16 || (R <= 17 && R <= ept)) per = std::min<int64_t>(per, (ept / R) * R);
  }
  int64_t t = (elems + per - 1) / per;
  t = ((t + 63) / 64) * 64;
  if (t > 1024) return -1;
  return (int)(t < 256 ? 256 : t);
}

// True if N has a prime factor other than 2 and 3.
inline bool fft_general(int64_t N) {
  if (N < 1) return false;
  while (N % 2 == 0) N /= 2;
  while (N % 3 == 0) N /= 3;
  return N != 1;
}

// True if N >= 1 and every prime factor of N is at most kFftMaxPrime.
inline bool fft_size_ok(int64_t N) {
  if (N < 1) return false;
  for (int64_t p = 2; p <= kFftMaxPrime; ++p)
    while (N % p == 0) N /= p;
  return N == 1;
}

}  // namespace tomo
