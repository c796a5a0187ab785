// Fourier-wavelet stripe removal (tomocupy remove_stripe_fw,
// src/tomocupy/processing/remove_stripe.py:253-293) for gfx950; scans of few
// angles take the band-by-band form of stripe_bands.hip (fw_few_angles).
//
// Per slice of a (nproj, nz, n) chunk: zero-pad the angles to
// nproj + nproj/8 (centred), `level` separable DWT levels (detector axis, then
// angle axis; half-sample symmetric extension, stride-2 correlation with the
// reversed decomposition taps, as afb1d :91-129), notch filter of the
// detector-high/angle-low band along angles, then the synthesis filter banks
// (sfb1d :132-156) back up and the crop to the original rows.
//
// The notch irfft(rfft(x) * (1 - g), my) with g_k = exp(-yhat_k^2/(2 sigma^2))
// (:270-281) equals x - irfft(rfft(x) * g); g falls below 1e-9 after a few
// frequencies, so the correction of the band is a sum over the kept
// frequencies, exact to far below float32 resolution.
//
// Only that band changes, and the synthesis bank is linear and reconstructs
// its analysis input exactly, so the output is x_0 + d_0 with d_0 the
// synthesis of the bands' corrections alone.  Every step from x_0 to d_0 is
// linear and separable in angle and detector, and the notch keeps only a few
// angular patterns (cosines and sines) of each level, so
//   d_0[p][j] = sum_r A_r[p] B_r[j],   B_r = S_r(-g_r D_r(P_r)),
//   P_r[j]    = sum_p T_r[p] x_0[p][j],
// one term r per level and kept cosine or sine: T_r is that pattern taken
// back through the levels' angle low-passes (their transposes), A_r the same
// pattern through the angle synthesis, D_r and S_r the level's detector
// analysis (low-pass on the levels above, then high-pass) and synthesis.  A_r
// and T_r depend on the sizes only and are built once, in FP64
// (k_fw_tables).  A chunk then takes three launches instead of four full-size
// filter passes per level:
//   k_fw_project   P = T x_0, a matrix product with K = angles
//   k_fw_detector  P_r -> B_r, one workgroup per term and slice, all levels
//   k_fw_apply     x_0 + A B, a matrix product with K = terms, fused with the
//                  dark/flat correction, -log and the swap to sinograms
// At sigma = 1 and 7 levels there are 83 terms (96 padded); the products are 9 GFLOP
// per 8 slices of 2048 x 1500, far below what the matrix cores take for the
// bytes of x_0.  Measured, 8 slices of 2048 x 1500 (sym16, 7 levels, sigma 1),
// us: 47 + 38 + 52 and 6 for the dark/flat means, against 456 for the filter
// passes over full-size bands (29 launches); proc_chunk 462 -> 150, whose floor,
// the counts read and the sinograms written at the rate of a copy, is 29.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>

#include "common.h"
#include "fft_lds.h"
#include "precision.h"
#include "preproc.h"
#include "wavelets.h"

using namespace tomo;

namespace {

constexpr int kMaxLevels = 16;
constexpr int kGroups = 8;      // angle groups (= waves) of a k_fw_project workgroup
constexpr int kRowTiles = 6;    // 16-term tiles a k_fw_project wave accumulates
constexpr int kApplyCols = 128; // columns of a k_fw_apply workgroup (32 per wave)

// Filter taps in FP64.  The wavelets are orthogonal: with a the analysis
// low-pass (reversed decomposition filter, DWTForward, :176-183), the synthesis
// low-pass (as given, DWTInverse, :221-225) is a too, and both high-passes are
// b[j] = (-1)^j a[L - 1 - j].  One set of taps, 64 scalar registers, stays
// resident through k_fw_detector (four sets spilled to vector lanes: 50 us
// against 46 at 83 terms x 8 slices x 2048).
struct Taps {
  double a[32];
};

// Tap j of the low (HI = 0) or high pass.
template <int L, int HI>
__device__ __forceinline__ double tap(const Taps &t, int j) {
  return HI ? (j & 1 ? -t.a[L - 1 - j] : t.a[L - 1 - j]) : t.a[j];
}

// Lengths of an axis: N[0] the axis, N[i + 1] = (N[i] + L - 1) / 2.
struct AxisLen {
  int N[kMaxLevels + 1];
};

// One term: the cosine (sin = 0) or sine (sin = 1) of frequency q of level k.
struct FwTerm {
  int k, q, sin;
  float gk;  // c_q g_q / my
};

// Compile-time filter lengths of the supported wavelets (haar 2, db5 and sym5
// 10, sym16 32).
template <int V>
using IC = std::integral_constant<int, V>;

template <typename F>
void with_len(int L, F &&f) {
  if (L == 2)
    f(IC<2>());
  else if (L == 10)
    f(IC<10>());
  else
    f(IC<32>());
}

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mma(bf8_t a, bf8_t b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x = p0 + p1 + p2 to 24 bits in bfloat16 parts (any float32 range).
__device__ __forceinline__ void split_bf16(float x, __bf16 &p0, __bf16 &p1, __bf16 &p2) {
  p0 = (__bf16)x;
  const float r = x - (float)p0;
  p1 = (__bf16)r;
  p2 = (__bf16)(r - (float)p1);
}

// Transpose of the angle low-pass (analysis length N -> No), one output h:
// the sum over the extended positions m that reflect to h.
__device__ double lowpass_t(const double *t, int N, int No, const double *a, int L, int h) {
  const int pad = (2 * (No - 1) - N + L) / 2, P = 2 * N;
  const int lo = -pad, hi = 2 * No + L - 2 - pad;
  double s = 0.0;
  for (int side = 0; side < 2; ++side) {
    int m = side ? -1 - h : h;
    while (m < lo) m += P;
    while (m - P >= lo) m -= P;
    for (; m < hi; m += P) {
      const int i = m + pad;
      for (int j = i & 1; j < L; j += 2) {
        const int o = (i - j) / 2;
        if (o >= 0 && o < No) s += a[j] * t[o];
      }
    }
  }
  return s;
}

// Synthesis low-pass (length N -> the first outputs), output t after the
// L - 2 crop of sfb1d.
__device__ __forceinline__ double synth_at(const double *x, const double *g, int L, int t) {
  const int tt = t + L - 2, i = tt >> 1;
  double s = 0.0;
  for (int m = 0; m < L / 2; ++m) s += g[2 * m + (tt & 1)] * x[i - m];
  return s;
}

// The tables of one term r per workgroup, in FP64 (once per plan and
// settings; scratch: two rows of `len` doubles per term):
//   T   T_r in matrix-operand order [part][p / 8][Rp][p % 8], three bfloat16
//       parts
//   TS  (kGroups, Rp): sums of T_r over the angle groups of k_fw_project
//   A   A_r in matrix-operand order [part][r / 8][Pa][r % 8], three bfloat16
//       parts
// Angles past nproj and terms past the last one are zero.
__global__ __launch_bounds__(256) void k_fw_tables(const FwTerm *__restrict__ terms, int R, int Rp,
                                                   Taps tp, int L, AxisLen H, int len, int st,
                                                   int nproj, int Pt, int Pa, int steps,
                                                   double *__restrict__ scratch, int r0,
                                                   __bf16 *__restrict__ T,
                                                   double *__restrict__ TS,
                                                   __bf16 *__restrict__ A) {
  __shared__ double sh[256];
  const int r = r0 + blockIdx.x, tid = threadIdx.x;
  const bool live = r < R;
  const FwTerm tm = live ? terms[r] : FwTerm{0, 0, 0, 0.f};
  double *buf[2] = {scratch + (size_t)blockIdx.x * 2 * len,
                    scratch + (size_t)blockIdx.x * 2 * len + len};
  for (int pass = 0; pass < 2; ++pass) {
    int cur = 0;
    if (live) {
      const int my = H.N[tm.k + 1];
      for (int i = tid; i < my; i += 256) {
        const double ang = 2.0 * (double)(((int64_t)tm.q * i) % my) / (double)my;
        buf[0][i] = tm.sin ? sinpi(ang) : cospi(ang);
      }
      __syncthreads();
      for (int k = tm.k; k >= 0; --k, cur ^= 1) {
        for (int h = tid; h < H.N[k]; h += 256)
          buf[cur ^ 1][h] = pass == 0 ? lowpass_t(buf[cur], H.N[k], H.N[k + 1], tp.a, L, h)
                                      : synth_at(buf[cur], tp.a, L, h);
        __syncthreads();
      }
    }
    const double *res = buf[cur] + st;
    if (pass == 1) {
      for (int p = tid; p < Pa; p += 256) {
        __bf16 q0, q1, q2;
        split_bf16(live && p < nproj ? (float)res[p] : 0.f, q0, q1, q2);
        const size_t o = ((size_t)(r / 8) * Pa + p) * 8 + r % 8, part = (size_t)Rp * Pa;
        A[o] = q0;
        A[o + part] = q1;
        A[o + 2 * part] = q2;
      }
      continue;
    }
    for (int p = tid; p < Pt; p += 256) {
      __bf16 q0, q1, q2;
      split_bf16(live && p < nproj ? (float)res[p] : 0.f, q0, q1, q2);
      const size_t o = ((size_t)(p / 8) * Rp + r) * 8 + p % 8, part = (size_t)Rp * Pt;
      T[o] = q0;
      T[o + part] = q1;
      T[o + 2 * part] = q2;
    }
    // 32 threads per angle group of 32 * steps angles
    const int grp = tid >> 5, p0 = grp * steps * 32;
    double s = 0.0;
    if (live)
      for (int p = p0 + (tid & 31); p < min(nproj, p0 + steps * 32); p += 32) s += res[p];
    sh[tid] = s;
    __syncthreads();
    if (tid < kGroups) {
      double t = 0.0;
      for (int i = 0; i < 32; ++i) t += sh[tid * 32 + i];
      TS[(size_t)tid * Rp + r] = t;
    }
    __syncthreads();
  }
}

// (count - d0) / f0 rounded as the division is, for many counts of a column:
// with y the rounded reciprocal of f0, q = a y is within an ulp of the
// quotient, its remainder a - q f0 is exact and one correction rounds to the
// quotient (Markstein).  f0 and y are far from overflow and underflow
// (a is 0 or a difference of a count and a mean); otherwise (y = 0) the
// division.
struct ColumnFlat {
  float d0, f0, y;
  __device__ __forceinline__ void set(float d, float fa) {
    d0 = d;
    f0 = flat0(fa, d);
    y = fabsf(f0) > 1e-20f && fabsf(f0) < 1e20f ? 1.0f / f0 : 0.0f;
  }
  __device__ __forceinline__ float operator()(float x) const {
    const float a = x - d0;
    if (y == 0.0f) return a / f0;
    const float q = a * y;
    return fmaf(fmaf(-q, f0, a), y, q);
  }
};

// P[z][r][j] = sum_p T_r[p] x_0[p][z][j], stored in FP64: the angle
// contraction of the stripe removal on the matrix cores.
//
// SRC 0: x_0 is the float32 chunk; 1: dark/flat corrected counts; 2: the same
// with the flat interpolated over the angles.
//
// A wave takes 16 CT columns (a lane CT neighbours of them: one load per angle
// where `vec`, the alignment, allows it) and one of the kGroups angle groups
// and accumulates up to kRowTiles x CT tiles of 16 terms x 16 columns, 32
// angles per instruction; the groups' sums are added in FP64, in group order, in LDS.
// So that the float32 accumulators only carry the variation of a column over
// the group's angles, each wave subtracts its column's value at the middle
// angle of the group and puts it back with the sum of T over the group
// (TS, FP64).  Three bfloat16 parts of x_0 and T (24 bits, any float32 range),
// the six products down to 2^-16 of a product.
//
// What bounds it (47 us per 8 slices of 2048 x 1500; 26 with one tile pair
// instead of six): vector work (the quotient and the split, about 12 instructions per
// value) for 36 % of the cycles, matrix work (11 us) for 24 %, which do not overlap,
// and between them the loads' latency; T is re-read from L2 for each
// 16 CT columns.  CT = 4 (half the reads of T, but 2 waves per SIMD instead of
// 4) measured 52 us against 46.
template <int SRC, int CT>
__global__ __launch_bounds__(64 * kGroups) void k_fw_project(
    const void *__restrict__ src_, const __bf16 *__restrict__ T, const double *__restrict__ TS,
    double *__restrict__ P, int nproj, int nz, int n, int Rp, int Pt, int steps, int ncb,
    int vec, DarkFlat df) {
  using RAW = typename std::conditional<SRC == 0, float, uint16_t>::type;
  __shared__ double red[kGroups][16][16 * CT];
  // neighbouring column blocks share cache lines of the counts: same XCD
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int c0 = (id % ncb) * 16 * CT, z = id / ncb, rt0 = blockIdx.y * kRowTiles;
  const int nrt = min(kRowTiles, Rp / 16 - rt0);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = lane & 15, g = lane >> 4;
  const int s0 = w * steps;
  const int s1 = min((w + 1) * steps, (nproj + 31) / 32);
  const size_t rs = (size_t)nz * n;  // elements from one angle to the next
  struct alignas(CT * sizeof(RAW)) RawN {
    RAW v[CT];
  };
  auto column = [&](int t) { return (size_t)z * n + min(c0 + CT * i + t, n - 1); };
  const RAW *src = static_cast<const RAW *>(src_);
  const RAW *src_v = src + (size_t)z * n + min(c0 + CT * i, n - CT);
  ColumnFlat cf[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    if constexpr (SRC == 1) cf[t].set(df.d0[column(t)], df.fa[column(t)]);
  }
  auto value = [&](RAW raw, int t, int p) {
    if constexpr (SRC == 2) {
      const size_t zx = column(t);
      const float v = nproj > 1 ? (float)((double)p / (double)(nproj - 1)) : 0.f;
      return darkflat((float)raw, df.d0[zx], df.fa[zx], df.fb[zx], v, 1);
    } else if constexpr (SRC == 1) {
      return cf[t]((float)raw);
    } else {
      return raw;
    }
  };
  floatx4 acc[kRowTiles][CT];
#pragma unroll
  for (int a = 0; a < kRowTiles; ++a)
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[a][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the column's value at the middle angle of the group
  float ref[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int pm = min(32 * s0 + 16 * steps, nproj - 1);
    ref[t] = s0 < s1 ? value(src[column(t) + (size_t)pm * rs], t, pm) : 0.f;
  }
  RawN raw[8];
  auto fetch = [&](int s) {
    const int p = 32 * s + 8 * g;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const size_t o = (size_t)min(p + u, nproj - 1) * rs;
      if (vec) {
        raw[u] = *reinterpret_cast<const RawN *>(src_v + o);
      } else {
#pragma unroll
        for (int t = 0; t < CT; ++t) raw[u].v[t] = src[column(t) + o];
      }
    }
  };
  if (s0 < s1) fetch(s0);
  const __bf16 *Tl = T + ((size_t)g * Rp + 16 * rt0 + i) * 8;
  const size_t part = (size_t)Rp * Pt;
  for (int s = s0; s < s1; ++s) {
    bf8_t x[CT][3];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        __bf16 q0, q1, q2;
        const int p = min(32 * s + 8 * g + u, nproj - 1);
        split_bf16(value(raw[u].v[t], t, p) - ref[t], q0, q1, q2);
        x[t][0][u] = q0;
        x[t][1][u] = q1;
        x[t][2][u] = q2;
      }
    if (s + 1 < s1) fetch(s + 1);
    const __bf16 *Ts = Tl + (size_t)(4 * s) * Rp * 8;
#pragma unroll
    for (int a = 0; a < kRowTiles; ++a) {
      if (a < nrt) {
        bf8_t m[3];
#pragma unroll
        for (int q = 0; q < 3; ++q)
          m[q] = *reinterpret_cast<const bf8_t *>(Ts + q * part + (size_t)(16 * a) * 8);
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int v = 0; q + v < 3; ++v) acc[a][t] = mma(m[q], x[t][v], acc[a][t]);
      }
    }
  }
  // add the groups' sums, one tile of terms at a time
#pragma unroll
  for (int a = 0; a < kRowTiles; ++a) {
    if (a >= nrt) break;
    const int rb = 16 * (rt0 + a);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 4 * g + j;
      const double ts = TS[(size_t)w * Rp + rb + row];
#pragma unroll
      for (int t = 0; t < CT; ++t)
        red[w][row][CT * i + t] = (double)acc[a][t][j] + (double)ref[t] * ts;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 256 * CT; e += 64 * kGroups) {
      const int row = e / (16 * CT), c = e % (16 * CT);
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < kGroups; ++q) s += red[q][row][c];
      if (c0 + c < n) P[((size_t)z * Rp + rb + row) * n + c0 + c] = s;
    }
  }
}

// A band of length N with its half-sample mirrored margins: the analysis reads
// positions [-(L - 2), N + L + 2).
template <int L>
__device__ __forceinline__ void put_mirrored(double *x, int N, int o, double v) {
  constexpr int kLo = L - 2, kHi = L + 2;
  x[o] = v;
  if (o < kLo) x[-1 - o] = v;
  if (o >= N - kHi) x[2 * N - 1 - o] = v;
  if (N < kHi) {  // a band shorter than its margins: the further images
    for (int m = 2 * N; m < N + kHi + kLo; m += 2 * N) {
      if (o - m >= -kLo) x[o - m] = v;
      if (-1 - o - m >= -kLo) x[-1 - o - m] = v;
      if (o + m < N + kHi) x[o + m] = v;
      if (2 * N - 1 - o + m < N + kHi) x[2 * N - 1 - o + m] = v;
    }
  }
}

// Analysis outputs o, o+1 of the mirrored band x: positions 2o - (L - 2) on.
template <int L, int HI>
__device__ __forceinline__ void analysis2(const double *x, const Taps &t, int o, double *y) {
  const double *p = x + 2 * o - (L - 2);
  double v[L + 2];
#pragma unroll
  for (int j = 0; j < L + 2; ++j) v[j] = p[j];
  // (even and odd taps apart: shorter chains)
  double s0 = 0.0, s1 = 0.0, u0 = 0.0, u1 = 0.0;
#pragma unroll
  for (int j = 0; j < L; j += 2) {
    s0 = fma(tap<L, HI>(t, j), v[j], s0);
    s1 = fma(tap<L, HI>(t, j), v[j + 2], s1);
    u0 = fma(tap<L, HI>(t, j + 1), v[j + 1], u0);
    u1 = fma(tap<L, HI>(t, j + 1), v[j + 3], u1);
  }
  y[0] = s0 + u0;
  y[1] = s1 + u1;
}

// Synthesis outputs 2q, 2q+1 (after the L - 2 crop) of x: both read x[q ..
// q + L/2 - 1], through the even and the odd taps.
template <int L, int HI>
__device__ __forceinline__ void synthesis2(const double *x, const Taps &t, int q, double *y) {
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int m = 0; m < L / 2; ++m) {
    const double v = x[q + L / 2 - 1 - m];
    s0 = fma(tap<L, HI>(t, 2 * m), v, s0);
    s1 = fma(tap<L, HI>(t, 2 * m + 1), v, s1);
  }
  y[0] = s0;
  y[1] = s1;
}

// P_r -> B_r for one term and slice per workgroup: the detector axis through
// the level's analysis (k low-passes, one high-pass), times -g_r, and back up
// (one high-pass, k low-passes), in FP64 (the contraction's large smooth part
// cancels in the high-pass), two rows of `len` doubles in LDS (GLOB: in
// scratch, for detectors too wide for the LDS).  B goes out as three bfloat16
// parts in matrix-operand order [z][part][r / 8][nPad][r % 8]; terms past the
// last one are zero.  Bound by the chain of up to 2 (k + 1) dependent passes:
// the mirrored margins are written with the bands, so that a pass is one round
// of constant-offset LDS reads and one barrier (38 us at 83 terms x 8 slices x
// 2048 columns; 63 with the reflection worked out per read).
template <int L, bool GLOB>
__global__ __launch_bounds__(256) void k_fw_detector(const double *__restrict__ P,
                                                     __bf16 *__restrict__ B,
                                                     const FwTerm *__restrict__ terms, int R,
                                                     int Rp, Taps tp, AxisLen W, int nPad,
                                                     int len, double *__restrict__ scratch) {
  extern __shared__ double rows[];
  const int r = blockIdx.x, z = blockIdx.y, n = W.N[0], tid = threadIdx.x;
  __bf16 *out = B + (size_t)z * 3 * Rp * nPad + (size_t)(r / 8) * nPad * 8 + r % 8;
  const size_t part = (size_t)Rp * nPad;
  if (r >= R) {
    for (int j = tid; j < n; j += 256)
      out[(size_t)j * 8] = out[(size_t)j * 8 + part] = out[(size_t)j * 8 + 2 * part] = (__bf16)0.f;
    return;
  }
  const FwTerm tm = terms[r];
  const double *Pr = P + ((size_t)z * Rp + r) * n;
  // row 0 or 1, past its margin (an offset, not a pointer table, so that the
  // accesses stay LDS accesses)
  auto row = [&](int c) -> double * {
    if constexpr (GLOB)
      return scratch + ((size_t)z * Rp + r) * 2 * len + c * len + L;
    else
      return rows + (c * len + L);
  };
  for (int j0 = tid; j0 < n; j0 += 8 * 256) {  // (8 loads of a thread in flight)
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = Pr[min(j0 + 256 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (j0 + 256 * u < n) put_mirrored<L>(row(0), n, j0 + 256 * u, v[u]);
  }
  __syncthreads();
  int cur = 0;
  for (int k = 0; k < tm.k; ++k, cur ^= 1) {
    const int No = W.N[k + 1];
    for (int o = 2 * tid; o < No; o += 512) {
      double v[2];
      analysis2<L, 0>(row(cur), tp, o, v);
      put_mirrored<L>(row(cur ^ 1), No, o, v[0]);
      if (o + 1 < No) put_mirrored<L>(row(cur ^ 1), No, o + 1, v[1]);
    }
    __syncthreads();
  }
  {
    const int No = W.N[tm.k + 1];
    double *y = row(cur ^ 1);
    for (int o = 2 * tid; o < No; o += 512) {
      double v[2];
      analysis2<L, 1>(row(cur), tp, o, v);
      y[o] = v[0] * -(double)tm.gk;
      if (o + 1 < No) y[o + 1] = v[1] * -(double)tm.gk;
    }
    __syncthreads();
    cur ^= 1;
  }
  for (int k = tm.k; k >= 0; --k, cur ^= 1) {
    const int N = W.N[k];
    const double *x = row(cur);
    double *y = row(cur ^ 1);
    for (int q = tid; 2 * q < N; q += 256) {
      double v[2];
      if (k == tm.k)
        synthesis2<L, 1>(x, tp, q, v);
      else
        synthesis2<L, 0>(x, tp, q, v);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int j = 2 * q + c;
        if (j >= N) break;
        if (k > 0) {
          y[j] = v[c];
        } else {
          __bf16 q0, q1, q2;
          split_bf16((float)v[c], q0, q1, q2);
          out[(size_t)j * 8] = q0;
          out[(size_t)j * 8 + part] = q1;
          out[(size_t)j * 8 + 2 * part] = q2;
        }
      }
    }
    __syncthreads();
  }
}

// x_0 + sum_r A_r[p] B_r[j].  MODE 1: x_0 and the result are the float32 chunk
// res[p][z][x], in place.  MODE 2: x_0 = darkflat(counts[p][z][x]) and the
// result goes out as TO in sinogram order out[z][p][x], after minus_log when
// take_log (proc_proj and the swap of rec.py:174); 3: the same with the flat
// interpolated over the angles.
//
// A workgroup takes 128 columns (a wave 32 of them) and na tiles of 16 angles
// (two at a time); columns are the rows of the matrix product, so a lane holds
// 4 neighbouring columns of one angle (8-byte loads of counts, 16-byte stores;
// `vec`: widths and arrays aligned for them).  Three bfloat16 parts of A and
// B, the six products down to 2^-16 of a term: the correction keeps 24 bits.
// KS > 0: Rp = 32 KS, the workgroup's part of B in LDS; 0: any number of
// terms, B from L2 for each angle tile.  8 slices of 2048 x 1500: 52 us at 96
// terms, 35 at 32; reading the counts and writing the sinograms alone takes 29,
// and 11 us of matrix work and the logarithm's vector work overlap them in
// part.  (B in registers, 2 waves per SIMD: 86 us.)
template <int MODE, typename TO, int KS>
__global__ __launch_bounds__(512, MODE == 3 ? 2 : 4) void k_fw_apply(const void *src_, TO *out_,
                                                     const __bf16 *__restrict__ A,
                                                     const __bf16 *__restrict__ B, int nproj,
                                                     int nz, int n, int Rp, int Pa, int nPad,
                                                     int na, int vec, int take_log, DarkFlat df) {
  extern __shared__ bf8_t sB[];  // [part][r / 8][128]
  const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int z = blockIdx.z;
  const int b0 = blockIdx.x * kApplyCols, cw = 32 * (w & 3), c0 = b0 + cw;
  const size_t apart = (size_t)Rp * Pa;
  const bf8_t *Bz = reinterpret_cast<const bf8_t *>(B) + (size_t)z * 3 * (Rp / 8) * nPad + b0;
  if constexpr (KS > 0) {
    constexpr int kN = 3 * 4 * KS * kApplyCols;
    for (int e = threadIdx.x; e < kN; e += 512)
      sB[e] = Bz[(size_t)(e / kApplyCols) * nPad + e % kApplyCols];
    __syncthreads();
  }
  auto ldB = [&](int ks, int t, int q) {
    const int row = q * (Rp / 8) + 4 * ks + g, c = cw + 16 * t + i;
    if constexpr (KS > 0)
      return sB[(q * 4 * KS + 4 * ks + g) * kApplyCols + c];
    else
      return Bz[(size_t)row * nPad + c];
  };
  if (c0 >= n) return;
  ColumnFlat cf[2][4];
  if constexpr (MODE == 2) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const size_t zx = (size_t)z * n + min(c0 + 16 * t + 4 * g + j, n - 1);
        cf[t][j].set(df.d0[zx], df.fa[zx]);
      }
  }
  using RAW = typename std::conditional<MODE >= 2, uint16_t, float>::type;
  struct alignas(4 * sizeof(RAW)) Raw4 {
    RAW v[4];
  };
  const int tiles = (nproj + 15) / 16;
  const int a1 = min(tiles, (int)(blockIdx.y + 1) * na);
  Raw4 raw[2];
  auto fetch = [&](int at) {
    const int pc = min(16 * at + i, nproj - 1);
    const RAW *row = static_cast<const RAW *>(src_) + ((size_t)pc * nz + z) * n;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = c0 + 16 * t + 4 * g;
      if (vec) {
        // (n % 4 == 0: the quadruple is inside or outside as a whole)
        raw[t] = *reinterpret_cast<const Raw4 *>(row + min(c, n - 4));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) raw[t].v[j] = row[min(c + j, n - 1)];
      }
    }
  };
  int at = blockIdx.y * na + (w >> 2);
  if (at < a1) fetch(at);
  for (; at < a1; at += 2) {
    asm volatile("" ::: "memory");  // keeps the LDS reads of B in the loop (72 registers)
    const int p = 16 * at + i;
    const bool live = p < nproj;
    bf8_t a[KS > 0 ? KS : 1][3];
    const __bf16 *Al = A + ((size_t)g * Pa + p) * 8;
    auto ldA = [&](int ks, bf8_t *ak) {
#pragma unroll
      for (int q = 0; q < 3; ++q)
        ak[q] = *reinterpret_cast<const bf8_t *>(Al + q * apart + (size_t)4 * ks * Pa * 8);
    };
    if constexpr (KS > 0) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) ldA(ks, a[ks]);
    }
    float x[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (MODE == 3) {
          const int pc = min(p, nproj - 1);
          const size_t zx = (size_t)z * n + min(c0 + 16 * t + 4 * g + j, n - 1);
          const float v = nproj > 1 ? (float)((double)pc / (double)(nproj - 1)) : 0.f;
          x[t][j] = darkflat((float)raw[t].v[j], df.d0[zx], df.fa[zx], df.fb[zx], v, 1);
        } else if constexpr (MODE == 2) {
          x[t][j] = cf[t][j]((float)raw[t].v[j]);
        } else {
          x[t][j] = raw[t].v[j];
        }
      }
    if (at + 2 < a1) fetch(at + 2);
    floatx4 acc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
    auto step = [&](int ks, const bf8_t *ak) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bf8_t bt[2] = {ldB(ks, 0, q), ldB(ks, 1, q)};
#pragma unroll
        for (int v = 0; q + v < 3; ++v)
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[t] = mma(bt[t], ak[v], acc[t]);
      }
    };
    if constexpr (KS > 0) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) step(ks, a[ks]);
    } else {
      for (int ks = 0; ks < Rp / 32; ++ks) {
        ldA(ks, a[0]);
        step(ks, a[0]);
      }
    }
    if (!live) continue;
    TO *orow = out_ + (MODE >= 2 ? ((size_t)z * nproj + p) * n : ((size_t)p * nz + z) * n);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = c0 + 16 * t + 4 * g;
      struct alignas(4 * sizeof(TO)) Out4 {
        TO v[4];
      } y;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[t][j] + x[t][j];
        if (MODE >= 2 && take_log) v = minus_log(v);
        y.v[j] = (TO)v;
      }
      if (vec) {
        if (c < n) *reinterpret_cast<Out4 *>(orow + c) = y;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c + j < n) orow[c + j] = y.v[j];
      }
    }
  }
}

const WaveletTaps *find_wavelet(const char *name) {
  for (const auto &w : kWavelets)
    if (std::strcmp(w.name, name) == 0) return &w;
  return nullptr;
}

AxisLen axis_len(int64_t N, int L, int level) {
  AxisLen a{};
  a.N[0] = (int)N;
  for (int k = 0; k < level; ++k) a.N[k + 1] = (a.N[k] + L - 1) / 2;
  return a;
}

Taps wavelet_taps(const WaveletTaps *wv) {
  Taps t{};
  for (int j = 0; j < wv->len; ++j) t.a[j] = wv->dec_lo[wv->len - 1 - j];
  return t;
}

// The relations of Taps hold for the wavelet's four filters.
bool orthogonal(const WaveletTaps *wv) {
  const int L = wv->len;
  for (int j = 0; j < L; ++j) {
    const double a = wv->dec_lo[L - 1 - j], b = (j & 1 ? -1.0 : 1.0) * wv->dec_lo[j];
    if (wv->rec_lo[j] != a || wv->rec_hi[j] != b || wv->dec_hi[L - 1 - j] != b) return false;
  }
  return true;
}

// The terms of a scan whose padded angle axis has the band lengths H.
int fw_terms(const AxisLen &H, int level, double sigma, std::vector<FwTerm> &terms) {
  for (int k = 0; k < level; ++k) {
    // kept frequencies q <= my/2 with g_q >= 1e-9 (yhat of :276-279)
    const int my = H.N[k + 1];
    int kept = 0;
    for (int q = 0; q <= my / 2; ++q) {
      // ifftshift((arange(-my, my, 2) + 1)/2)[q]
      const int idx = (q + my / 2) % my;
      const double yh = (double)(-my + 2 * idx + 1) / 2.0;
      const double gv = std::exp(-yh * yh / (2.0 * sigma * sigma));
      if (gv < 1e-9) continue;
      ++kept;
      const bool one = q == 0 || (my % 2 == 0 && q == my / 2);
      const float gk = (float)((one ? 1.0 : 2.0) * gv / my);
      terms.push_back(FwTerm{k, q, 0, gk});
      if (!one) terms.push_back(FwTerm{k, q, 1, gk});
    }
    TOMO_REQUIRE(kept <= kFwMaxNotch,
                 "pre_remove_stripe_fw: sigma=%g keeps %d frequencies at level %d (max %d)", sigma,
                 kept, k + 1, kFwMaxNotch);
  }
  return TOMO_OK;
}

// True where the band-by-band form (stripe_bands.hip) is the faster one: scans of
// few angles and many columns.  Its passes move about S = sum H_k / 2^k rows per
// column, this form's R terms, each through P and B: with fewer rows than terms
// the contraction is an expansion.  Both times, in us, are estimated from the
// counts by a fit to 620 measured calls (8 to 360 angles, 1 to 128 slices of 500 to
// 11000 columns, sigma 1 to 8, 2 to 7 levels, the three filter lengths), which picks
// the slower form, by more than 5 %, in 3 % of them; past 360 angles the low-rank
// form won or tied in all.  Low-rank against bands, sym16, 7 levels: 32 angles, 128
// slices of 1024, sigma 1 328 against 289, sigma 3 714 against 446; 128 angles, 128 x
// 2048, sigma 3 1618 against 1267; 24, 8 x 2048, sigma 3 114 against 192; 1500, 8 x
// 2048, sigma 8 792 against 1758.
bool fw_few_angles(const tomo_pre_plan *P, const WaveletTaps *wv, double sigma, int level) {
  if (P->nproj > 360 || P->n > 16000 || P->nz > 65535) return false;  // (a row fits 64 KB)
  const int L = wv->len;
  const AxisLen H = axis_len(P->nproj + P->nproj / 8, L, level);
  std::vector<FwTerm> terms;
  if (fw_terms(H, level, sigma, terms) != TOMO_OK) return false;  // (setup_fw says why)
  int kept = 0;
  for (int k = 0, c = 0; k < level; ++k, kept = std::max(kept, c))
    c = (int)std::count_if(terms.begin(), terms.end(),
                           [&](const FwTerm &t) { return t.k == k && !t.sin; });
  if (terms.empty()) return false;
  const double R = (double)terms.size(), Rp = (double)(ceil_div((int64_t)R, 32) * 32);
  const double p = (double)P->nproj, cols = 1e-6 * (double)P->nz * (double)P->n;
  double S = 0.0;
  for (int k = 0; k < level; ++k) S += std::ldexp((double)H.N[k], -k);
  const int KM = kept <= 8 ? 8 : kept <= 16 ? 16 : kept <= 32 ? 32 : 64;
  const double low = 21 + cols * (17.1 * Rp + 0.028 * Rp * p + 0.158 * R * L + 1.2 * p);
  const double bands = L == 2    ? 18 + 10 * level + cols * S * (4.0 + 0.223 * KM)
                       : L == 10 ? 34 + 8.2 * level + cols * (46 + S * (4.6 + 0.348 * KM))
                                 : 21.5 * level + cols * (337 + S * (3.75 + 0.541 * KM));
  return bands < low;
}

// Tables and scratch for a wavelet, sigma and level count (kept in the plan).
int setup_fw(tomo_pre_plan *P, const WaveletTaps *wv, double sigma, int level, hipStream_t st) {
  FwPlan &f = P->fw;
  const int L = wv->len;
  const int64_t nz = P->nz, n = P->n, nproj = P->nproj;
  const int npad = (int)(nproj + nproj / 8);
  TOMO_REQUIRE(orthogonal(wv), "pre_remove_stripe_fw: wavelet '%s' is not orthogonal", wv->name);
  const AxisLen H = axis_len(npad, L, level), W = axis_len(n, L, level);
  std::vector<FwTerm> terms;
  const int rc0 = fw_terms(H, level, sigma, terms);
  if (rc0) return rc0;
  f.release();
  f.R = (int)terms.size();
  f.Rp = (int)ceil_div(f.R, 32) * 32;
  f.steps = (int)ceil_div(ceil_div(nproj, 32), kGroups);
  f.Pt = 32 * kGroups * f.steps;
  f.Pa = (int)ceil_div(nproj, 16) * 16;
  f.nPad = (int)ceil_div(n, kApplyCols) * kApplyCols;
  // k_fw_detector: two rows of the longest band with L in front and behind,
  // two more for the pair of outputs past an odd end
  f.len = 0;
  for (int k = 0; k <= level; ++k) f.len = std::max(f.len, W.N[k] + 2 * L + 4);
  f.lds = sizeof(double) * 2 * (size_t)f.len;
  f.glob = f.lds > max_lds_per_block();
  if (f.R > 0) {
    int rc;
    int hlen = H.N[0];
    for (int k = 1; k <= level; ++k) hlen = std::max(hlen, H.N[k]);
    // terms per table launch: at most 64 MB of scratch rows
    const int batch =
        (int)std::max<int64_t>(1, std::min<int64_t>(f.Rp, ((int64_t)64 << 20) / (16 * hlen)));
    DevBuf scr;
    if ((rc = f.terms.alloc(sizeof(FwTerm) * f.R)) ||
        (rc = f.T.alloc(sizeof(uint16_t) * 3 * f.Rp * f.Pt)) ||
        (rc = f.TS.alloc(sizeof(double) * kGroups * f.Rp)) ||
        (rc = f.A.alloc(sizeof(uint16_t) * 3 * f.Rp * f.Pa)) ||
        (rc = f.P.alloc(sizeof(double) * nz * f.Rp * n)) ||
        (rc = f.B.alloc(sizeof(uint16_t) * 3 * nz * f.Rp * f.nPad)) ||
        (f.glob && (rc = f.row.alloc(sizeof(double) * 2 * nz * f.Rp * f.len))) ||
        (rc = scr.alloc(sizeof(double) * 2 * hlen * batch)))
      return rc;
    hipError_t e = hipMemcpyAsync(f.terms.p, terms.data(), sizeof(FwTerm) * f.R,
                                  hipMemcpyHostToDevice, st);
    for (int r0 = 0; r0 < f.Rp && e == hipSuccess; r0 += batch) {
      hipLaunchKernelGGL(k_fw_tables, dim3((unsigned)std::min(batch, f.Rp - r0)), dim3(256), 0, st,
                         f.terms.as<FwTerm>(), f.R, f.Rp, wavelet_taps(wv), L, H, hlen,
                         (npad - (int)nproj) / 2, (int)nproj, f.Pt, f.Pa, f.steps,
                         scr.as<double>(), r0, f.T.as<__bf16>(), f.TS.as<double>(),
                         f.A.as<__bf16>());
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);  // before the scratch goes
    scr.release();
    if (e != hipSuccess) {
      set_error("pre_remove_stripe_fw: building the tables failed: %s", hipGetErrorString(e));
      return TOMO_EHIP;
    }
  }
  f.name = wv->name;
  f.level = level;
  f.sigma = sigma;
  return TOMO_OK;
}

// 16-column tiles of a k_fw_project wave: 2 read T half as often, 1 where 2
// would leave CUs without a workgroup.
template <typename F>
void with_ct(int64_t n, int64_t nz, F &&f) {
  if (n > 1 && nz * ceil_div(n, 32) >= 192)
    f(IC<2>());
  else
    f(IC<1>());
}

// The Fourier-wavelet stripe removal.  src_mode 0: src is the float32
// transmission chunk res[p][z][x]; 2: src is the raw uint16 chunk (means in
// the plan).  dst_mode 1: dst is the float32 chunk res[p][z][x] (in place);
// 2: dst is the sinogram-order output of dtype out_dtype, after minus_log when
// take_log.
int fw_run(tomo_pre_plan *P, const WaveletTaps *wv, double sigma, int level, const void *src,
           int src_mode, DarkFlat df, void *dst, int dst_mode, int out_dtype, int take_log,
           hipStream_t st) {
  TOMO_REQUIRE((src_mode == 0 && dst_mode == 1) || (src_mode == 2 && dst_mode == 2),
               "fw_run: counts to sinograms or the chunk in place");
  int rc;
  if (!(P->fw.name == wv->name && P->fw.level == level && P->fw.sigma == sigma)) {
    // new settings, or those of the band-by-band form
    const FwBands &b = P->fwb;
    const bool bands = b.name == wv->name && b.level == level && b.sigma == sigma;
    if (bands || fw_few_angles(P, wv, sigma, level)) {
      if (!bands) P->fw.release();
      return fw_bands(P, wv, sigma, level, src, src_mode, df, dst, dst_mode, out_dtype, take_log,
                      st);
    }
    P->fwb.release();
    if ((rc = setup_fw(P, wv, sigma, level, st))) return rc;
  }
  const FwPlan &f = P->fw;
  const int L = wv->len, nz = (int)P->nz, nproj = (int)P->nproj, n = (int)P->n;
  hipError_t ea = hipSuccess;
  if (f.R > 0) {
    const AxisLen W = axis_len(n, L, level);
    with_ct(n, nz, [&](auto ctc) {
      constexpr int CT = decltype(ctc)::value;
      const int ncb = (int)ceil_div(n, 16 * CT);
      // (n % CT == 0: a lane's columns are inside or outside as a whole)
      const int vec = n % CT == 0 && ((uintptr_t)src & (CT * (src_mode == 0 ? 4 : 2) - 1)) == 0;
      const dim3 gp((unsigned)(ncb * nz), (unsigned)ceil_div(f.Rp / 16, kRowTiles));
      ProfScope ps_("k_fw_project", st);
      if (src_mode == 0)
        hipLaunchKernelGGL((k_fw_project<0, CT>), gp, dim3(64 * kGroups), 0, st, src, f.T.as<__bf16>(),
                           f.TS.as<double>(), f.P.as<double>(), nproj, nz, n, f.Rp, f.Pt, f.steps,
                           ncb, vec, df);
      else if (!df.flat_linear)
        hipLaunchKernelGGL((k_fw_project<1, CT>), gp, dim3(64 * kGroups), 0, st, src, f.T.as<__bf16>(),
                           f.TS.as<double>(), f.P.as<double>(), nproj, nz, n, f.Rp, f.Pt, f.steps,
                           ncb, vec, df);
      else
        hipLaunchKernelGGL((k_fw_project<2, CT>), gp, dim3(64 * kGroups), 0, st, src, f.T.as<__bf16>(),
                           f.TS.as<double>(), f.P.as<double>(), nproj, nz, n, f.Rp, f.Pt, f.steps,
                           ncb, vec, df);
    });
    TOMO_LAUNCH_CHECK();
    with_len(L, [&](auto lc) {
      constexpr int LC = decltype(lc)::value;
      const Taps tp = wavelet_taps(wv);
      const dim3 gd((unsigned)f.Rp, (unsigned)nz);
      ProfScope ps_("k_fw_detector", st);
      if (f.glob) {
        hipLaunchKernelGGL((k_fw_detector<LC, true>), gd, dim3(256), 0, st, f.P.as<double>(),
                           f.B.as<__bf16>(), f.terms.as<FwTerm>(), f.R, f.Rp, tp, W, f.nPad, f.len,
                           f.row.as<double>());
      } else {
        ea = hipFuncSetAttribute((const void *)k_fw_detector<LC, false>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)f.lds);
        if (ea == hipSuccess)
          hipLaunchKernelGGL((k_fw_detector<LC, false>), gd, dim3(256), f.lds, st,
                             f.P.as<double>(), f.B.as<__bf16>(), f.terms.as<FwTerm>(), f.R, f.Rp,
                             tp, W, f.nPad, f.len, (double *)nullptr);
      }
    });
    TOMO_HIP(ea);
    TOMO_LAUNCH_CHECK();
  }
  // angle tiles per workgroup: 24 (B loaded once for them), fewer for short
  // scans and few columns, so that the launch still fills the CUs
  const int tiles = (int)ceil_div(nproj, 16);
  const int64_t cols = ceil_div(n, kApplyCols) * (int64_t)nz;
  int na = 24;
  while (na > 2 && cols * ceil_div(tiles, na) < 512) na -= 2;
  const dim3 ga((unsigned)ceil_div(n, kApplyCols), (unsigned)ceil_div(tiles, na), (unsigned)nz);
  const size_t osz = out_dtype == TOMO_F32 ? 4 : 2;
  const size_t isz = src_mode == 0 ? 4 : 2;
  const int vec = n % 4 == 0 && ((uintptr_t)src & (4 * isz - 1)) == 0 &&
                  ((uintptr_t)dst & (4 * osz - 1)) == 0;
  auto apply = [&](auto mode, auto *out) {
    constexpr int MODE = decltype(mode)::value;
    using TO = typename std::remove_pointer<decltype(out)>::type;
    auto go = [&](auto ksc) {
      constexpr int KS = decltype(ksc)::value;
      const int lds = 3 * 4 * KS * kApplyCols * (int)sizeof(bf8_t);
      if (lds > 0)
        ea = hipFuncSetAttribute((const void *)k_fw_apply<MODE, TO, KS>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (ea != hipSuccess) return;
      ProfScope ps_("k_fw_apply", st);
      hipLaunchKernelGGL((k_fw_apply<MODE, TO, KS>), ga, dim3(512), lds, st, src, out,
                         f.A.as<__bf16>(), f.B.as<__bf16>(), nproj, nz, n, f.Rp, f.Pa, f.nPad, na,
                         vec, take_log, df);
    };
    if (f.Rp == 96)
      go(IC<3>());
    else if (f.Rp == 64)
      go(IC<2>());
    else if (f.Rp == 32)
      go(IC<1>());
    else
      go(IC<0>());
  };
  auto apply_counts = [&](auto *out) {
    if (df.flat_linear)
      apply(IC<3>(), out);
    else
      apply(IC<2>(), out);
  };
  if (dst_mode == 1)
    apply(IC<1>(), (float *)dst);
  else if (out_dtype == TOMO_F16)
    apply_counts((_Float16 *)dst);
  else if (out_dtype == TOMO_BF16)
    apply_counts((__bf16 *)dst);
  else
    apply_counts((float *)dst);
  TOMO_HIP(ea);
  TOMO_LAUNCH_CHECK();
  return TOMO_OK;
}

const WaveletTaps *check_wavelet(const char *fn, const char *wname, double sigma, int level) {
  if (!(sigma > 0 && std::isfinite(sigma))) {
    set_error("%s: sigma must be > 0", fn);
    return nullptr;
  }
  if (level < 1 || level > kMaxLevels) {
    set_error("%s: level=%d out of range", fn, level);
    return nullptr;
  }
  const WaveletTaps *wv = find_wavelet(wname);
  if (!wv) {
    set_error("%s: unknown wavelet '%s'", fn, wname);
    return nullptr;
  }
  if (wv->len != 2 && wv->len != 10 && wv->len != 32) {
    set_error("%s: wavelet '%s' has %d taps (2, 10 or 32 supported)", fn, wname, wv->len);
    return nullptr;
  }
  return wv;
}

}  // namespace
extern "C" int pre_remove_stripe_fw(tomo_pre_plan *P, float *res, double sigma, const char *wname,
                                    int level, void *stream) {
  clear_error();
  TOMO_REQUIRE(P != nullptr && res != nullptr && wname != nullptr,
               "pre_remove_stripe_fw: NULL argument");
  const WaveletTaps *wv = check_wavelet("pre_remove_stripe_fw", wname, sigma, level);
  if (!wv) return TOMO_EINVAL;
  return fw_run(P, wv, sigma, level, res, 0, DarkFlat{nullptr, nullptr, nullptr, 0}, res, 1,
                TOMO_F32, 0, (hipStream_t)stream);
}

extern "C" int pre_process_fw(tomo_pre_plan *P, const uint16_t *data, const uint16_t *dark,
                              const uint16_t *flat, void *out, int out_dtype, double bright_ratio,
                              int flat_linear, int minus_log, double sigma, const char *wname,
                              int level, void *stream) {
  clear_error();
  TOMO_REQUIRE(P != nullptr && data && dark && flat && out && wname,
               "pre_process_fw: NULL argument");
  TOMO_REQUIRE(out_dtype == TOMO_F32 || out_dtype == TOMO_F16 || out_dtype == TOMO_BF16,
               "pre_process_fw: unknown out_dtype %d", out_dtype);
  const WaveletTaps *wv = check_wavelet("pre_process_fw", wname, sigma, level);
  if (!wv) return TOMO_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  int rc = pre_launch_means(P, dark, flat, bright_ratio, flat_linear, st);
  if (rc) return rc;
  const DarkFlat df{P->dark0.as<float>(), P->flatA.as<float>(), P->flatB.as<float>(),
                    flat_linear};
  return fw_run(P, wv, sigma, level, data, 2, df, out, 2, out_dtype, minus_log, st);
}
