// Internal: the preprocessing plan shared by preproc.hip and stripe.hip.
#pragma once

#include <string>
#include <vector>

#include "common.h"

struct tomo_pre_plan;

namespace tomo {

constexpr int kMaxDezinger = 9;  // largest median window of pre_remove_outliers
constexpr int kVoMaxProj = 8192;  // vo-all: angles of a column sorted in LDS
constexpr int kVoMaxWin = 255;    // vo-all: largest detector median window
constexpr int kVoMaxN = 16384;    // vo-all: detector width of a slice's stripe test

// Scratch of pre_remove_all_stripe (allocated on the plan's first call)
struct VoBufs {
  DevBuf T, S, M;  // (nz, n, nproj) float: columns, sorted columns, smoothed
  DevBuf I;        // (nz, n, nproj) uint16: angle of each sorted rank
  DevBuf rowf;     // 5 x (nz, n) float: roughness, its median, two means, ratio
  DevBuf mask;     // (nz, n) uint8: located columns
  void release() {
    T.release();
    S.release();
    M.release();
    I.release();
    rowf.release();
    mask.release();
  }
};

// Tables and scratch of the Fourier-wavelet stripe removal's low-rank form (stripe.hip),
// (re)built when the settings change.
struct FwPlan {
  std::string name;  // wavelet; empty: nothing built
  int level = 0;
  double sigma = 0.0;
  int R = 0, Rp = 0;    // terms, padded to the matrix products' 32
  int steps = 0;        // 32-angle steps of an angle group
  int Pt = 0, Pa = 0;   // padded angles of T and of A
  int nPad = 0;         // padded columns of B
  int len = 0;          // longest band along the detector
  size_t lds = 0;       // k_fw_detector: its two rows; glob: they do not fit
  bool glob = false;
  DevBuf terms, T, TS, A;  // see k_fw_tables
  DevBuf P, B, row;             // see k_fw_project, k_fw_detector
  void release() {
    name.clear();
    for (DevBuf *b : {&terms, &T, &TS, &A, &P, &B, &row}) b->release();
  }
};

// One level of the band-by-band form (stripe_bands.hip): analysis input H x W,
// bands Ho x Wo; the notch keeps nk angular frequencies of the stripe band.
struct FwLevel {
  int H = 0, W = 0, Ho = 0, Wo = 0;
  int nk = 0;
  int KM = 8;   // notch frequencies a kernel instance holds (8, 16, 32 or 64 >= nk)
  int R = 4;    // output rows per wave of the column analysis
  int nrb = 0;  // row blocks of the column analysis
  DevBuf tw;    // (nk, Ho) float2: cos/sin(2 pi k t / Ho)
  DevBuf gk;    // (nk,) float: c_k g_k / Ho
  DevBuf ll;    // (nz, Ho, Wo): low band = input of the next level
  DevBuf part;  // (nz, nrb, KM, Wo) float2: partial notch DFTs of the stripe band
  DevBuf X;     // (nz, KM, Wo) float2: notch coefficients, kept until the synthesis
};

struct FwBands {
  std::string name;  // wavelet; empty: nothing built
  int level = 0;
  double sigma = 0.0;
  std::vector<FwLevel> lv;
  DevBuf rowlo, rowhi, synlo, synhi, syn[2];
  void release() {
    name.clear();
    for (auto &l : lv)
      for (DevBuf *b : {&l.tw, &l.gk, &l.ll, &l.part, &l.X}) b->release();
    lv.clear();
    for (DevBuf *b : {&rowlo, &rowhi, &synlo, &synhi, &syn[0], &syn[1]}) b->release();
  }
};

// Dark/flat means (k_pre_means output).
struct DarkFlat {
  const float *d0, *fa, *fb;
  int flat_linear;
};

constexpr int kFwMaxNotch = 64;  // kept notch frequencies per level: sigma up to about 9.8

struct WaveletTaps;
int fw_bands(tomo_pre_plan *P, const WaveletTaps *wv, double sigma, int level, const void *src,
             int src_mode, DarkFlat df, void *dst, int dst_mode, int out_dtype, int take_log,
             hipStream_t st);

// flat0 of a mean flat fa and a mean dark d0: fa * float32(1 + 1e-5) - d0
// (proc_functions.py:71-72)
__device__ __forceinline__ float flat0(float fa, float d0) {
  const float eps = 1.0f + 1e-5f;
  return fa * eps - d0;
}

// dark/flat correction of one count (proc_functions.py:67-74): flat0 of the
// flat mean (or of the linear interpolation v of the two halves' means,
// :62-66); result (x - dark0) / flat0
__device__ __forceinline__ float darkflat(float x, float d0, float fa, float fb, float v,
                                          int flat_linear) {
  const float f0 = flat0(flat_linear ? (1.0f - v) * fa + v * fb : fa, d0);
  return (x - d0) / f0;
}

__device__ __forceinline__ float minus_log(float x) {
  // x <= 0 -> 1; -log; NaN -> 6; +-inf -> 0 (proc_functions.py:76-83)
  if (x <= 0.f) x = 1.f;
  float r = -logf(x);
  if (isnan(r)) r = 6.0f;
  if (isinf(r)) r = 0.0f;
  return r;
}

// dark0 = mean(dark), flat means, in the plan's scratch (k_pre_means)
int pre_launch_means(tomo_pre_plan *P, const uint16_t *dark, const uint16_t *flat,
                     double bright_ratio, int flat_linear, hipStream_t st);

}  // namespace tomo

struct tomo_pre_plan {
  int64_t nproj = 0, nz = 0, n = 0, ndark = 0, nflat = 0;
  tomo::DevBuf dark0, flatA, flatB;
  tomo::FwPlan fw;
  tomo::FwBands fwb;
  tomo::DevBuf outl;  // medians of pre_remove_outliers, allocated on first use
  tomo::DevBuf ti;    // column means and corrections of pre_remove_stripe_ti (first use)
  tomo::VoBufs vo;    // scratch of pre_remove_all_stripe (first use)
};
