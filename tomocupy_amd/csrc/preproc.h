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

// Tables and scratch of the Fourier-wavelet stripe removal (stripe.hip),
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
  tomo::DevBuf outl;  // medians of pre_remove_outliers, allocated on first use
  tomo::DevBuf ti;    // column means and corrections of pre_remove_stripe_ti (first use)
  tomo::VoBufs vo;    // scratch of pre_remove_all_stripe (first use)
};
