// Single-step phase retrieval for gfx950 (tomocupy processing/retrieve_phase.py:
// paganin_filter :59-104, farago_filter :106-141, _retrieve_phase :143-161,
// applied by ProcFunctions.proc_proj, proc_functions.py:169-181) on float32
// projections (nproj, dy, dz) in place:
//   prj  = projection edge-replicated to Ny x Nx (pads py rows and pz columns
//          on each side, Ny = dy + 2 py and Nx = dz + 2 pz powers of two)
//   proj = Re ifft2(fft2(prj) * H / max H)[py : py + dy, pz : pz + dz]
// with H = fftshift of the method's factor on the reciprocal grid:
//   paganin   1 / (lambda dist w2 / (4 pi) + alpha),          w2 = u^2 + v^2
//   Gpaganin  1 / (1 - 2 aph / W^2 (kf - 2)),  aph = db dist lambda / (4 pi),
//             kf = cos(2 pi ps u) + cos(2 pi ps v)
//   farago    1 / (cos(pi lambda dist w2) + db sin(pi lambda dist w2))
// u, v the reference's reciprocal coordinates (k - (N-1)/2) / ((N-1) ps),
// half a sample off zero for even N.
//
// H is real but not even (half a sample off zero), and the projection is real,
// so Re ifft2(F H) = ifft2(F He) with the even part He(k) = (H(k) + H(-k)) / 2:
// F He is Hermitian, and half of its columns hold it all.
//
// Three kernels per batch of projections, through a complex work buffer of
// the left half of the dy real rows' spectra (the py padded rows above and
// below a projection are copies of its first and last rows, so their row
// spectra are those rows' spectra): rows (two real rows packed into one complex
// FFT, split into their two half spectra), columns (the padded column rebuilt
// from the edge spectra, forward FFT, filter He / max H / (Ny Nx), inverse FFT,
// the dy rows the crop keeps written back), and inverse rows (two half spectra
// extended and packed into one inverse FFT, whose real and imaginary parts are
// the two real rows).  The columns 0 and Nx / 2 of a real row's spectrum are
// real, so column 0 of the buffer holds both, as its real and imaginary parts.
// The buffer is blocked by 2^lgB columns, F[projection][block][row][column]: two
// rows of a block are adjacent.  The
// FFTs are the LDS Stockham transforms of fft_lds.h; the filter is evaluated
// in float32 (the reference's precision) from 1-D tables built in FP64.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

#include "common.h"
#include "fft_lds.h"

using namespace tomo;

struct tomo_ph_plan {
  int64_t dy = 0, dz = 0, batch = 0;
  int method = 0;
  int py = 0, pz = 0, Ny = 0, Nx = 0;
  int lgC = 0;     // log2 of the columns per workgroup of the column pass
  int lgB = 0;     // log2 of the columns per block of F
  size_t Fb = 0;   // elements of F per projection
  float cHi = 0.f, cLo = 0.f;  // 1 / (2 max H Ny Nx) as an unrounded sum
  float A = 0.f, B = 0.f, alpha = 0.f, db = 0.f, hmax = 1.f;
  int rowThreads = 0, colThreads = 0;
  size_t rowLds = 0, colLds = 0;
  FftPlan fy, fx;
  DevBuf ty, tx;  // fftshifted 1-D terms of the filter (rows, columns)
  DevBuf h0;      // float4 per padded row: the filter of column 0 (k_ph_col0)
  int div = 0;    // ph_even's div
  DevBuf F;       // (batch, Nx/2 >> lgB, dy, 2^lgB) float2: half spectra of the real rows
};

namespace {

constexpr double kPi = 3.14159265359;               // retrieve_phase.py:48
constexpr double kPlanck = 6.58211928e-19;          // [keV s], :49
constexpr double kLight = 299792458e+2;             // [cm/s], :47

// Padded lengths are powers of two: f(integral_constant<int, N>) for the
// compiled lengths 512 .. 8192, f(integral_constant<int, 0>) (run-time plan)
// below.
template <typename F>
void with_ph_size(int N, F &&f) {
  switch (N) {
    case 512: f(std::integral_constant<int, 512>()); break;
    case 1024: f(std::integral_constant<int, 1024>()); break;
    case 2048: f(std::integral_constant<int, 2048>()); break;
    case 4096: f(std::integral_constant<int, 4096>()); break;
    case 8192: f(std::integral_constant<int, 8192>()); break;
    default: f(std::integral_constant<int, 0>()); break;
  }
}

// log2 of the columns of a column-pass workgroup: compiled lengths, as many as
// 512 threads hold in registers, so that two workgroups share a CU and one's
// loads run under the other's butterflies; run-time lengths, 8 (ph_create)
constexpr int ph_lg(int N) { return N > 0 ? split_lg(N) - (N > 1024) : 3; }
// log2 of the columns of a block of the work buffer: 8 or a workgroup's, so
// that the row passes store and load 128-byte segments (8 columns of 2 rows)
constexpr int ph_lgb(int N) { return ph_lg(N) > 3 ? ph_lg(N) : 3; }

// the reciprocal of the method's factor at one grid point, from the sum of the
// two 1-D terms
__device__ __forceinline__ float ph_denom(int method, float s, float A, float B, float alpha,
                                          float db) {
  if (method == 0) return A * s + alpha;             // paganin
  if (method == 1) return 1.f - B * (s - 2.f);       // Gpaganin
  float sn, cs;                                      // farago
  sincosf(A * s, &sn, &cs);
  return cs + db * sn;
}

// row maxima of the factor over the grid (the normalisation max H)
__global__ __launch_bounds__(256) void k_ph_fmax(const float *__restrict__ ty,
                                                 const float *__restrict__ tx, int Nx,
                                                 int method, float A, float B, float alpha,
                                                 float db, float *__restrict__ rowmax) {
  __shared__ float red[256];
  const int ky = blockIdx.x;
  float m = -INFINITY;
  for (int kx = threadIdx.x; kx < Nx; kx += 256)
    m = fmaxf(m, 1.f / ph_denom(method, ty[ky] + tx[kx], A, B, alpha, db));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) rowmax[ky] = red[0];
}

// 1 / d for a normal d with a normal reciprocal: the hardware's reciprocal (1 ulp)
// and one Newton step, whose single rounding leaves it correctly rounded but next
// to a tie.  A division takes three times the instructions.
__device__ __forceinline__ float ph_rcp(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(r, fmaf(-d, r, 1.f), r);
}

// The even part of the factor, times 2 (c_hi + c_lo).  div: the factor's maximum
// is so small that its reciprocals may be subnormal.
__device__ __forceinline__ float ph_even(int method, float s0, float s1, float A, float B,
                                         float alpha, float db, float c_hi, float c_lo, int div) {
  const float d0 = ph_denom(method, s0, A, B, alpha, db);
  const float d1 = ph_denom(method, s1, A, B, alpha, db);
  const float r0 = div ? 1.f / d0 : ph_rcp(d0), r1 = div ? 1.f / d1 : ph_rcp(d1);
  const float h = r0 + r1, e = r1 - (h - r0);  // (the sum's rounding; r0 and r1 are alike)
  return fmaf(h, c_hi, fmaf(e, c_hi, h * c_lo));
}

// Column 0 of the work buffer is P = A + i B with A column 0 and B column
// Nx / 2 of a real image's spectrum: times their even, real factors hA and hB
// that is P[k] (hA + hB) / 2 + conj(P[-k]) (hA - hB) / 2.  It holds the image's
// mean, of which a rounding of the factor would scale every pixel (rms of the
// mean's error over 16 images of 1024 x 1024: 8.4e-8 with two float32 factors,
// 3.8e-8 so, of 1.49e-7 and 1.29e-7 in all), so the two go out as high and low
// parts, and the float32 factor over its maximum is exactly 1 where it is largest.
__global__ __launch_bounds__(256) void k_ph_col0(const float *__restrict__ ty,
                                                 const float *__restrict__ tx, int Ny, int Nx,
                                                 int method, float A, float B, float alpha,
                                                 float db, double c, float4 *__restrict__ h0) {
  const int ky = blockIdx.x * 256 + threadIdx.x;
  if (ky >= Ny) return;
  const float t0 = ty[ky], t1 = ty[ky == 0 ? 0 : Ny - ky];
  auto even = [&](float x) {
    return c * ((double)(1.f / ph_denom(method, t0 + x, A, B, alpha, db)) +
                (double)(1.f / ph_denom(method, t1 + x, A, B, alpha, db)));
  };
  const double a = even(tx[0]), b = even(tx[Nx / 2]);
  const double s = 0.5 * (a + b), d = 0.5 * (a - b);
  const float sh = (float)s, dh = (float)d;
  h0[ky] = make_float4(sh, dh, (float)(s - sh), (float)(d - dh));
}

// P[k] and P[-k] times the factors of k_ph_col0.
__device__ __forceinline__ float2 ph_mix0(float2 p, float2 m, float4 h) {
  return make_float2(fmaf(p.x, h.x, fmaf(m.x, h.y, fmaf(p.x, h.z, m.x * h.w))),
                     fmaf(p.y, h.x, fmaf(-m.y, h.y, fmaf(p.y, h.z, -m.y * h.w))));
}

// Forward FFTs of the column-padded real rows 2 pr and 2 pr + 1 of
// projection blockIdx.y: z = row0 + i row1, Z = fft(z);
// X0 = (Z[k] + conj Z[-k]) / 2, X1 = (Z[k] - conj Z[-k]) / (2i), k < Nx / 2.
template <int NS>
__global__ __launch_bounds__(512) void k_ph_rows_fwd(const float *__restrict__ data,
                                                      float2 *__restrict__ F, FftDesc fd, int dy,
                                                      int dz, int pz, int lgB, size_t Fb) {
  extern __shared__ float2 sm[];
  const int pr = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int Nx = NS > 0 ? NS : fd.N;
  const int iy0 = 2 * pr;
  const float *img = data + (size_t)b * dy * dz;
  const float *r0 = img + (size_t)iy0 * dz;
  const float *r1 = r0 + dz;
  auto ld = [&](int ix, int) {
    const int sx = min(max(ix - pz, 0), dz - 1);
    return make_float2(r0[sx], r1[sx]);
  };
  if constexpr (NS > 0) {
    fft_c_from_global<NS, -1, kFftEPT, 0>(sm, fd.tw, tid, nt, ld);
  } else {
    for (int ix = tid; ix < Nx; ix += nt) sm[ix] = ld(ix, 0);
    __syncthreads();
    lds_fft<-1>(sm, fd, 0, tid, nt);
  }
  // (a block's columns of the first row, then of the second, then the next
  // block's: 16 << lgB contiguous bytes)
  float2 *f = F + (size_t)b * Fb + ((size_t)iy0 << lgB);
  for (int e = tid; e < max(Nx, 2 << lgB); e += nt) {
    const int c = e & ((1 << lgB) - 1), blk = e >> (lgB + 1), row = (e >> lgB) & 1;
    const int k = (blk << lgB) + c;
    if (2 * k >= Nx) continue;  // (Nx / 2 may be less than a block)
    float2 x;
    if (k == 0) {
      const float2 z0 = sm[0], zn = sm[lidx<NS>(Nx / 2)];
      x = row ? make_float2(z0.y, zn.y) : make_float2(z0.x, zn.x);
    } else {
      const float2 zk = sm[lidx<NS>(k)], zm = cconj(sm[lidx<NS>(Nx - k)]);
      x = row ? make_float2(0.5f * (zk.y - zm.y), -0.5f * (zk.x - zm.x))
              : make_float2(0.5f * (zk.x + zm.x), 0.5f * (zk.y + zm.y));
    }
    f[(((size_t)blk * dy + row) << lgB) + c] = x;
  }
}

// Column pass over 2^lgC columns of a projection: the padded column (padded row ky holds real row clamp(ky - py, 0, dy - 1)),
// forward FFT, times He / max H / (Ny Nx), inverse FFT; rows py .. py+dy-1
// written back in place.  Compiled lengths keep a column's values in registers
// from the load to the store; what bounds them is vector arithmetic (two
// transforms and the factor).  Measured for 4 projections of 2048 x 2048
// (padded 4096 x 4096): 164 us with two workgroups of 4 columns per CU, 195
// with one of 8 columns (and divisions for the factor); 443 for all 4096
// columns through LDS passes.  The row passes, half a spectrum each, 52 and 46
// us, were 90 and 90.
template <int NS>
__global__ __launch_bounds__(1024) void k_ph_cols(float2 *__restrict__ F, FftDesc fd, int lgC,
                                                   int Nx, int dy, int py,
                                                   const float *__restrict__ ty,
                                                   const float *__restrict__ tx,
                                                   const float4 *__restrict__ h0, int method,
                                                   float A, float B, float alpha, float db,
                                                   float c_hi, float c_lo, int div, size_t Fb) {
  extern __shared__ float2 sm[];
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lgB = ph_lgb(NS);
  if (NS > 0) lgC = ph_lg(NS);
  const int Ny = NS > 0 ? NS : fd.N, C = 1 << lgC;
  // workgroups of one block of the work buffer go to the same XCD
  const int L = xcd_remap(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
  const int kx0 = (L % gridDim.x) << lgC, b = L / gridDim.x;
  float2 *fb = F + (size_t)b * Fb + (((size_t)(kx0 >> lgB) * dy) << lgB) + (kx0 & ((1 << lgB) - 1));
  auto row = [&](int ky) { return min(max(ky - py, 0), dy - 1); };
  if constexpr (NS > 0) {
    // Values stay in registers from the load to the store.
    constexpr int LG = ph_lg(NS), E = kFftSplitEPT, T = split_threads(NS, LG), U = NS / E;
    float *buf = reinterpret_cast<float *>(sm);
    const int t = tid & (C - 1), kx = kx0 + t;
    int j = tid >> LG;
    const bool live = 2 * kx < Nx;  // (Nx / 2 may be less than a block)
    // (32-bit offsets: a thread's 32 addresses would not fit its registers)
    auto at = [&](int y, int c) {
      return reinterpret_cast<float2 *>(reinterpret_cast<char *>(fb) +
                                        ((unsigned)((y << lgB) + c) * 8u));
    };
    float2 a[E];
#pragma unroll
    for (int s = 0; s < E; ++s) a[s] = *at(row(j + s * U), live ? t : 0);
    asm volatile("" : "+v"(j));  // recompute what hangs on j: held, it would spill
    fft_split_regs<NS, -1, LG>(a, buf, fd.tw, tid);
    // the factors in a rolled loop (one copy of the method's code), through
    // the thread's own LDS words
    __syncthreads();
    const float x0 = tx[live ? kx : 0], x1 = tx[live && kx > 0 ? Nx - kx : 0];
#pragma unroll 2
    for (int s = 0; s < E; ++s) {
      const int ky = j + s * U;
      const float h = ph_even(method, ty[ky] + x0, ty[ky == 0 ? 0 : NS - ky] + x1, A, B, alpha,
                              db, c_hi, c_lo, div);
      buf[s * T + tid] = kx == 0 ? 1.f : h;
    }
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const float h = buf[s * T + tid];
      a[s] = make_float2(a[s].x * h, a[s].y * h);
    }
    if (kx0 == 0) {  // column 0 is two
      __syncthreads();
      if (t == 0) {
#pragma unroll
        for (int s = 0; s < E; ++s) sm[j + s * U] = a[s];
      }
      __syncthreads();
      if (t == 0) {
#pragma unroll
        for (int s = 0; s < E; ++s) {
          const int ky = j + s * U;
          a[s] = ph_mix0(a[s], sm[ky == 0 ? 0 : NS - ky], h0[ky]);
          asm volatile("" ::: "memory");  // the loads of all s at once would spill
        }
      }
    }
    fft_split_regs<NS, 1, LG>(a, buf, fd.tw, tid);
    asm volatile("" : "+v"(j));
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const int y = j + s * U - py;
      if (live && y >= 0 && y < dy) *at(y, t) = a[s];
    }
  } else {
    for (int e = tid; e < (Ny << lgC); e += nt) {
      const int ky = e >> lgC, c = e & (C - 1);
      sm[e] = 2 * (kx0 + c) < Nx ? fb[((size_t)row(ky) << lgB) + c] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    lds_fft<-1>(sm, fd, lgC, tid, nt);
    for (int e = tid; e < (Ny << lgC); e += nt) {
      const int ky = e >> lgC, c = e & (C - 1), kx = kx0 + c, km = ky == 0 ? 0 : Ny - ky;
      if (2 * kx >= Nx) continue;
      const float2 v = sm[e];
      if (kx > 0) {
        const float h = ph_even(method, ty[ky] + tx[kx], ty[km] + tx[Nx - kx], A, B, alpha, db,
                                c_hi, c_lo, div);
        sm[e] = make_float2(v.x * h, v.y * h);
      } else if (2 * ky <= Ny) {  // this thread does rows ky and -ky
        const float2 m = sm[km << lgC];
        sm[e] = ph_mix0(v, m, h0[ky]);
        if (km != ky) sm[km << lgC] = ph_mix0(m, v, h0[km]);
      }
    }
    __syncthreads();
    lds_fft<1>(sm, fd, lgC, tid, nt);
    for (int e = tid; e < (dy << lgC); e += nt) {
      const int y = e >> lgC, c = e & (C - 1);
      if (2 * (kx0 + c) < Nx) fb[((size_t)y << lgB) + c] = sm[((y + py) << lgC) + c];
    }
  }
}

// Inverse row FFTs for output rows 2 pr and 2 pr + 1 from their half spectra
// G0, G1: z[k] = G0[k] + i G1[k], z[-k] = conj G0[k] + i conj G1[k]; cropped
// columns written back to the projection.
template <int NS>
__global__ __launch_bounds__(512) void k_ph_rows_inv(float *__restrict__ data,
                                                      const float2 *__restrict__ F, FftDesc fd,
                                                      int dy, int dz, int pz, int lgB, size_t Fb) {
  extern __shared__ float2 sm[];
  const int pr = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int Nx = NS > 0 ? NS : fd.N;
  const int oy0 = 2 * pr, oy1 = oy0 + 1;  // dy is even: both rows exist
  const float2 *g = F + (size_t)b * Fb + ((size_t)oy0 << lgB);
  for (int k = tid; 2 * k < Nx; k += nt) {
    const float2 *gk = g + (((size_t)(k >> lgB) * dy) << lgB) + (k & ((1 << lgB) - 1));
    const float2 x0 = gk[0], x1 = gk[1 << lgB];
    sm[lidx<NS>(k)] = k == 0 ? make_float2(x0.x, x1.x) : make_float2(x0.x - x1.y, x0.y + x1.x);
    sm[lidx<NS>(k == 0 ? Nx / 2 : Nx - k)] =
        k == 0 ? make_float2(x0.y, x1.y) : make_float2(x0.x + x1.y, x1.x - x0.y);
  }
  __syncthreads();
  float *img = data + (size_t)b * dy * dz;
  auto st = [&](int o, int, float2 v) {
    const int x = o - pz;
    if (x < 0 || x >= dz) return;
    img[(size_t)oy0 * dz + x] = v.x;
    img[(size_t)oy1 * dz + x] = v.y;
  };
  if constexpr (NS > 0) {
    using SP = StaticPlan<NS>;
    constexpr int RL = SP::radix(SP::passes - 1);
    lds_fft_c<NS, 1, kFftEPT, 0, 0, 1, SP::passes - 1>(sm, fd.tw, tid, nt);
    fft_pass_c_last<RL, NS / RL, NS, 1, kFftEPT, 0>(sm, fd.tw, tid, nt, st);
  } else {
    lds_fft<1>(sm, fd, 0, tid, nt);
    for (int o = tid; o < Nx; o += nt) st(o, 0, sm[o]);
  }
}

// the reference's _calc_pad_width (retrieve_phase.py:214-216)
int pad_width(int64_t dim, double pad_pix) {
  const double p2 = std::pow(2.0, std::ceil(std::log2((double)dim + pad_pix)));
  return (int)((p2 - (double)dim) * 0.5);
}

bool pow2(int v) { return v >= 2 && (v & (v - 1)) == 0; }

}  // namespace

extern "C" void ph_destroy(tomo_ph_plan *P) {
  if (!P) return;
  P->fy.release();
  P->fx.release();
  P->ty.release();
  P->tx.release();
  P->h0.release();
  P->F.release();
  delete P;
}

extern "C" int ph_create(tomo_ph_plan **plan, int64_t dy, int64_t dz, int64_t batch, int method,
                         double pixel_size, double dist, double energy, double alpha, double db,
                         double W) {
  clear_error();
  TOMO_REQUIRE(plan != nullptr, "ph_create: plan pointer is NULL");
  *plan = nullptr;
  TOMO_REQUIRE(dy >= 2 && dz >= 2 && dy % 2 == 0 && dz % 2 == 0,
               "ph_create: projection size %lld x %lld must be even (powers of two after "
               "padding)", (long long)dy, (long long)dz);
  TOMO_REQUIRE(batch >= 1 && batch <= 65535, "ph_create: batch out of range");
  TOMO_REQUIRE(method >= 0 && method <= 2, "ph_create: method %d (0 paganin, 1 Gpaganin, 2 farago)",
               method);
  TOMO_REQUIRE(pixel_size > 0 && dist > 0 && energy > 0 && std::isfinite(pixel_size) &&
                   std::isfinite(dist) && std::isfinite(energy),
               "ph_create: pixel size, distance and energy must be > 0");
  TOMO_REQUIRE(std::isfinite(alpha) && std::isfinite(db) && std::isfinite(W) &&
                   (method != 1 || W > 0),
               "ph_create: invalid alpha, delta/beta or W");
  auto *P = new (std::nothrow) tomo_ph_plan();
  if (!P) {
    set_error("ph_create: host allocation failed");
    return TOMO_ENOMEM;
  }
  P->dy = dy;
  P->dz = dz;
  P->batch = batch;
  P->method = method;
  const double lambda = 2 * kPi * kPlanck * kLight / energy;  // _wavelength, :52-53
  const double pad_pix = std::ceil(kPi * lambda * dist / (pixel_size * pixel_size));
  P->py = pad_width(dy, pad_pix);
  P->pz = pad_width(dz, pad_pix);
  P->Ny = (int)(dy + 2 * P->py);
  P->Nx = (int)(dz + 2 * P->pz);
  if (!pow2(P->Ny) || !pow2(P->Nx) || P->Ny > 8192 || P->Nx > 8192) {
    set_error("ph_create: padded size %d x %d not a power of two <= 8192", P->Ny, P->Nx);
    ph_destroy(P);
    return TOMO_EINVAL;
  }
  if (method == 0) {
    P->A = (float)(lambda * dist / (4 * kPi));
  } else if (method == 1) {
    const double aph = db * (dist * lambda) / (4 * kPi);
    P->B = (float)(2 * aph / (W * W));
  } else {
    P->A = (float)(kPi * lambda * dist);
  }
  P->alpha = (float)alpha;
  P->db = (float)db;
  // fftshifted 1-D terms: u_k = (2k - (N-1)) * 0.5 / ((N-1) ps) at index
  // (k - N/2) mod N (_reciprocal_coord :296-304, fftshift :89-95)
  auto terms = [&](int N) {
    std::vector<float> t(N);
    for (int k = 0; k < N; ++k) {
      const int j = ((k - N / 2) % N + N) % N;
      const double u = (2.0 * j - (N - 1)) * 0.5 / ((N - 1) * pixel_size);
      t[k] = (float)(method == 1 ? std::cos(u * 2 * kPi * pixel_size) : u * u);
    }
    return t;
  };
  const std::vector<float> hy = terms(P->Ny), hx = terms(P->Nx);
  int rc = P->fy.init(P->Ny);
  if (!rc) rc = P->fx.init(P->Nx);
  if (!rc) rc = P->ty.alloc(sizeof(float) * P->Ny);
  if (!rc) rc = P->tx.alloc(sizeof(float) * P->Nx);
  // columns per block of the work buffer; one block at least
  with_ph_size(P->Ny, [&](auto ns) {
    P->lgC = ph_lg(decltype(ns)::value);
    P->lgB = ph_lgb(decltype(ns)::value);
  });
  // Run-time column lengths (below 512): launches of few short columns, which last
  // as long as a workgroup's chain, so narrow images take 4 columns a workgroup and
  // all of them many threads.  us for a call, 8 columns with as few threads as hold
  // the butterflies | 8, 256 threads | 4, 512: 4 images padded to 128 x 128 21.3
  // 18.7 16.7, 8 to 256 x 256 69.1 54.6 42.4, 8 to 256 x 512 52.2 42.0 33.3, 16 to
  // 256 x 4096 158 146 208, 32 to 32 x 2048 150 137 183.
  const bool shortCols = P->Ny < 512, narrow = P->Nx <= 512;
  if (shortCols && narrow) P->lgC = 2;
  P->Fb = (size_t)std::max(P->Nx / 2, 1 << P->lgB) * dy;
  if (!rc) rc = P->h0.alloc(sizeof(float4) * P->Ny);
  if (!rc) rc = P->F.alloc(sizeof(float2) * (size_t)batch * P->Fb);
  if (rc) {
    ph_destroy(P);
    return rc;
  }
  TOMO_HIP(hipMemcpy(P->ty.p, hy.data(), sizeof(float) * P->Ny, hipMemcpyHostToDevice));
  TOMO_HIP(hipMemcpy(P->tx.p, hx.data(), sizeof(float) * P->Nx, hipMemcpyHostToDevice));
  // max H over the grid, with the kernels' float32 factor
  {
    DevBuf rowmax;
    rc = rowmax.alloc(sizeof(float) * P->Ny);
    if (rc) {
      ph_destroy(P);
      return rc;
    }
    hipLaunchKernelGGL(k_ph_fmax, dim3((unsigned)P->Ny), dim3(256), 0, 0, P->ty.as<float>(),
                       P->tx.as<float>(), P->Nx, method, P->A, P->B, P->alpha, P->db,
                       rowmax.as<float>());
    std::vector<float> rm(P->Ny);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
      e = hipMemcpy(rm.data(), rowmax.p, sizeof(float) * P->Ny, hipMemcpyDeviceToHost);
    if (e != hipSuccess) {
      set_error("ph_create: %s", hipGetErrorString(e));
      ph_destroy(P);
      return TOMO_EHIP;
    }
    P->hmax = *std::max_element(rm.begin(), rm.end());
    if (!(std::isfinite(P->hmax) && P->hmax != 0.f)) {
      set_error("ph_create: the filter maximum is %g (check the parameters)", (double)P->hmax);
      ph_destroy(P);
      return TOMO_EINVAL;
    }
  }
  const double cs = 0.5 / ((double)P->hmax * P->Ny * P->Nx);
  P->cHi = (float)cs;
  P->cLo = (float)(cs - (double)P->cHi);
  P->div = std::fabs(P->hmax) < 0x1p-100f;
  hipLaunchKernelGGL(k_ph_col0, dim3((unsigned)((P->Ny + 255) / 256)), dim3(256), 0, 0,
                     P->ty.as<float>(), P->tx.as<float>(), P->Ny, P->Nx, method, P->A, P->B,
                     P->alpha, P->db, cs, P->h0.as<float4>());
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(0);
  if (e != hipSuccess) {
    set_error("ph_create: %s", hipGetErrorString(e));
    ph_destroy(P);
    return TOMO_EHIP;
  }
  // launch shapes: rows one transform per workgroup, columns 2^lgC interleaved
  // transforms
  auto lds_attr = [&](const void *k, size_t bytes) {
    if (e == hipSuccess)
      e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  };
  with_ph_size(P->Nx, [&](auto ns) {
    constexpr int NS = decltype(ns)::value;
    P->rowThreads = NS > 0 ? fft_threads(P->fx.rule, NS) : fft_rt_threads(P->fx.d, 0);
    if (NS == 0 && P->rowThreads > 0)  // (one value a thread: short rows, as for the columns)
      P->rowThreads = std::max(P->rowThreads, std::min(256, P->Nx / 64 * 64));
    P->rowLds = sizeof(float2) * (NS > 0 ? lds_padded_len(NS) : P->Nx);
    lds_attr((const void *)k_ph_rows_fwd<NS>, P->rowLds);
    lds_attr((const void *)k_ph_rows_inv<NS>, P->rowLds);
  });
  with_ph_size(P->Ny, [&](auto ns) {
    constexpr int NS = decltype(ns)::value;
    P->colThreads = NS > 0 ? split_threads(NS, P->lgC) : fft_rt_threads(P->fy.d, P->lgC);
    if (shortCols && P->colThreads > 0)
      P->colThreads = std::max(P->colThreads, std::min(narrow ? 512 : 256,
                                                       (P->Ny << P->lgC) / 128 * 64));
    P->colLds = NS > 0 ? sizeof(float) * ((size_t)lds_padded_len(NS) << P->lgC)
                       : sizeof(float2) * ((size_t)P->Ny << P->lgC);
    lds_attr((const void *)k_ph_cols<NS>, P->colLds);
  });
  if (P->rowThreads <= 0 || P->rowThreads > 512 || P->colThreads <= 0 ||
      P->colThreads > 1024 || P->rowLds > max_lds_per_block() ||
      P->colLds > max_lds_per_block()) {
    set_error("ph_create: padded size %d x %d too large for one workgroup", P->Ny, P->Nx);
    ph_destroy(P);
    return TOMO_EINVAL;
  }
  if (e != hipSuccess) {
    set_error("ph_create: hipFuncSetAttribute failed: %s", hipGetErrorString(e));
    ph_destroy(P);
    return TOMO_EHIP;
  }
  *plan = P;
  return TOMO_OK;
}

extern "C" int ph_get_pads(const tomo_ph_plan *P, int64_t *py, int64_t *pz, int64_t *Ny,
                           int64_t *Nx) {
  clear_error();
  TOMO_REQUIRE(P != nullptr, "ph_get_pads: plan is NULL");
  if (py) *py = P->py;
  if (pz) *pz = P->pz;
  if (Ny) *Ny = P->Ny;
  if (Nx) *Nx = P->Nx;
  return TOMO_OK;
}

extern "C" int ph_apply(tomo_ph_plan *P, float *data, int64_t nproj, void *stream) {
  clear_error();
  TOMO_REQUIRE(P != nullptr && data != nullptr, "ph_apply: NULL argument");
  TOMO_REQUIRE(nproj >= 0, "ph_apply: nproj < 0");
  hipStream_t st = (hipStream_t)stream;
  const int dy = (int)P->dy, dz = (int)P->dz;
  for (int64_t b0 = 0; b0 < nproj; b0 += P->batch) {
    const unsigned nb = (unsigned)std::min<int64_t>(P->batch, nproj - b0);
    float *img = data + (size_t)b0 * dy * dz;
    {
      ProfScope ps_("k_ph_rows_fwd", st);
      with_ph_size(P->Nx, [&](auto ns) {
        hipLaunchKernelGGL(k_ph_rows_fwd<decltype(ns)::value>, dim3((unsigned)(dy / 2), nb),
                           dim3(P->rowThreads), P->rowLds, st, img, P->F.as<float2>(), P->fx.d,
                           dy, dz, P->pz, P->lgB, P->Fb);
      });
    }
    TOMO_LAUNCH_CHECK();
    {
      ProfScope ps_("k_ph_cols", st);
      with_ph_size(P->Ny, [&](auto ns) {
        hipLaunchKernelGGL(k_ph_cols<decltype(ns)::value>, dim3((unsigned)std::max(P->Nx / 2 >> P->lgC, 1), nb),
                           dim3(P->colThreads), P->colLds, st, P->F.as<float2>(), P->fy.d,
                           P->lgC, P->Nx, dy, P->py, P->ty.as<float>(), P->tx.as<float>(),
                           P->h0.as<float4>(), P->method, P->A, P->B, P->alpha, P->db, P->cHi,
                           P->cLo, P->div, P->Fb);
      });
    }
    TOMO_LAUNCH_CHECK();
    {
      ProfScope ps_("k_ph_rows_inv", st);
      with_ph_size(P->Nx, [&](auto ns) {
        hipLaunchKernelGGL(k_ph_rows_inv<decltype(ns)::value>, dim3((unsigned)(dy / 2), nb),
                           dim3(P->rowThreads), P->rowLds, st, img, P->F.as<float2>(), P->fx.d,
                           dy, dz, P->pz, P->lgB, P->Fb);
      });
    }
    TOMO_LAUNCH_CHECK();
  }
  return TOMO_OK;
}
