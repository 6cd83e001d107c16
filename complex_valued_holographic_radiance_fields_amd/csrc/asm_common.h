// asm_common.h — what the fused propagation passes share: the transfer
// function's geometry, its host constants, and the layout of the
// intermediate spectra.
#pragma once

#include <hip/hip_runtime.h>

#include "fast_trig.h"
#include "hrf_internal.h"

namespace hrf {
namespace {

constexpr int kFftBatch = 4;  // columns of an intermediate tile
constexpr double kTwoPiD = 2.0 * 3.14159265358979323846;

// Transfer-function geometry of natural-order spectral element (row i,
// column k): frequencies as torch.fft.fftfreq float32 values and the
// aperture on the fftshifted grid (same mapping as asm_prop.hip).
__device__ __forceinline__ void coords(int i, int kcol, int M, float sfreq, float ap,
                                       float* fxv, float* fyv, bool* inap) {
  const int h = M / 2;
  int kr = i + h;
  if (kr >= M) kr -= M;
  int kc = kcol + h;
  if (kc >= M) kc -= M;
  *fxv = static_cast<float>(kr - h) * sfreq;
  *fyv = static_cast<float>(kc - h) * sfreq;
  bool a = true;
  if (ap > 0.0f) {
    const float off = static_cast<float>(M) / 2.0f - 0.5f;
    const float x = static_cast<float>(kc) - off;
    const float y = static_cast<float>(kr) - off;
    a = x * x + y * y < ap * ap;
  }
  *inap = a;
}

// kz^2 and kz exactly as the reference kernel evaluates them
// (bandlimited_propagation_cuda.cu:60,65-67); kz2 <= 0 -> evanescent.
__device__ __forceinline__ float kz_of(float k, float fxv, float fyv, bool* prop) {
  const double a = kTwoPiD * static_cast<double>(fxv);
  const double b = kTwoPiD * static_cast<double>(fyv);
  const float kz2 = static_cast<float>((static_cast<double>(k * k) - a * a) - b * b);
  *prop = kz2 > 0.0f;
  return *prop ? sqrtf(kz2) : 0.0f;
}

struct AsmFftConsts {
  float k[kMaxChannels];
  float d[kMaxPlanes];
  float fxmax[kMaxPlanes * kMaxChannels];
  float fymax[kMaxPlanes * kMaxChannels];
  // 1 when the band limit of (plane, channel) passes every frequency of the
  // grid (decided on the host with the device's float arithmetic), so the
  // per-element test can be skipped.
  unsigned char band_all[kMaxPlanes * kMaxChannels];
};

// Intermediate spectra are stored tile-major: image `img` (h rows of N
// columns) as N/B column tiles, each h x B with the B columns innermost, at
// ((img * N/B + tile) * h + row) * B + col.  A column pass then reads and
// writes one contiguous h*B*8-byte run per tile, and a row pass touches
// B*B*8 = 128-byte runs.
__device__ __forceinline__ int64_t tile_off(int img, int ncb, int cb, int h, int r, int b, int B) {
  return ((static_cast<int64_t>(img) * ncb + cb) * h + r) * B + b;
}

__device__ __forceinline__ void map_cblock(int bid, int nblk, int* chan, int* cb, int ncb) {
  // XCD-aware: consecutive column tiles of a channel go to one XCD, so the
  // tiles of neighbouring blocks stream through the same L2.
  const int q = nblk >> 3, r = nblk & 7;
  const int x = bid & 7, i = bid >> 3;
  const int logical = (x < r) ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
  *chan = logical / ncb;
  *cb = logical - (*chan) * ncb;
}

// kz of spectral element (row frequency i, column frequency k), -1 where the
// evanescent cut or the aperture zeroes the transfer function.
__device__ __forceinline__ float kz_or_cut(float k0, int i, int k, int M, float sfreq, float ap) {
  float fx, fy;
  bool inap, prop;
  coords(i, k, M, sfreq, ap, &fx, &fy, &inap);
  const float kk = kz_of(k0, fx, fy, &prop);
  return prop && inap ? kk : -1.0f;
}

struct Band {
  float fxm, fym, d;
  bool all;
};
__device__ __forceinline__ Band band_of(const AsmFftConsts& mc, int p, int c) {
  return Band{mc.fxmax[p * kMaxChannels + c], mc.fymax[p * kMaxChannels + c], mc.d[p],
              mc.band_all[p * kMaxChannels + c] != 0};
}
// Whether the transfer function passes (i, k), given its kz.
__device__ __forceinline__ bool passes(const Band& bd, float kz, int i, int k, int M,
                                       float sfreq) {
  if (kz < 0.0f) return false;
  if (bd.all) return true;
  float fx, fy;
  bool inap;
  coords(i, k, M, sfreq, -1.0f, &fx, &fy, &inap);
  return fabsf(fx) < bd.fxm && fabsf(fy) < bd.fym;
}
__device__ __forceinline__ float2 turn(float2 x, float phase) {
  float sn, cs;
  sincos_big_ff(phase, &sn, &cs);
  return make_float2(x.x * cs - x.y * sn, x.x * sn + x.y * cs);
}

// The block's channel, intermediate tile, first column in it and first
// spectrum column.
template <int B>
__device__ __forceinline__ void column_block(int M, int* c, int* cb, int* col0, int* k0) {
  int hb;
  map_cblock(blockIdx.x, gridDim.x, c, &hb, M / B);
  *cb = hb / (kFftBatch / B);
  *col0 = (hb % (kFftBatch / B)) * B;
  *k0 = hb * B;
}

inline AsmFftConsts fft_consts(int P, int C, int M, double pitch, const float* wl, const float* dist) {
  AsmFftConsts mc{};
  for (int c = 0; c < C; ++c) mc.k[c] = asm_consts(wl[c], 0.0f, static_cast<float>(pitch), M, M).k;
  for (int p = 0; p < P; ++p) {
    mc.d[p] = dist[p];
    for (int c = 0; c < C; ++c) {
      const AsmConsts a = asm_consts(wl[c], dist[p], static_cast<float>(pitch), M, M);
      mc.fxmax[p * kMaxChannels + c] = a.fx_max;
      mc.fymax[p * kMaxChannels + c] = a.fy_max;
      // |fx| on the grid is at most float(M/2) * (float)(1/(M*pitch)), the
      // value of the most negative bin; the device tests |f| < f_max.
      const float fmax_grid = static_cast<float>(M / 2) *
                              static_cast<float>(1.0 / (static_cast<double>(M) * pitch));
      mc.band_all[p * kMaxChannels + c] = (fmax_grid < a.fx_max && fmax_grid < a.fy_max) ? 1 : 0;
    }
  }
  return mc;
}

inline float freq_step_of(int N, double pitch) {
  return static_cast<float>(1.0 / (static_cast<double>(N) * pitch));
}

// The transfer constants with the propagation direction reversed: k_col_fwd
// applies exp(+i d kz) and k_col_adj exp(-i d kz), so negated distances give
// the conjugate transfer function in the one and the plain one in the other.
// The band limits depend on d^2 and stay those of the given distances.
inline AsmFftConsts fft_consts_reversed(int P, int C, int M, double pitch, const float* wl,
                                 const float* dist) {
  AsmFftConsts mc = fft_consts(P, C, M, pitch, wl, dist);
  for (int p = 0; p < P; ++p) mc.d[p] = -mc.d[p];
  return mc;
}

}  // namespace
}  // namespace hrf
