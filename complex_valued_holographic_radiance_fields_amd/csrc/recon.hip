// recon.hip — the loss side's hologram reconstruction around the
// propagation: the per-(frame, channel) hologram field from the phase map and
// the amplitude, the reconstructed intensity |u|^2, and the backward of both.
//
// Reference: propagator._reconstruct_impl (utils/propagator.py:548-636):
// for every frame f and channel c with laser power w = laser_powers[f][c],
// hologram = generate_complex_field(w * amplitude[c], phase[f] *
// phase_scale[c]) (= w a e^{i s phi}), zero pad, propagate to every depth,
// crop, then calculate_amplitude(.)**2.  Only pairs with w != 0 are formed
// (the reference's training uses laser_channel_power = eye(3): one channel
// per frame), as K fields in one array; the propagation between these
// kernels is the multi-distance band-limited ASM.
#include <cmath>
#include <cstdint>

#include "hrf_internal.h"

namespace hrf {
namespace {

constexpr int kReconThreads = 256;
constexpr int kMaxReconPairs = 64;

struct ReconPairs {
  int frame[kMaxReconPairs];
  int channel[kMaxReconPairs];
  float power[kMaxReconPairs];
  float scale[kMaxReconPairs];  // phase_scale[channel]
  // Is pair k the first of its frame / channel in the list?
  uint64_t first_frame, first_channel;
  int count;
};

// V consecutive values per thread, as wide loads and stores.
template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
  T v[V];
};

// Elements between consecutive frames, depths, channels and pixels.
struct PlaneStrides {
  int64_t f, d, c, i;
};

// fields[k][i] = power_k * amp[c_k][i] * e^{i scale_k * phase[f_k][i]}
__global__ __launch_bounds__(kReconThreads) void k_recon_fields(
    const float* __restrict__ amp, const float* __restrict__ phase, int64_t hw, ReconPairs pr,
    float2* __restrict__ fields) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kReconThreads + threadIdx.x;
  const int k = blockIdx.y;
  if (i >= hw) return;
  const float a = pr.power[k] * amp[static_cast<int64_t>(pr.channel[k]) * hw + i];
  const float th = phase[static_cast<int64_t>(pr.frame[k]) * hw + i] * pr.scale[k];
  float s, c;
  sincosf(th, &s, &c);
  fields[static_cast<int64_t>(k) * hw + i] = make_float2(a * c, a * s);
}

__global__ __launch_bounds__(kReconThreads) void k_recon_intensity(const float2* __restrict__ u,
                                                                   int64_t n,
                                                                   float* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kReconThreads + threadIdx.x;
  if (i >= n) return;
  const float2 v = u[i];
  out[i] = v.x * v.x + v.y * v.y;
}

// d|u|^2: grad_u = 2 g u (torch's convention for a real loss of complex u).
__global__ __launch_bounds__(kReconThreads) void k_recon_intensity_bwd(
    const float2* __restrict__ u, const float* __restrict__ g, int64_t n,
    float2* __restrict__ gu) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kReconThreads + threadIdx.x;
  if (i >= n) return;
  const float2 v = u[i];
  const float t = 2.0f * g[i];
  gu[i] = make_float2(t * v.x, t * v.y);
}

// Intensities of the lit pairs straight into the (F, D, C, hw) result, zeros
// where no pair falls: out[f][d][c][i] = |u[d][k][i]|^2 for pair k = (f, c).
// Bound by memory (8 bytes read and 4 written per lit pixel, 4 per unlit one);
// one pass in place of a fill of the whole result, the (D, K) intensities and
// a copy per pair: 17.4 us instead of 41 for 3 frames x 3 depths x 3 channels
// of 800^2, 3 pairs lit.
template <int V>
__global__ __launch_bounds__(kReconThreads) void k_recon_intensity_planes(
    const float2* __restrict__ u, int64_t hw, int D, int C, int bpp, ReconPairs pr,
    float* __restrict__ out) {
  const int plane = blockIdx.x / bpp;  // (f D + d) C + c
  const int64_t i =
      (static_cast<int64_t>(blockIdx.x - plane * bpp) * kReconThreads + threadIdx.x) * V;
  if (i >= hw) return;
  const int c = plane % C, fd = plane / C, d = fd % D, f = fd / D;
  int pair = -1;
  for (int k = 0; k < pr.count; ++k)
    if (pr.frame[k] == f && pr.channel[k] == c) pair = k;
  Pack<float, V> r;
#pragma unroll
  for (int j = 0; j < V; ++j) r.v[j] = 0.0f;
  if (pair >= 0) {
    const Pack<float2, V> z = *reinterpret_cast<const Pack<float2, V>*>(
        u + (static_cast<int64_t>(d) * pr.count + pair) * hw + i);
#pragma unroll
    for (int j = 0; j < V; ++j) r.v[j] = z.v[j].x * z.v[j].x + z.v[j].y * z.v[j].y;
  }
  *reinterpret_cast<Pack<float, V>*>(out + plane * hw + i) = r;
}

// The backward of that pass: gu[d][k][i] = 2 g[f][d][c][i] u[d][k][i], the
// gradient read in place (its strides; V > 1 needs contiguous pixels) instead
// of gathered into (D, K) first.  Bound by memory, 20 bytes per lit pixel: at
// the sizes above 21 us (5.5 TB/s) instead of 38.
template <int V>
__global__ __launch_bounds__(kReconThreads) void k_recon_intensity_planes_bwd(
    const float2* __restrict__ u, const float* __restrict__ g, PlaneStrides gs, int64_t hw,
    int bpp, ReconPairs pr, float2* __restrict__ gu) {
  const int plane = blockIdx.x / bpp;  // d K + k
  const int64_t i =
      (static_cast<int64_t>(blockIdx.x - plane * bpp) * kReconThreads + threadIdx.x) * V;
  if (i >= hw) return;
  const int d = plane / pr.count, k = plane - d * pr.count;
  const float* src = g + pr.frame[k] * gs.f + d * gs.d + pr.channel[k] * gs.c;
  Pack<float, V> t;
  if (V > 1)
    t = *reinterpret_cast<const Pack<float, V>*>(src + i);
  else
    t.v[0] = src[i * gs.i];
  const Pack<float2, V> z = *reinterpret_cast<const Pack<float2, V>*>(u + plane * hw + i);
  Pack<float2, V> r;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const float w = 2.0f * t.v[j];
    r.v[j] = make_float2(w * z.v[j].x, w * z.v[j].y);
  }
  *reinterpret_cast<Pack<float2, V>*>(gu + plane * hw + i) = r;
}

// z = w a e^{i s phi}: dL/da = w Re(gz e^{-i s phi}), dL/dphi = s Im(gz conj(z))
// summed over the pairs that use the channel / frame (each pixel loops over
// the pairs, so there are no atomics).  A channel's or frame's first pair
// writes its map and the later ones add to it; only maps of no pair are
// cleared (16.8 -> 14.2 us at 3 pairs of 800^2 against clearing every map).
__global__ __launch_bounds__(kReconThreads) void k_recon_fields_bwd(
    const float* __restrict__ amp, const float* __restrict__ phase, int64_t hw, ReconPairs pr,
    const float2* __restrict__ gfields, int F, int C, uint64_t lit_frames,
    uint64_t lit_channels, float* __restrict__ g_amp, float* __restrict__ g_phase) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kReconThreads + threadIdx.x;
  if (i >= hw) return;
  for (int c = 0; c < C; ++c)
    if (c >= 64 || !((lit_channels >> c) & 1)) g_amp[static_cast<int64_t>(c) * hw + i] = 0.0f;
  for (int f = 0; f < F; ++f)
    if (f >= 64 || !((lit_frames >> f) & 1)) g_phase[static_cast<int64_t>(f) * hw + i] = 0.0f;
  for (int k = 0; k < pr.count; ++k) {
    const int64_t ic = static_cast<int64_t>(pr.channel[k]) * hw + i;
    const int64_t jf = static_cast<int64_t>(pr.frame[k]) * hw + i;
    const float th = phase[jf] * pr.scale[k];
    float s, c;
    sincosf(th, &s, &c);
    const float2 gz = gfields[static_cast<int64_t>(k) * hw + i];
    const float re = gz.x * c + gz.y * s;    // Re(gz e^{-i th})
    const float im = gz.y * c - gz.x * s;    // Im(gz e^{-i th})
    const float a = pr.power[k] * amp[ic];
    const float va = pr.power[k] * re;
    const float vp = pr.scale[k] * a * im;   // Im(gz conj(z)) = a Im(gz e^{-i th})
    g_amp[ic] = ((pr.first_channel >> k) & 1) ? va : g_amp[ic] + va;
    g_phase[jf] = ((pr.first_frame >> k) & 1) ? vp : g_phase[jf] + vp;
  }
}

int pairs_of(const int32_t* frames, const int32_t* channels, const float* powers,
             const float* scales, int32_t K, int F, int C, ReconPairs* pr) {
  if (K < 1 || K > kMaxReconPairs || !frames || !channels || !powers || !scales) {
    set_error("reconstruction: 1..%d (frame, channel) pairs needed", kMaxReconPairs);
    return HRF_ERR_INVALID;
  }
  *pr = ReconPairs{};
  for (int k = 0; k < K; ++k) {
    if (frames[k] < 0 || frames[k] >= F || channels[k] < 0 || channels[k] >= C) {
      set_error("reconstruction: pair %d = (%d, %d) outside %d frames x %d channels", k,
                frames[k], channels[k], F, C);
      return HRF_ERR_INVALID;
    }
    pr->frame[k] = frames[k];
    pr->channel[k] = channels[k];
    pr->power[k] = powers[k];
    pr->scale[k] = scales[k];
    bool ff = true, fc = true;
    for (int j = 0; j < k; ++j) {
      ff = ff && frames[j] != frames[k];
      fc = fc && channels[j] != channels[k];
    }
    // (maps past the 64 that the clearing masks hold are cleared, then added to)
    if (ff && frames[k] < 64) pr->first_frame |= uint64_t{1} << k;
    if (fc && channels[k] < 64) pr->first_channel |= uint64_t{1} << k;
  }
  pr->count = K;
  return HRF_OK;
}

bool aligned(const void* p, size_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }

// Launch of the plane kernels at v pixels per thread: 4 where every plane
// starts and every access lands on a multiple of 4 values (16-byte loads and
// stores), else 1.  bpp: blocks per plane; false when planes x blocks exceeds
// a launch's blocks.
bool plane_grid(int64_t planes, int64_t hw, int v, int* bpp, uint32_t* blocks) {
  const int64_t per = (hw + int64_t{v} * kReconThreads - 1) / (int64_t{v} * kReconThreads);
  if (per > INT32_MAX || planes > INT32_MAX / per) return false;
  *bpp = static_cast<int>(per);
  *blocks = static_cast<uint32_t>(planes * per);
  return true;
}

}  // namespace
}  // namespace hrf

using namespace hrf;

extern "C" {

int hrf_recon_fields(const float* amplitude, const float* phase, int32_t F, int32_t C,
                     int64_t hw, const int32_t* frames, const int32_t* channels,
                     const float* powers, const float* scales, int32_t K, void* fields,
                     void* stream) {
  ReconPairs pr;
  HRF_TRY(pairs_of(frames, channels, powers, scales, K, F, C, &pr));
  if (hw <= 0 || !amplitude || !phase || !fields) {
    set_error("reconstruction fields: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_fields", s);
  hipLaunchKernelGGL(k_recon_fields, dim3(blocks_for(hw, kReconThreads), K),
                     dim3(kReconThreads), 0, s, amplitude, phase, hw, pr,
                     static_cast<float2*>(fields));
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

int hrf_recon_intensity(const void* field, int64_t n, float* intensity, void* stream) {
  if (n < 0 || (n > 0 && (!field || !intensity))) {
    set_error("reconstruction intensity: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  if (n == 0) return HRF_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_intensity", s);
  hipLaunchKernelGGL(k_recon_intensity, dim3(blocks_for(n, kReconThreads)), dim3(kReconThreads),
                     0, s, static_cast<const float2*>(field), n, intensity);
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

int hrf_recon_intensity_backward(const void* field, const float* grad_intensity, int64_t n,
                                 void* grad_field, void* stream) {
  if (n < 0 || (n > 0 && (!field || !grad_intensity || !grad_field))) {
    set_error("reconstruction intensity backward: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  if (n == 0) return HRF_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_intensity", s);
  hipLaunchKernelGGL(k_recon_intensity_bwd, dim3(blocks_for(n, kReconThreads)),
                     dim3(kReconThreads), 0, s, static_cast<const float2*>(field),
                     grad_intensity, n, static_cast<float2*>(grad_field));
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

int hrf_recon_intensity_planes(const void* field, int32_t F, int32_t D, int32_t C, int64_t hw,
                               const int32_t* frames, const int32_t* channels,
                               const float* powers, const float* scales, int32_t K,
                               float* intensity, void* stream) {
  ReconPairs pr;
  HRF_TRY(pairs_of(frames, channels, powers, scales, K, F, C, &pr));
  const int v = hw % 4 == 0 && aligned(field, 32) && aligned(intensity, 16) ? 4 : 1;
  const int64_t fd = static_cast<int64_t>(F) * D;
  int bpp = 0;
  uint32_t blocks = 0;
  if (hw <= 0 || D < 1 || !field || !intensity || fd > INT32_MAX / C ||
      !plane_grid(fd * C, hw, v, &bpp, &blocks)) {
    set_error("reconstruction intensity planes: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_intensity", s);
  auto* kern = v == 4 ? k_recon_intensity_planes<4> : k_recon_intensity_planes<1>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kReconThreads), 0, s,
                     static_cast<const float2*>(field), hw, D, C, bpp, pr, intensity);
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

int hrf_recon_intensity_planes_backward(const void* field, const float* grad_intensity,
                                        const int64_t* grad_strides, int32_t F, int32_t D,
                                        int32_t C, int64_t hw, const int32_t* frames,
                                        const int32_t* channels, const float* powers,
                                        const float* scales, int32_t K, void* grad_field,
                                        void* stream) {
  ReconPairs pr;
  HRF_TRY(pairs_of(frames, channels, powers, scales, K, F, C, &pr));
  if (hw <= 0 || D < 1 || !field || !grad_intensity || !grad_strides || !grad_field) {
    set_error("reconstruction intensity planes backward: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  const PlaneStrides gs{grad_strides[0], grad_strides[1], grad_strides[2], grad_strides[3]};
  const int v = hw % 4 == 0 && gs.i == 1 && gs.f % 4 == 0 && gs.d % 4 == 0 && gs.c % 4 == 0 &&
                        aligned(field, 32) && aligned(grad_intensity, 16) &&
                        aligned(grad_field, 32)
                    ? 4
                    : 1;
  int bpp = 0;
  uint32_t blocks = 0;
  if (!plane_grid(static_cast<int64_t>(D) * K, hw, v, &bpp, &blocks)) {
    set_error("reconstruction intensity planes backward: too many planes");
    return HRF_ERR_INVALID;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_intensity", s);
  auto* kern = v == 4 ? k_recon_intensity_planes_bwd<4> : k_recon_intensity_planes_bwd<1>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kReconThreads), 0, s,
                     static_cast<const float2*>(field), grad_intensity, gs, hw, bpp, pr,
                     static_cast<float2*>(grad_field));
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

int hrf_recon_fields_backward(const float* amplitude, const float* phase, int32_t F, int32_t C,
                              int64_t hw, const int32_t* frames, const int32_t* channels,
                              const float* powers, const float* scales, int32_t K,
                              const void* grad_fields, float* grad_amplitude,
                              float* grad_phase, void* stream) {
  ReconPairs pr;
  HRF_TRY(pairs_of(frames, channels, powers, scales, K, F, C, &pr));
  if (hw <= 0 || !amplitude || !phase || !grad_fields || !grad_amplitude || !grad_phase) {
    set_error("reconstruction fields backward: invalid size or null pointer");
    return HRF_ERR_INVALID;
  }
  uint64_t lit_frames = 0, lit_channels = 0;
  for (int k = 0; k < K; ++k) {
    if (frames[k] < 64) lit_frames |= uint64_t{1} << frames[k];
    if (channels[k] < 64) lit_channels |= uint64_t{1} << channels[k];
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  HRF_STAGE("recon_fields", s);
  hipLaunchKernelGGL(k_recon_fields_bwd, dim3(blocks_for(hw, kReconThreads)), dim3(kReconThreads),
                     0, s, amplitude, phase, hw, pr, static_cast<const float2*>(grad_fields), F,
                     C, lit_frames, lit_channels, grad_amplitude, grad_phase);
  HRF_LAUNCH_CHECK();
  return HRF_OK;
}

}  // extern "C"
