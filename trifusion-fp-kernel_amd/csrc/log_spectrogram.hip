// Log power spectrogram of the TriFusion front end (front.py:46-90) in one pass:
// masking (samples past each clip's length, channels past its channel count),
// zero padding and framing (512 points every 160 samples, centred), the 400-point
// window, the real DFT, the channel sum of |X|^2, log(1e-6 + sum / channels), and
// frames past the clip's count cleared. Replaces a masked copy of the waveform, a
// padded copy, a copy of every windowed frame, two FFT launches and the log power
// pass: at 8 stereo clips of 8 s, ~70 us in seven launches against 14.5 us.
//
// One wave per frame, channels in turn. The 512 real points are 256 complex ones
// (x[2n] + i x[2n+1]), transformed by four radix-4 passes (decimation in
// frequency), a butterfly per lane and pass, exchanged through 2.5 KB of LDS per
// wave; bins follow from Z[k] and conj Z[256 - k]. What bounds it is the vector
// work, ~450 instructions per frame and channel; the waveform is read 3.2 times
// (overlapping frames), from L2.
#include "mfma_tile.h"

namespace tf {
namespace {

constexpr int kFft = 512, kHop = 160, kWindow = 400, kBins = 257, kWaves = 4;
constexpr int kPad0 = (kFft - kWindow) / 2;  // the window's place in the frame

// LDS place of point i: four points of padding per 16, so that every pass reads
// and writes its groups of 4 or 16 points on distinct banks.
__device__ __forceinline__ int place(int i) { return i + 4 * (i >> 4); }

__device__ __forceinline__ float2 cmul(float2 a, float2 w) {
  return make_float2(a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x);
}

// Base-4 digits of an index below 256 in reverse order.
__device__ __forceinline__ int reversed(int k) {
  return ((k & 3) << 6) | ((k & 12) << 2) | ((k >> 2) & 12) | ((k >> 6) & 3);
}

__global__ __launch_bounds__(64 * kWaves) void log_spectrogram_kernel(const float* __restrict__ audio,
                                                                      const float* __restrict__ window,
                                                                      const int64_t* __restrict__ lengths,
                                                                      const int64_t* __restrict__ channels,
                                                                      float* __restrict__ y, int C, int64_t N, int F,
                                                                      int64_t frames) {
  __shared__ float2 tw[384];  // exp(-2 pi i k / 512)
  __shared__ float win[kWindow];
  __shared__ float2 z[kWaves][256 + 64];
  const int tid = static_cast<int>(threadIdx.x);
  for (int k = tid; k < 384; k += 64 * kWaves) {
    float s, c;
    sincospif(-static_cast<float>(k) / 256.f, &s, &c);
    tw[k] = make_float2(c, s);
  }
  for (int k = tid; k < kWindow; k += 64 * kWaves) win[k] = window[k];
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  float2* zw = z[w];
  // the lane's twiddles of the first three passes (quarter spans 64, 16, 4; the last needs none)
  float2 t[3][3];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const int span = 64 >> (2 * p), step = 2 << (2 * p);
#pragma unroll
    for (int q = 1; q < 4; ++q) t[p][q - 1] = tw[step * q * (lane & (span - 1))];
  }
  for (int64_t fr = static_cast<int64_t>(blockIdx.x) * kWaves + w; fr < frames;
       fr += static_cast<int64_t>(gridDim.x) * kWaves) {
    const int64_t b = fr / F;
    const int f = static_cast<int>(fr - b * F);
    const int64_t len = lengths[b];
    float* out = y + fr * kBins;
    if (f >= len / kHop + 1) {
#pragma unroll
      for (int q = 0; q < 4; ++q) out[lane + 64 * q] = 0.f;
      if (lane == 0) out[256] = 0.f;
      continue;
    }
    const int64_t nch = channels[b];
    const int64_t first = static_cast<int64_t>(f) * kHop - kFft / 2;  // sample of point 0
    const int64_t stop = len < N ? len : N;
    float power[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < C && c < nch; ++c) {
      const float* x = audio + (b * C + c) * N;
      float2 a[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int p0 = 2 * (lane + 64 * q);  // points p0, p0 + 1 of the frame
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int j = p0 + e - kPad0;
          const int64_t s = first + p0 + e;
          v[e] = j >= 0 && j < kWindow && s >= 0 && s < stop ? x[s] * win[j] : 0.f;
        }
        a[q] = make_float2(v[0], v[1]);
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int span = 64 >> (2 * p);
        const int base = (lane / span) * 4 * span + (lane & (span - 1));
        if (p > 0) {
#pragma unroll
          for (int q = 0; q < 4; ++q) a[q] = zw[place(base + span * q)];
        }
        const float2 s02 = make_float2(a[0].x + a[2].x, a[0].y + a[2].y);
        const float2 d02 = make_float2(a[0].x - a[2].x, a[0].y - a[2].y);
        const float2 s13 = make_float2(a[1].x + a[3].x, a[1].y + a[3].y);
        const float2 d13 = make_float2(a[1].y - a[3].y, a[3].x - a[1].x);  // -i (a1 - a3)
        float2 o[4] = {make_float2(s02.x + s13.x, s02.y + s13.y), make_float2(d02.x + d13.x, d02.y + d13.y),
                       make_float2(s02.x - s13.x, s02.y - s13.y), make_float2(d02.x - d13.x, d02.y - d13.y)};
        if (p < 3) {
#pragma unroll
          for (int q = 1; q < 4; ++q) o[q] = cmul(o[q], t[p][q - 1]);
        }
        wave_sync();  // the pass's reads come before its writes to other lanes' places
#pragma unroll
        for (int q = 0; q < 4; ++q) zw[place(base + span * q)] = o[q];
        wave_sync();
      }
      // X[k] = (Z[k] + conj Z[256-k]) / 2 - i/2 exp(-2 pi i k / 512) (Z[k] - conj Z[256-k])
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        const int k = lane + 64 * q;
        if (q == 4 && lane > 0) break;
        const float2 u = zw[place(reversed(k & 255))], v = zw[place(reversed((256 - k) & 255))];
        const float2 e = make_float2(u.x + v.x, u.y - v.y), d = make_float2(u.x - v.x, u.y + v.y);
        const float2 r = cmul(d, tw[k]);
        const float re = 0.5f * (e.x + r.y), im = 0.5f * (e.y - r.x);
        power[q] += re * re + im * im;
      }
      wave_sync();
    }
    const float n = static_cast<float>(nch);
#pragma unroll
    for (int q = 0; q < 4; ++q) out[lane + 64 * q] = logf(1e-6f + power[q] / n);
    if (lane == 0) out[256] = logf(1e-6f + power[4] / n);
  }
}

}  // namespace
}  // namespace tf

extern "C" int tf_log_spectrogram(const float* audio, const float* window, const int64_t* lengths,
                                  const int64_t* channels, float* y, int64_t batch, int64_t chans, int64_t samples,
                                  void* stream) {
  if (!audio || !window || !lengths || !channels || !y) return TF_ERR_NULL;
  if (batch < 0 || chans < 1 || chans > 65535 || samples < 1 || samples > (int64_t(1) << 31)) return TF_ERR_SHAPE;
  if (batch == 0) return TF_OK;
  const int64_t frames_per = samples / tf::kHop + 1;
  if (batch > (int64_t(1) << 40) / (frames_per * tf::kBins)) return TF_ERR_SHAPE;
  const int64_t frames = batch * frames_per;
  // four frames per workgroup up to eight workgroups per CU, then several each
  const int64_t blocks = (frames + tf::kWaves - 1) / tf::kWaves;
  hipLaunchKernelGGL(tf::log_spectrogram_kernel, dim3(static_cast<uint32_t>(blocks < 2048 ? blocks : 2048)),
                     dim3(64 * tf::kWaves), 0, static_cast<hipStream_t>(stream), audio, window, lengths, channels, y,
                     static_cast<int>(chans), samples, static_cast<int>(frames_per), frames);
  return tf::launch_status();
}
