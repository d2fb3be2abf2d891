// logmel.hip — gfx950 kernels for Whisper's log-mel front end.
//
// Replaces LogMelSpectrogram (src/whisperdrz/audio.py:81-156), which the reference runs on the
// CPU per 30-s window (transcriber.py:1091-1092):
//   stft(n_fft 400, hop 160, periodic Hann, center + reflect padding) -> |X|^2 of all frames but
//   the last -> slaney mel filterbank (torchaudio MelScale, norm/mel_scale "slaney") ->
//   log10(max(mel, 1e-10)) -> max(log, max_over_window - 8) -> (x + 4) / 4 -> pad with -1.5 /
//   truncate to target_frames.
//
// Two launches:
//   logmel_spec_kernel   one workgroup per (30 frames, window), 5 wavefronts of 6 frames. The
//                        frames' samples (overlapping by 240) are staged once in LDS with the
//                        reflect padding; each wavefront runs its frames' real 400-point
//                        transforms as complex 200-point ones (even samples + i odd samples) in
//                        registers and LDS, the powers go to LDS, and the filterbank is applied
//                        as the two weights each bin has; (log10 + 4) / 4 is stored, and the workgroup's
//                        maximum of its window goes to the workspace.
//   logmel_finish_kernel raises what lies below max - 8, and writes -1.5 past the last frame.
// fp32 throughout, like the reference; window, twiddles and filterbank are computed in double and
// rounded once.
//
// Why an FFT: the direct transform on the fp32 matrix cores (a [32 x 400] x [400 x 512] product
// per 32 frames, the form before this one) took 240 us for 16 windows of 30 s and 50 us for one,
// after an init launch that rebuilt its tables (3.3 us); the 55 MB this must move take 11 us. Now
// 62-67 us for 16 windows and 14-15 us for one (a whole call 237 -> 71 and 53.6 -> 16.4 us), and nearer
// to 64-bit results (3.6e-7 against 5.3e-7). What bounds it, by counters (16 windows): VALU issue
// takes 46% of the SIMDs' busy cycles (1940 instructions per wavefront, i.e. per 6 frames) with 1.8
// wavefronts on a SIMD on average; a wavefront issues them for a quarter of its time and waits for
// half of it, for samples, LDS and the other wavefronts at a barrier. No part's removal takes more than a sixth
// (transforms' arithmetic 3 us, filterbank loop 12, filter weights 3, stores 4 of the call's 76 us
// when it was measured).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wdrz_common.h"
#include "wdrz_launch.h"

namespace wdrz {
namespace {

constexpr int kNfft = 400;
constexpr int kHop = 160;
constexpr int kBins = kNfft / 2 + 1;  // 201
constexpr int kHalf = kNfft / 2;      // length of the complex transform
constexpr int kWaveFrames = 6;        // 60 of 64 lanes: 10 lanes a frame, then 20 lanes two frames
constexpr int kWaves = 5;
constexpr int kThreads = 64 * kWaves;
constexpr int kFrames = kWaveFrames * kWaves;  // 30 a workgroup: 100 workgroups a 30-s window
constexpr int kSeg = (kFrames - 1) * kHop + kNfft;  // samples a workgroup stages
constexpr int kSegLoads = (kSeg + kThreads - 1) / kThreads;
// Samples are stored with 52 floats of padding per hop: the frames of a wavefront then start 20
// banks apart, so the 10 float2 each reads at once fall in different banks.
constexpr int kHopPad = 52;
__device__ __forceinline__ int seg_pos(int j) { return j + kHopPad * (j / kHop); }
// A frame's 200 complex values, and 2 of padding (202 = 10 mod 32: the 10-lane groups of the first
// stage write different banks). A wavefront's 6 frames are its own region, reused for the powers.
constexpr int kFramePitch = kHalf + 2;                   // float2
constexpr int kWaveFloats = 2 * kWaveFrames * kFramePitch;
// Powers: four bins of a frame together, [bin / 4][frame][4] within the wavefront's region, so that
// the filterbank reads four bins per lane at once. Odd wavefronts' powers start 32 floats in: the
// 30 frames' reads then spread evenly over the banks.
constexpr int kPGroups = (kBins + 3) / 4;  // the last 3 of 204 stay zero
__device__ __forceinline__ int power_pos(int wave, int fr, int k) {
  return wave * kWaveFloats + 32 * (wave & 1) + ((k >> 2) * kWaveFrames + fr) * 4 + (k & 3);
}
constexpr int kMaxMels = 128;
// filter m's weights, in groups of four bins aligned like the powers: the groups from bin
// start[m] / 4 * 4 on, at group (start[m] + start[m + 1] + 6 m) / 4. A filter of n bins touches at
// most (n + 6) / 4 groups, which is what the next filter's place is further on.
constexpr int kWeights = ((2 * kBins + 6 * kMaxMels) / 4 + 4) * 4;
constexpr int kMaxParts = 128;  // workgroups a window (= maxima in the workspace)
static_assert(kSeg + kHopPad * (kSeg / kHop) + 1 <= kWaves * kWaveFloats, "sample buffer");
static_assert(32 + 4 * kWaveFrames * kPGroups <= kWaveFloats, "power tile");

// Three workgroups a CU need at most 42 of the 128 units of 1280 bytes that LDS is given out in.
static_assert(4 * (kWaves * kWaveFloats + kWeights + kMaxMels) <= 42 * 1280, "three workgroups a CU");

// ---- tables, computed at compile time in double -------------------------------------------------
constexpr double kPi = 3.14159265358979323846;
// Taylor series on |x| <= pi/4 (the next term is below 1e-20)
constexpr double sin_series(double x) {
  double t = x, s = x;
  for (int i = 1; i < 10; ++i) {
    t *= -x * x / ((2 * i) * (2 * i + 1));
    s += t;
  }
  return s;
}
constexpr double cos_series(double x) {
  double t = 1.0, s = 1.0;
  for (int i = 1; i < 10; ++i) {
    t *= -x * x / ((2 * i - 1) * (2 * i));
    s += t;
  }
  return s;
}
// cos(2 pi t / n) for 0 <= t <= n, n a multiple of 8, folded to the first eighth of a turn
constexpr double cos_turn(int t, int n) {
  if (2 * t > n) t = n - t;
  if (4 * t > n) return -cos_turn(n / 2 - t, n);
  if (8 * t > n) return sin_series(2.0 * kPi * (n / 4 - t) / n);
  return cos_series(2.0 * kPi * t / n);
}
constexpr double sin_turn(int t, int n) { return 4 * t >= n ? cos_turn(t - n / 4, n) : cos_turn(t + 3 * n / 4, n); }

struct MelTables {
  float window[kNfft];      // periodic Hann, halved (the even / odd split's 1/2)
  float2 tw[20 * 10];       // e^(-2 pi i n1 k1 / 200) at [k1][n1]
  float2 split[kHalf / 2 + 1];  // e^(-2 pi i k / 400)
};
constexpr MelTables make_tables() {
  MelTables m{};
  for (int i = 0; i < kNfft; ++i) m.window[i] = 0.5f * (float)(0.5 - 0.5 * cos_turn(i, kNfft));
  for (int k1 = 0; k1 < 20; ++k1)
    for (int n1 = 0; n1 < 10; ++n1) {
      m.tw[k1 * 10 + n1].x = (float)cos_turn(n1 * k1, kHalf);
      m.tw[k1 * 10 + n1].y = (float)-sin_turn(n1 * k1, kHalf);
    }
  for (int k = 0; k <= kHalf / 2; ++k) {
    m.split[k].x = (float)cos_turn(k, kNfft);
    m.split[k].y = (float)-sin_turn(k, kNfft);
  }
  return m;
}
__device__ constexpr MelTables kTables = make_tables();

// ---- small transforms (forward, e^(-i)) -----------------------------------------------------------
struct Cplx {
  float r, i;
};
__device__ __forceinline__ Cplx operator+(Cplx a, Cplx b) { return {a.r + b.r, a.i + b.i}; }
__device__ __forceinline__ Cplx operator-(Cplx a, Cplx b) { return {a.r - b.r, a.i - b.i}; }

__device__ __forceinline__ void dft5(const Cplx* x, Cplx* y) {
  constexpr float c1 = (float)cos_turn(8, 40), c2 = (float)cos_turn(16, 40);
  constexpr float s1 = (float)sin_turn(8, 40), s2 = (float)sin_turn(16, 40);
  const Cplx t1 = x[1] + x[4], t2 = x[2] + x[3], t3 = x[1] - x[4], t4 = x[2] - x[3];
  y[0] = x[0] + t1 + t2;
  const Cplx m1 = {x[0].r + c1 * t1.r + c2 * t2.r, x[0].i + c1 * t1.i + c2 * t2.i};
  const Cplx m2 = {x[0].r + c2 * t1.r + c1 * t2.r, x[0].i + c2 * t1.i + c1 * t2.i};
  const Cplx n1 = {s1 * t3.r + s2 * t4.r, s1 * t3.i + s2 * t4.i};
  const Cplx n2 = {s2 * t3.r - s1 * t4.r, s2 * t3.i - s1 * t4.i};
  y[1] = {m1.r + n1.i, m1.i - n1.r};  // m1 - i n1
  y[4] = {m1.r - n1.i, m1.i + n1.r};
  y[2] = {m2.r + n2.i, m2.i - n2.r};
  y[3] = {m2.r - n2.i, m2.i + n2.r};
}

// 20 and 10 points by the prime-factor map (n = 5a + 4b, k = 5q + 16r mod 20; n = 5a + 2b,
// k = 5q + 6r mod 10): no twiddles between the factors.
__device__ __forceinline__ void dft20(Cplx* v) {
  Cplx f[4][5];
#pragma unroll
  for (int b = 0; b < 5; ++b) {
    const Cplx x0 = v[(4 * b) % 20], x1 = v[(5 + 4 * b) % 20], x2 = v[(10 + 4 * b) % 20], x3 = v[(15 + 4 * b) % 20];
    const Cplx p = x0 + x2, m = x0 - x2, q = x1 + x3, n = x1 - x3;
    f[0][b] = p + q;
    f[2][b] = p - q;
    f[1][b] = {m.r + n.i, m.i - n.r};  // m - i n
    f[3][b] = {m.r - n.i, m.i + n.r};
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    Cplx y[5];
    dft5(f[q], y);
#pragma unroll
    for (int r = 0; r < 5; ++r) v[(5 * q + 16 * r) % 20] = y[r];
  }
}
__device__ __forceinline__ void dft10(Cplx* v) {
  Cplx f[2][5];
#pragma unroll
  for (int b = 0; b < 5; ++b) {
    const Cplx x0 = v[(2 * b) % 10], x1 = v[(5 + 2 * b) % 10];
    f[0][b] = x0 + x1;
    f[1][b] = x0 - x1;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    Cplx y[5];
    dft5(f[q], y);
#pragma unroll
    for (int r = 0; r < 5; ++r) v[(5 * q + 6 * r) % 10] = y[r];
  }
}

// Edge j of the slaney mel filters (3 mels per 200 Hz below 1 kHz, 27 mels per factor 6.4 above):
// n_mels + 2 points evenly spaced in mels over [0, 8 kHz].
__device__ __forceinline__ double mel_edge(int j, int n_mels) {
  const double f_sp = 200.0 / 3.0, logstep = 0.068751777420949123;  // log(6.4) / 27
  const double mel_max = 15.0 + 2.0794415416798357 / logstep;       // log(8000 / 1000) = 2.079...
  const double m = mel_max * j / (n_mels + 1);
  return m < 15.0 ? f_sp * m : 1000.0 * exp(logstep * (m - 15.0));
}

// log10 of a normal number or infinity: log2 (one instruction, no denormals to scale) times log10(2) in
// two parts (inf - inf between them, so infinity is returned as it is).
__device__ __forceinline__ float log10_normal(float x) {
  constexpr float hi = 0.30102999f, lo = (float)(0.30102999566398119521 - (double)hi);
  const float y = __builtin_amdgcn_logf(x);
  const float r = y * hi;
  const float v = r + __builtin_fmaf(y, lo, __builtin_fmaf(y, hi, -r));
  return y < INFINITY ? v : y;
}

// LDS ops of one wavefront run in order: between its own writes and reads only the compiler has to
// be kept from moving them.
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

__global__ __launch_bounds__(kThreads) void logmel_spec_kernel(LogMelArgs a) {
  const int b = blockIdx.y;
  const int N = a.n_samples;

  __shared__ __align__(16) float buf[kWaves * kWaveFloats];  // samples, then transforms and powers
  __shared__ __align__(16) float wts[kWeights];
  __shared__ uint32_t filt[kMaxMels];      // first power group, groups << 8, first weight << 16
  // until the first samples are stored: the edges, and the first bin at or above each
  double* edges = reinterpret_cast<double*>(buf);
  uint8_t* start = reinterpret_cast<uint8_t*>(edges + kMaxMels + 2);
  auto wt_base = [&](int m) { return (start[m] + start[m + 1] + 6 * m) / 4 * 4; };

  const float* x = a.audio + (int64_t)b * a.audio_stride;
  const int n_tiles = (a.n_frames + kFrames - 1) / kFrames;
  float vmax = -INFINITY;
  for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
    const int f0 = tile * kFrames;
    // tables and addresses are formed again for each tile: kept across tiles they would spill
    const MelTables* tab = &kTables;
    int tid = threadIdx.x;
    asm volatile("" : "+s"(tab), "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Padded sample j of this tile is original sample 160 f0 + j - 200, reflected at both ends.
    float smp[kSegLoads];
    const int o0 = kHop * f0 - kNfft / 2;
    const bool inside = o0 >= 0 && o0 + kSeg <= N;
#pragma unroll
    for (int i = 0; i < kSegLoads; ++i) {
      const int j = tid + kThreads * i;
      int o = o0 + j;
      if (!inside) {
        o = o < 0 ? -o : o;
        o = o >= N ? 2 * (N - 1) - o : o;
        o = o < 0 ? 0 : o;  // frames past the end only
      }
      smp[i] = j < kSeg ? x[o] : 0.f;
    }
    if (tile == (int)blockIdx.x) {
      // the filterbank, while the samples are on their way: bin k lies between edges j and j + 1,
      // so it is on the rising side of filter j and on the falling side of filter j - 1
      for (int j = tid; j < a.n_mels + 2; j += kThreads) {
        const double f = mel_edge(j, a.n_mels);
        edges[j] = f;
        start[j] = j == a.n_mels + 1 ? kBins : (int)ceil(f / 40.0);  // bins are 40 Hz apart
      }
      for (int i = tid; i < kWeights; i += kThreads) wts[i] = 0.f;
      __syncthreads();
      for (int k = tid; k < kBins; k += kThreads) {
        int lo = 0, hi = a.n_mels + 1;  // the last edge interval whose first bin is <= k
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (start[mid] <= k) lo = mid;
          else hi = mid;
        }
        const double f = 40.0 * k, e0 = edges[lo], e1 = edges[lo + 1];
        const double down = (f - e0) / (e1 - e0), up = (e1 - f) / (e1 - e0);
        if (lo < a.n_mels)
          wts[wt_base(lo) + k - (start[lo] & ~3)] = (float)((down > 0.0 ? down : 0.0) * 2.0 / (edges[lo + 2] - e0));
        if (lo > 0)
          wts[wt_base(lo - 1) + k - (start[lo - 1] & ~3)] = (float)((up > 0.0 ? up : 0.0) * 2.0 / (e1 - edges[lo - 1]));
      }
      for (int m = tid; m < a.n_mels; m += kThreads) {
        const int g0 = start[m] >> 2, g1 = (start[m + 2] + 3) >> 2;
        filt[m] = (uint32_t)g0 | (uint32_t)(g1 - g0) << 8 | (uint32_t)wt_base(m) << 16;
      }
      __syncthreads();  // the samples take the edges' place
    }
#pragma unroll
    for (int i = 0; i < kSegLoads; ++i) {
      const int j = tid + kThreads * i;
      if (j < kSeg) buf[seg_pos(j)] = smp[i];
    }
    __syncthreads();

    // ---- stage 1: lane (frame, n1) transforms z[n1 + 10 n2] over n2, z[n] = x[2n] + i x[2n + 1] ----
    const int l = lane < 60 ? lane : 59;  // the last four lanes repeat lane 59
    Cplx v[20];
    {
      const int fr = l / 10, n1 = l % 10;
      const float* s = buf + (kHop + kHopPad) * (kWaveFrames * wave + fr) + 2 * n1;
#pragma unroll
      for (int n2 = 0; n2 < 20; ++n2) {
        const float2 z = *reinterpret_cast<const float2*>(s + 20 * n2 + kHopPad * (n2 / 8));
        const float2 w = *reinterpret_cast<const float2*>(&tab->window[2 * n1 + 20 * n2]);
        v[n2] = {z.x * w.x, z.y * w.y};
      }
      __builtin_amdgcn_sched_barrier(0);
      dft20(v);
      __builtin_amdgcn_sched_barrier(0);  // the twiddles' loads above would take 40 registers more
      __syncthreads();  // every wavefront has read its samples: the buffer becomes the transforms'
      float2* A = reinterpret_cast<float2*>(buf + wave * kWaveFloats) + fr * kFramePitch + n1;
#pragma unroll
      for (int k1 = 0; k1 < 20; ++k1) {
        const float2 t = tab->tw[k1 * 10 + n1];
        A[10 * k1] = make_float2(v[k1].r * t.x - v[k1].i * t.y, v[k1].r * t.y + v[k1].i * t.x);
      }
    }
    wave_fence();
    // ---- stage 2: lane (frame pair, k1) transforms over n1, for both frames: Z[k1 + 20 k2] ----
    {
      const int k1 = l % 20;
      float2* A = reinterpret_cast<float2*>(buf + wave * kWaveFloats) + 2 * (l / 20) * kFramePitch;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int n = 0; n < 10; n += 2) {
          const float4 z = *reinterpret_cast<const float4*>(A + u * kFramePitch + 10 * k1 + n);
          v[10 * u + n] = {z.x, z.y};
          v[10 * u + n + 1] = {z.z, z.w};
        }
      wave_fence();
      dft10(v);
      dft10(v + 10);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int k2 = 0; k2 < 10; ++k2)
          A[u * kFramePitch + k1 + 20 * k2] = make_float2(v[10 * u + k2].r, v[10 * u + k2].i);
    }
    wave_fence();
    // ---- powers of bins k and 200 - k from Z[k] and Z[200 - k] (even +- e^(-2 pi i k / 400) odd) ----
    {
      constexpr int kPairs = kHalf / 2 + 1, kAll = kWaveFrames * kPairs, kRounds = (kAll + 63) / 64;
      const float2* Z = reinterpret_cast<const float2*>(buf + wave * kWaveFloats);
      float lo[kRounds], hi[kRounds];
#pragma unroll
      for (int i = 0; i < kRounds; ++i) {
        const int q = min(lane + 64 * i, kAll - 1);
        const int fr = q / kPairs, k = q % kPairs;
        const float2 z = Z[fr * kFramePitch + k];
        const float2 y = Z[fr * kFramePitch + (k ? kHalf - k : 0)];
        const float2 w = tab->split[k];
        const float er = z.x + y.x, ei = z.y - y.y;     // even part (of the halved samples)
        const float od = z.y + y.y, oi = y.x - z.x;     // odd part
        const float tr = w.x * od - w.y * oi, ti = w.x * oi + w.y * od;
        lo[i] = (er + tr) * (er + tr) + (ei + ti) * (ei + ti);
        hi[i] = (er - tr) * (er - tr) + (ei - ti) * (ei - ti);
      }
      wave_fence();
#pragma unroll
      for (int i = 0; i < kRounds; ++i) {
        const int q = min(lane + 64 * i, kAll - 1);
        const int fr = q / kPairs, k = q % kPairs;
        buf[power_pos(wave, fr, k)] = lo[i];
        buf[power_pos(wave, fr, kHalf - k)] = hi[i];
      }
      if (lane < 3 * kWaveFrames) buf[power_pos(wave, lane / 3, kBins + lane % 3)] = 0.f;
    }
    __syncthreads();

    // ---- filterbank and log10: half-wavefront = one mel, lane = frame; mels 2p and 2p + 1 are
    // about equally wide, so the halves' loops end together ----
    {
      const int fr = min(lane & 31, kFrames - 1), f = f0 + fr;
      const float* P = buf + power_pos(fr / kWaveFrames, fr % kWaveFrames, 0);
      const bool mine = (lane & 31) < kFrames && f < a.n_frames;  // frames past the last: no maximum
      int mel = 2 * wave + (lane >> 5);
      float* out = a.out + (int64_t)b * a.os[0] + (int64_t)mel * a.os[1] + f;
      const int64_t step = 2 * kWaves * a.os[1];
      for (; mel < a.n_mels; mel += 2 * kWaves, out += step) {
        const uint32_t d = filt[mel];
        const float* p = P + 4 * kWaveFrames * (d & 0xff);
        const float* w = wts + (d >> 16);
        const float* end = w + 4 * ((d >> 8) & 0xff);
        float acc = 0.f;
        for (; w != end; w += 4, p += 4 * kWaveFrames) {  // weights of the bins outside the filter are zero
          const f32x4 pv = *reinterpret_cast<const f32x4*>(p);
          const f32x4 wv = *reinterpret_cast<const f32x4*>(w);
          acc += (pv[0] * wv[0] + pv[1] * wv[1]) + (pv[2] * wv[2] + pv[3] * wv[3]);
        }
        const float lv = log10_normal(fmaxf(acc, 1e-10f));
        if (mine) {
          vmax = fmaxf(vmax, lv);
          if (f < a.out_frames) *out = (lv + 4.0f) / 4.0f;
        }
      }
    }
    __syncthreads();  // the next tile's samples overwrite the powers
  }
  // this workgroup's maximum of the window
  const int tid = threadIdx.x;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o));
  if ((tid & 63) == 0) buf[tid >> 6] = vmax;
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < kWaves; ++w) vmax = fmaxf(vmax, buf[w]);
    a.part_max[(int64_t)b * kMaxParts + blockIdx.x] = vmax;
  }
}

// One row (window, mel) piece of 256 VEC frames per workgroup. The rows hold (x + 4) / 4 already;
// rounding keeps the order, so max(x, max - 8) scaled is the larger of the two scaled values, and
// only frames below that floor (and the padding) are written. VEC 4: 16-byte accesses, for rows that
// start 16-byte aligned and hold whole groups of four. Reading and writing every frame took 10.4 us
// of 16 windows' call, this 8.6.
template <int VEC>
__global__ __launch_bounds__(256) void logmel_finish_kernel(LogMelArgs a) {
  const int b = blockIdx.z, m = blockIdx.y;
  const int f = (blockIdx.x * 256 + threadIdx.x) * VEC;
  float* p = a.out + (int64_t)b * a.os[0] + (int64_t)m * a.os[1] + f;
  float v[VEC];
  const bool any = f < a.n_frames && f < a.out_frames;
  if (any) __builtin_memcpy(v, p, sizeof(v));
  // the window's maximum: every wavefront reduces the workgroups' maxima
  float vmax = -INFINITY;
  for (int i = threadIdx.x & 63; i < a.parts; i += 64) vmax = fmaxf(vmax, a.part_max[(int64_t)b * kMaxParts + i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o));
  if (f >= a.out_frames) return;
  const float floor_v = (vmax - 8.0f + 4.0f) / 4.0f;
  bool write = false;
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    const float old = v[i];
    v[i] = f + i < a.n_frames ? fmaxf(old, floor_v) : -1.5f;  // audio.py:133-137
    write = write || f + i >= a.n_frames || old < floor_v;
  }
  if (write) __builtin_memcpy(p, v, sizeof(v));
}

}  // namespace

// Workspace: kMaxParts maxima per window.
size_t logmel_workspace_bytes(int64_t B, int64_t n_mels) {
  (void)n_mels;
  return (size_t)B * kMaxParts * sizeof(float);
}

hipError_t launch_logmel(LogMelArgs a, void* ws, hipStream_t stream) {
  a.part_max = static_cast<float*>(ws);
  const int tiles = (a.n_frames + kFrames - 1) / kFrames;
  a.parts = tiles < kMaxParts ? tiles : kMaxParts;
  hipLaunchKernelGGL(logmel_spec_kernel, dim3(a.parts, a.B), dim3(kThreads), 0, stream, a);
  const bool vec = (reinterpret_cast<uintptr_t>(a.out) & 15u) == 0 && a.out_frames % 4 == 0 && a.os[0] % 4 == 0 &&
                   a.os[1] % 4 == 0;
  if (vec)
    hipLaunchKernelGGL(logmel_finish_kernel<4>, dim3((a.out_frames + 1023) / 1024, a.n_mels, a.B), dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL(logmel_finish_kernel<1>, dim3((a.out_frames + 255) / 256, a.n_mels, a.B), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace wdrz
