// layernorm.h — one row of the residual add + LayerNorm, by one wavefront: shared by the kernel that
// writes the normalised rows (decode_ops.hip) and the Linear that takes them as its input
// (linear.hip).
#pragma once

#include "wdrz_common.h"
#include "wdrz_launch.h"

namespace wdrz {
namespace {

template <typename T> struct Elem;
template <> struct Elem<Bf16> {
  static __device__ __forceinline__ float lo(uint32_t w) { return bf16_lo(w); }
  static __device__ __forceinline__ float hi(uint32_t w) { return bf16_hi(w); }
  static __device__ __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
  static __device__ __forceinline__ float round(float v) { return (float)(__bf16)v; }
  static __device__ __forceinline__ float load1(const void* p, int64_t i) {
    return (float)static_cast<const __bf16*>(p)[i];
  }
  static __device__ __forceinline__ float word(const uint32_t* w, int e) {  // element e of loaded words
    return (e & 1) ? hi(w[e >> 1]) : lo(w[e >> 1]);
  }
};
template <> struct Elem<F16> {
  static __device__ __forceinline__ float lo(uint32_t w) { return f16_lo(w); }
  static __device__ __forceinline__ float hi(uint32_t w) { return f16_hi(w); }
  static __device__ __forceinline__ uint32_t pack(float a, float b) { return pack_f16x2(a, b); }
  static __device__ __forceinline__ float round(float v) { return (float)(_Float16)v; }
  static __device__ __forceinline__ float load1(const void* p, int64_t i) {
    return (float)static_cast<const _Float16*>(p)[i];
  }
  static __device__ __forceinline__ float word(const uint32_t* w, int e) {  // element e of loaded words
    return (e & 1) ? hi(w[e >> 1]) : lo(w[e >> 1]);
  }
};
template <> struct Elem<F32> {
  static __device__ __forceinline__ float round(float v) { return v; }
  static __device__ __forceinline__ float load1(const void* p, int64_t i) {
    return static_cast<const float*>(p)[i];
  }
  static __device__ __forceinline__ float word(const uint32_t* w, int e) { return __uint_as_float(w[e]); }
};

__device__ __forceinline__ float wave_sum64(float v) {
  v = group_sum<16>(v);
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
}

// NC = 16-byte chunks per lane (n <= 512 * NC). The LayerNorm weight and bias are loaded with the
// row, so the only dependent round trip is the row itself. NP > 0: the delta is a Linear's output
// given as NP fp32 split-K partials [NP][rows][n] plus its bias, rounded to the storage type
// after the sum, as the Linear's own output is.
template <typename T, int NC, int NP> struct LnRow {
  u32x4 xw[NC], dw[NC], ww[NC], bw[NC];
  f32x4 pw[NC][NP > 0 ? 2 * NP : 1];

  __device__ __forceinline__ void load(const AddLnArgs& a, int64_t row, int lane) {
    const int nc = a.n >> 3;  // 8-element chunks
    const char* xrow = static_cast<const char*>(a.x) + row * a.x_stride * 2;
    const char* drow = NP ? nullptr : a.delta ? static_cast<const char*>(a.delta) + row * a.d_stride * 2 : nullptr;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int ci = lane + 64 * c;
      xw[c] = dw[c] = ww[c] = bw[c] = u32x4{0, 0, 0, 0};
      if (ci < nc) {
        xw[c] = *reinterpret_cast<const u32x4*>(xrow + ci * 16);
        if (drow) dw[c] = *reinterpret_cast<const u32x4*>(drow + ci * 16);
        if constexpr (NP > 0) {
          dw[c] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(a.dbias) + ci * 16);
#pragma unroll
          for (int z = 0; z < NP; ++z) {
            const float* pr = a.dpart + ((int64_t)z * a.rows + row) * a.n + ci * 8;
            pw[c][2 * z] = *reinterpret_cast<const f32x4*>(pr);
            pw[c][2 * z + 1] = *reinterpret_cast<const f32x4*>(pr + 4);
          }
        }
        ww[c] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(a.weight) + ci * 16);
        bw[c] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(a.bias) + ci * 16);
      }
    }
  }

  // store_x(chunk, words): the new residual, when there is a delta; store_y: the normalised row.
  template <typename StoreX, typename StoreY>
  __device__ __forceinline__ void finish(const AddLnArgs& a, int lane, StoreX store_x, StoreY store_y) {
    const int nc = a.n >> 3;
    const bool has_delta = NP > 0 || a.delta != nullptr;
    float v[NC][8];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int ci = lane + 64 * c;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[c][i] = 0.f;
      if (ci < nc) {
        float dl[8];
        if constexpr (NP > 0) {
          // the Linear's output: partials summed in split order, bias added, one rounding
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            float t = pw[c][i >> 2][i & 3];
#pragma unroll
            for (int z = 1; z < NP; ++z) t += pw[c][2 * z + (i >> 2)][i & 3];
            const float bb = (i & 1) ? Elem<T>::hi(dw[c][i >> 1]) : Elem<T>::lo(dw[c][i >> 1]);
            dl[i] = Elem<T>::round(t + bb);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            dl[2 * j] = Elem<T>::lo(dw[c][j]);
            dl[2 * j + 1] = Elem<T>::hi(dw[c][j]);
          }
        }
        u32x4 sw;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float s0 = Elem<T>::lo(xw[c][j]), s1 = Elem<T>::hi(xw[c][j]);
          if (has_delta) {
            s0 = Elem<T>::round(s0 + dl[2 * j]);
            s1 = Elem<T>::round(s1 + dl[2 * j + 1]);
            sw[j] = Elem<T>::pack(s0, s1);
          }
          v[c][2 * j] = s0;
          v[c][2 * j + 1] = s1;
          sum += s0 + s1;
        }
        if (has_delta) store_x(ci, sw);
      }
    }
    const float inv_n = 1.f / (float)a.n;
    const float mean = wave_sum64(sum) * inv_n;
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (lane + 64 * c < nc)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float d = v[c][i] - mean;
          sq += d * d;
        }
    const float rstd = 1.f / sqrtf(wave_sum64(sq) * inv_n + a.eps);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int ci = lane + 64 * c;
      if (ci < nc) {
        u32x4 yw;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float y0 = (v[c][2 * j] - mean) * rstd * Elem<T>::lo(ww[c][j]) + Elem<T>::lo(bw[c][j]);
          const float y1 = (v[c][2 * j + 1] - mean) * rstd * Elem<T>::hi(ww[c][j]) + Elem<T>::hi(bw[c][j]);
          yw[j] = Elem<T>::pack(y0, y1);
        }
        store_y(ci, yw);
      }
    }
  }
};

}  // namespace
}  // namespace wdrz
