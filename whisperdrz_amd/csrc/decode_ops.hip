// decode_ops.hip — the small per-step operations of the captured decode step, fused.
//
// 1. wdrz_add_layernorm: the residual add that closes a sub-layer and the LayerNorm that opens
//    the next one (src/whisperdrz/model.py:420-433: x = x + attn(attn_ln(x)); x = x +
//    cross_attn(cross_attn_ln(x)); x = x + mlp(mlp_ln(x)); the next block's attn_ln, or the
//    final ln, model.py:609-613). x += delta is rounded to the storage type as torch's add is;
//    the LayerNorm (eps 1e-5, affine) is computed in fp32 from the rounded sum, as torch's
//    LayerNorm does for 16-bit inputs, and rounded once. One wavefront per row; the row stays in
//    registers between the mean and the variance pass.
// 2. wdrz_step_begin / wdrz_step_end: what a cached step does around its blocks (src/whisperdrz/
//    model.py:586-613): x = token embedding + positional embedding with the first LayerNorm, the
//    int32 slot map and every layer's gathered cache lengths; after the blocks the lengths' bump.
//    One launch each instead of six and three of torch's (2-4 us each for a few KB).
// 3. wdrz_masked_argmax: decode_batch's greedy sampling tail (src/whisperdrz/decoding.py:
//    1729-1761): masked = logits + (-65504 where blocked), then the repetition penalty
//    (x > 0 ? x / 1.2 : x * 1.2 where penalised), argmax. Each step rounds to the logits' type
//    as the torch ops do; ties go to the lowest index, as torch.argmax. One workgroup per row.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layernorm.h"
#include "wdrz_common.h"
#include "wdrz_launch.h"

namespace wdrz {
namespace {

// ---- residual add + LayerNorm (16-bit rows of n <= 64*8*NC elements), one wavefront per row ----
template <typename T, int NC, int NP>
__global__ __launch_bounds__(256) void add_layernorm_kernel(AddLnArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= a.rows) return;
  char* xrow = static_cast<char*>(a.x) + row * a.x_stride * 2;
  char* yrow = static_cast<char*>(a.y) + row * a.y_stride * 2;
  LnRow<T, NC, NP> r;
  r.load(a, row, lane);
  r.finish(a, lane, [&](int c, u32x4 w) { *reinterpret_cast<u32x4*>(xrow + c * 16) = w; },
           [&](int c, u32x4 w) { *reinterpret_cast<u32x4*>(yrow + c * 16) = w; });
}

// ---- step prologue and epilogue -------------------------------------------------------------
// Workgroups [0, ceil(rows / 4)): a wavefront per row (b, t) looks up its two embedding rows, adds
// them (rounded as torch's add) and normalises the sum. The workgroups behind them: one thread per
// (layer, batch row) gathers a cache length, one per batch row converts a slot id. Slots and
// positions count from the end when negative, as in torch's indexing (the slot map keeps the id as
// it is: attention gives such a row NaN); a token, position or slot out of range reads nothing and
// gives a NaN row (a slot through its length -1).
template <typename T, int NC>
__global__ __launch_bounds__(256) void step_begin_kernel(StepArgs a, AddLnArgs ln) {
  const int row_wgs = (a.B * a.sq + 3) / 4;
  if ((int)blockIdx.x >= row_wgs) {
    const int i = ((int)blockIdx.x - row_wgs) * 256 + threadIdx.x;
    const int b = i % a.B, l = i / a.B;
    if (l > a.n_layers) return;
    const int64_t slot = a.slots ? a.slots[b] : b;
    if (l == a.n_layers) {
      if (a.slots) a.slots32[b] = (int32_t)slot;
    } else {
      const int64_t s = slot < 0 ? slot + a.n_slots : slot;
      a.seqlens[(int64_t)l * a.B + b] = s >= 0 && s < a.n_slots ? a.lens[(int64_t)l * a.n_slots + s] : -1;
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.B * a.sq) return;
  const int b = row / a.sq, t = row % a.sq;
  const int64_t tok = a.tokens[b * a.ts[0] + t * a.ts[1]];
  int64_t pos = a.positions[b * a.ps[0] + t * a.ps[1]];
  pos = pos < 0 ? pos + a.n_ctx : pos;
  char* xrow = static_cast<char*>(a.x) + (int64_t)row * ln.n * 2;
  char* yrow = static_cast<char*>(ln.y) + (int64_t)row * ln.n * 2;
  auto store_x = [&](int c, u32x4 w) { *reinterpret_cast<u32x4*>(xrow + c * 16) = w; };
  auto store_y = [&](int c, u32x4 w) { *reinterpret_cast<u32x4*>(yrow + c * 16) = w; };
  if (tok < 0 || tok >= a.n_vocab || pos < 0 || pos >= a.n_ctx) {
    const u32x4 nan = {0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu};
    for (int c = lane; c < ln.n / 8; c += 64) {
      store_x(c, nan);
      store_y(c, nan);
    }
    return;
  }
  ln.x = static_cast<char*>(ln.x) + tok * ln.x_stride * 2;
  ln.delta = static_cast<const char*>(ln.delta) + pos * ln.d_stride * 2;
  LnRow<T, NC, 0> r;
  r.load(ln, 0, lane);
  r.finish(ln, lane, store_x, store_y);
}

// lens[l, slot of b] = the length gathered at the start + sq: repeated slots store the same value,
// as torch's indexed add does.
__global__ __launch_bounds__(256) void step_end_kernel(StepArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int b = i % a.B, l = i / a.B;
  if (l >= a.n_layers) return;
  int64_t s = a.slots ? a.slots[b] : b;
  s = s < 0 ? s + a.n_slots : s;
  if (s >= 0 && s < a.n_slots) a.lens[(int64_t)l * a.n_slots + s] = a.seqlens[(int64_t)l * a.B + b] + a.sq;
}

// ---- masked greedy sampling --------------------------------------------------------------
// argmax order of torch.argmax: NaN above every number (the first NaN wins), otherwise the
// larger value, ties to the lower index.
__device__ __forceinline__ bool argmax_beats(float v, int i, float b, int bi) {
  const bool vn = v != v, bn = b != b;
  if (vn != bn) return vn;
  if (vn) return i < bi;
  return v > b || (v == b && i < bi);
}

// Bound: the row's bytes through one CU (2 or 4 B of logits plus 2 mask bytes per token) and the
// latency of getting them. A workgroup (1024 threads, for short rows 256) takes a row, each thread 8 tokens
// at a time with whole-word loads (logits 16 / 32 bytes, each mask 8 bytes; rows start at any element, so
// the loads are unaligned), kArgmaxBatch of them requested before the first is used: a 51866-token
// row is one round of requests. The 256-thread form before it loaded one token and two mask bytes
// at a time. 52 rows x 51866 bf16 with both masks: 81 -> 12.3 us (kernel), 131 -> 11.9 us a call.
constexpr int kArgmaxVec = 8;    // tokens per load
constexpr int kArgmaxBatch = 7;  // loads in flight per thread: 57344 tokens per round of 1024 threads

template <typename T, int kArgmaxThreads>
__global__ __launch_bounds__(kArgmaxThreads) void masked_argmax_kernel(ArgmaxArgs a) {
  constexpr int kWords = kArgmaxVec * ElemBytes<T>::value / 4;
  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const char* lr = static_cast<const char*>(a.logits) + (int64_t)row * a.l_stride * ElemBytes<T>::value;
  const uint8_t* bm = a.blocked ? a.blocked + (int64_t)row * a.m_stride : nullptr;
  const uint8_t* pm = a.penalty ? a.penalty + (int64_t)row * a.p_stride : nullptr;
  // -65504 in the logits' type, as the additive mask holds it (decoding.py:1736-1738)
  const float neg = Elem<T>::round(-65504.f);
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  auto take = [&](float v, uint32_t blocked, uint32_t penalised, int i) {
    v = Elem<T>::round(v + (blocked ? neg : 0.f));  // logits + additive_mask
    if (penalised) v = Elem<T>::round(v > 0.f ? v / 1.2f : v * 1.2f);
    // argmax_beats for an index above best_i: larger, or the first NaN
    if (!(v <= best) && best == best) {
      best = v;
      best_i = i;
    }
  };

  const int n_vec = a.V / kArgmaxVec;
  for (int c0 = tid; c0 < n_vec; c0 += kArgmaxBatch * kArgmaxThreads) {
    uint32_t w[kArgmaxBatch][kWords];
    u32x2 mb[kArgmaxBatch], mp[kArgmaxBatch];
#pragma unroll
    for (int u = 0; u < kArgmaxBatch; ++u) {
      const int c = c0 + u * kArgmaxThreads;
      mb[u] = mp[u] = u32x2{0, 0};
      if (c < n_vec) {
        __builtin_memcpy(w[u], lr + (int64_t)c * kArgmaxVec * ElemBytes<T>::value, sizeof(w[u]));
        if (bm) __builtin_memcpy(&mb[u], bm + (int64_t)c * kArgmaxVec, 8);
        if (pm) __builtin_memcpy(&mp[u], pm + (int64_t)c * kArgmaxVec, 8);
      }
    }
#pragma unroll
    for (int u = 0; u < kArgmaxBatch; ++u) {
      const int c = c0 + u * kArgmaxThreads;
      if (c < n_vec) {
#pragma unroll
        for (int e = 0; e < kArgmaxVec; ++e) {
          const uint32_t byte = 0xffu << (8 * (e & 3));
          take(Elem<T>::word(w[u], e), mb[u][e >> 2] & byte, mp[u][e >> 2] & byte, c * kArgmaxVec + e);
        }
      }
    }
  }
  const int it = n_vec * kArgmaxVec + tid;  // the last V % 8 tokens, one per thread
  if (it < a.V) take(Elem<T>::load1(lr, it), bm ? bm[it] : 0, pm ? pm[it] : 0, it);

  // workgroup argmax in the same order
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float ob = __shfl_xor(best, o);
    const int oi = __shfl_xor(best_i, o);
    if (argmax_beats(ob, oi, best, best_i)) {
      best = ob;
      best_i = oi;
    }
  }
  constexpr int kWaves = kArgmaxThreads / 64;
  __shared__ float sb[kWaves];
  __shared__ int si[kWaves];
  if ((tid & 63) == 0) {
    sb[tid >> 6] = best;
    si[tid >> 6] = best_i;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kWaves; ++w)
      if (argmax_beats(sb[w], si[w], best, best_i)) {
        best = sb[w];
        best_i = si[w];
      }
    a.out[row] = best_i == 0x7fffffff ? 0 : best_i;
  }
}

}  // namespace

// One row per workgroup up to here: a workgroup's rows are fetched by one CU, and four of them (18 KB
// each with four partials) take longer than one. 52 rows of 1280 behind 2 / 4 partials 3.59 / 3.96 ->
// 3.17 / 3.44 us, 1024 rows 5.64 / 7.01 -> 5.22 / 6.90, 2048 rows 7.8 / 10.8 either way.
constexpr int64_t kLnSpreadRows = 1024;
hipError_t launch_add_layernorm(int dtype, const AddLnArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  const unsigned per_wg = a.rows <= kLnSpreadRows ? 1 : 4;
  const dim3 grid((unsigned)((a.rows + per_wg - 1) / per_wg)), block(64 * per_wg);
  const int nc = (a.n + 511) / 512;
  const int np = a.dpart ? a.n_part : 0;
  // the partials form keeps 2 NP fp32 quads per chunk in registers: n <= 1536 (NC <= 3)
  if ((np != 0 && np != 2 && np != 4) || (np != 0 && nc > 3)) return hipErrorInvalidValue;
#define WDRZ_LN3(NC, NP)                                                                                 \
  if (dtype == 2) hipLaunchKernelGGL((add_layernorm_kernel<Bf16, NC, NP>), grid, block, 0, stream, a); \
  else hipLaunchKernelGGL((add_layernorm_kernel<F16, NC, NP>), grid, block, 0, stream, a);
#define WDRZ_LNP(NC)     \
  case NC:               \
    if (np == 0) {       \
      WDRZ_LN3(NC, 0)    \
    } else if (np == 2) { \
      WDRZ_LN3(NC, 2)    \
    } else {             \
      WDRZ_LN3(NC, 4)    \
    }                    \
    break;
#define WDRZ_LN(NC)   \
  case NC:            \
    WDRZ_LN3(NC, 0)   \
    break;
  switch (nc) {
    WDRZ_LNP(1) WDRZ_LNP(2) WDRZ_LNP(3) WDRZ_LN(4) WDRZ_LN(5) WDRZ_LN(6) WDRZ_LN(7) WDRZ_LN(8)
    default:
      return hipErrorInvalidValue;
  }
#undef WDRZ_LN
#undef WDRZ_LNP
#undef WDRZ_LN3
  return hipGetLastError();
}

hipError_t launch_step_begin(int dtype, const StepArgs& a, const AddLnArgs& ln, hipStream_t stream) {
  const int64_t meta = (int64_t)(a.n_layers + 1) * a.B;
  const dim3 grid((unsigned)((a.B * a.sq + 3) / 4 + (meta + 255) / 256));
#define WDRZ_SB(NC)                                                                                       \
  case NC:                                                                                                \
    if (dtype == 2) hipLaunchKernelGGL((step_begin_kernel<Bf16, NC>), grid, dim3(256), 0, stream, a, ln); \
    else hipLaunchKernelGGL((step_begin_kernel<F16, NC>), grid, dim3(256), 0, stream, a, ln);             \
    break;
  switch ((ln.n + 511) / 512) {
    WDRZ_SB(1) WDRZ_SB(2) WDRZ_SB(3) WDRZ_SB(4)
    default:
      return hipErrorInvalidValue;
  }
#undef WDRZ_SB
  return hipGetLastError();
}

hipError_t launch_step_end(const StepArgs& a, hipStream_t stream) {
  const int64_t n = (int64_t)a.n_layers * a.B;
  hipLaunchKernelGGL(step_end_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

template <typename T>
static void launch_argmax_t(const ArgmaxArgs& a, hipStream_t stream) {
  // 256 threads where 1024 mostly launch and reduce idle lanes: rows of two loads a thread, and more rows
  // than two full workgroups a CU while one round of 256 threads' loads holds a row. Both masks, bf16, us,
  // 1024 / 256 threads: 52 rows of 1000 5.1 / 3.9, of 4000 5.4 / 4.7; 600 rows of 1000 9.6 / 4.6, of 14000
  // 17.4 / 14.5; 2000 rows of 8000 32.6 / 17.8.
  const dim3 grid((unsigned)a.rows);
  if (a.V <= 4096 || (a.rows > 512 && a.V <= 256 * kArgmaxVec * kArgmaxBatch))
    hipLaunchKernelGGL((masked_argmax_kernel<T, 256>), grid, dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((masked_argmax_kernel<T, 1024>), grid, dim3(1024), 0, stream, a);
}

hipError_t launch_masked_argmax(int dtype, const ArgmaxArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  if (dtype == 2) launch_argmax_t<Bf16>(a, stream);
  else if (dtype == 1) launch_argmax_t<F16>(a, stream);
  else launch_argmax_t<F32>(a, stream);
  return hipGetLastError();
}

}  // namespace wdrz
