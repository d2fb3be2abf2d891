// attn_dense_f32.hip — dense attention in fp32 on the matrix cores (gfx950).
//
// Replaces F.scaled_dot_product_attention at reference src/whisperdrz/model.py:288-296 when the
// model runs in fp32 (the reference's CPU-runnable configuration: one encoder layer B=1 H=20
// L=1500 D=64, and the uncached decoder with a top-left causal mask). O = softmax(scale Q K^T) V
// per (b, h), online softmax in the log2 domain, fp32 results.
//
// Products on the bf16 matrix cores, exactly split (split_tile): an fp32 operand of magnitude 2^-110
// or more is the sum of three bf16 values, x = x0 + x1 + x2 (8 + 8 + 8 bits of the 24-bit significand,
// each rounded to nearest), and x y is taken as x0 y0 + x0 y1 + x1 y0 + x1 y1 + x0 y2 + x2 y0,
// accumulated in fp32; what is left out (x1 y2, x2 y1, x2 y2) is up to about 2^-24 of |x y|, one fp32
// unit roundoff. 48 v_mfma_f32_32x32x16_bf16 of 32 cycles then do the work of 64
// v_mfma_f32_32x32x2_f32 of 64 cycles per 32 x 32 step, and, unlike beside those, the softmax's VALU
// instructions issue meanwhile. Measured, one encoder layer (B=1 H=20 L=1500): 110.6 -> 70.4 us, B=16
// 1641 -> 1081; causal 448 x 448, B=16: 176 -> 109; error against 64 bits 5.3e-7 -> 4.5e-7. Bound now,
// by counters: VALU issue (softmax, and the split of K, V and P, 11 instructions a pair) takes 56% and the
// MFMAs (24 for S^T, 24 for O^T a step) 47% of the SIMDs' busy cycles, 20% both at once.
// Where the split falls short, the workgroup repeats its queries on the fp32 matrix cores (f32_tile),
// whose result stands. Infinities and NaN do not survive it (inf - inf): they give NaN output. Below
// 2^-110 the third part is below the smallest bf16 value and up to 2^-134 is lost: in V that shows
// as an output below kTinyOut (zero among them, which values below 2^-134 alone give), in a query or
// key only beside a huge partner, which queries of magnitude 2^-90 to 2^90 (or zero) rule out. (What
// remains is a probability below 2^-110 times a value 2^110 above the others.)
//
// f32_tile: both products on v_mfma_f32_32x32x2_f32 (32x32 output, K = 2 per instruction, lane halves
// h = lane / 32 supplying the two K slots):
//   * S^T = K Q^T per 32-key step: 32 MFMAs over the 64 head dims. The K slot of lane half h at
//     instruction kk is head dim 32h + kk, for K (A operand, row = key lane % 32) and Q (B
//     operand, column = query lane % 32) alike, so each lane reads 32 contiguous floats of its
//     K row (eight 16-byte LDS reads) and keeps its 32 Q floats in registers. Two accumulator
//     chains (even / odd kk) keep the matrix pipe busy.
//   * O^T += V^T P^T: 16 MFMAs per 32 output dims. Accumulator i = 4j + r of lane l holds key
//     8j + 4h + r of S^T, so at instruction kk = i both operands use that key in K slot h: P is
//     the accumulator itself (no shuffles) and V^T is one 4-byte LDS read of row 8j + 4h + r.
// Either way a 512-thread workgroup holds four 32-query groups, each served by two wavefronts on
// the same SIMD that take alternate 32-key steps (so every SIMD has two wavefronts to cover each
// other's stalls) and merge their (m, l, O) through LDS at the end. 64-key K and V stages go through
// registers into three LDS buffers (two stages ahead), one barrier per stage; each wavefront issues
// its next step's S^T before its own softmax, and the output is rescaled only when a row max grows.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "wdrz_common.h"
#include "wdrz_launch.h"

namespace wdrz {
namespace {

constexpr int kF32Groups = 4;                 // 32-query groups per workgroup
constexpr int kF32Waves = 2 * kF32Groups;     // two key halves per group
constexpr int kF32Threads = kF32Waves * 64;
constexpr int kF32BM = 32 * kF32Groups;  // queries per workgroup
constexpr int kF32BS = 32;               // keys per step (one wavefront)
constexpr int kF32Stage = 2 * kF32BS;    // keys per LDS stage (both halves)
constexpr int kF32Pitch = kHeadDim + 4;  // LDS row pitch in floats (16-byte pad: conflict-free b128 reads)

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Both tile functions' place in the launch.
struct F32Tile {
  int lane, qg, kh, hl, l32;  // qg: query group; kh: key half, steps 2u + kh of each 64-key stage u
  const float *Q, *K, *V;
  float* O;
  int q_wave0, q_me;  // q_me: this lane's query (may be >= Lq: computed, not stored)
  int k_lim_w;        // keys this wavefront needs (top-left causal: query i sees keys 0..i)
  int n_units;        // 64-key stages the workgroup needs
};
template <bool CAUSAL>
__device__ __forceinline__ F32Tile f32_place(const DenseArgs& a) {
  F32Tile p;
  p.lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  p.qg = wave % kF32Groups;
  p.kh = wave / kF32Groups;
  p.hl = p.lane >> 5;
  p.l32 = p.lane & 31;
  const int n_qblk = (a.Lq + kF32BM - 1) / kF32BM;
  const int tile_id = remap_xcd(blockIdx.x, gridDim.x);
  const int qblk = tile_id % n_qblk;
  const int bh = tile_id / n_qblk;
  const int b = bh / a.H, h = bh % a.H;
  p.Q = static_cast<const float*>(a.q) + b * a.qs[0] + h * a.qs[1];
  p.K = static_cast<const float*>(a.k) + b * a.ks[0] + h * a.ks[1];
  p.V = static_cast<const float*>(a.v) + b * a.vs[0] + h * a.vs[1];
  p.O = static_cast<float*>(a.o) + b * a.os[0] + h * a.os[1];
  const int q_blk0 = qblk * kF32BM;
  p.q_wave0 = q_blk0 + p.qg * 32;
  p.q_me = p.q_wave0 + p.l32;
  const int k_lim = CAUSAL ? min(a.Lk, q_blk0 + kF32BM) : a.Lk;
  p.k_lim_w = CAUSAL ? min(a.Lk, p.q_wave0 + 32) : a.Lk;
  p.n_units = (k_lim + kF32Stage - 1) / kF32Stage;
  return p;
}

// Online softmax of step st on sc (P written back into sc).
template <bool CAUSAL>
__device__ __forceinline__ void f32_softmax(const DenseArgs& a, const F32Tile& p, int st, f32x16& sc, float& m_run,
                                            float& l_run, f32x16 (&acc_o)[2]) {
  const int k0 = st * kF32BS;
  if (k0 + kF32BS > a.Lk || (CAUSAL && k0 + kF32BS - 1 > p.q_wave0)) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int key = k0 + 8 * (x >> 2) + 4 * p.hl + (x & 3);
      if (key >= a.Lk || (CAUSAL && key > p.q_me)) sc[x] = -INFINITY;
    }
  }
  float mx = sc[0];
#pragma unroll
  for (int x = 1; x < 16; ++x) mx = fmaxf(mx, sc[x]);
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  if (__any(mx > m_run)) {  // some row's max grows: rescale what was accumulated
    const float m_new = fmaxf(m_run, mx);
    const float alpha = fast_exp2(m_run - m_new);  // 0 on the first step (m_run = -inf)
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      acc_o[0][x] *= alpha;
      acc_o[1][x] *= alpha;
    }
  }
  float psum = 0.f;
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    sc[x] = fast_exp2(sc[x] - m_run);
    psum += sc[x];
  }
  l_run += psum;
}

// Outputs below this (or NaN) and scaled queries beyond these are not left to the split operands.
constexpr float kTinyOut = 0x1p-100f, kTinyQ = 0x1p-90f, kHugeQ = 0x1p90f;

// Merges the two key halves of each query group through LDS (smem, free by now), normalises and
// stores; true in a lane that stored a NaN or a value below kTinyOut.
__device__ __forceinline__ bool f32_merge_store(const DenseArgs& a, const F32Tile& p, float* smem, float m_run,
                                                float l_run, const f32x16 (&acc_o)[2]) {
  const int lane = p.lane;
  float* mg = smem + p.qg * (34 * 64);  // [34][64]: acc_o (32), m, l per lane
  if (p.kh == 1) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      mg[x * 64 + lane] = acc_o[0][x];
      mg[(16 + x) * 64 + lane] = acc_o[1][x];
    }
    mg[32 * 64 + lane] = m_run;
    mg[33 * 64 + lane] = l_run;
  }
  __syncthreads();
  if (p.kh == 1 || p.q_me >= a.Lq) return false;
  const float m1 = mg[32 * 64 + lane];
  const float m = fmaxf(m_run, m1);  // finite: half 0 always sees key 0
  const float a0 = fast_exp2(m_run - m), a1 = fast_exp2(m1 - m);
  const float l_me = l_run * a0 + mg[33 * 64 + lane] * a1;
  const float inv = 1.f / (l_me + __shfl_xor(l_me, 32));
  bool tiny = false;
  // lane holds dims 32 db + 8j + 4h + r (r = 0..3) of its query
  float* orow = p.O + (int64_t)p.q_me * a.os[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 w;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = 4 * j + r;
        w[r] = (acc_o[db][x] * a0 + mg[(16 * db + x) * 64 + lane] * a1) * inv;
        tiny = tiny || !(fabsf(w[r]) >= kTinyOut);
      }
      store16(orow + 32 * db + 8 * j + 4 * p.hl, __builtin_bit_cast(u32x4, w));
    }
  return tiny;
}

// ---- the tile on the fp32 matrix cores -------------------------------------------------------------
template <bool CAUSAL>
__device__ void f32_tile(const DenseArgs& a, float* smem) {
  float (*sK)[kF32Stage * kF32Pitch] = reinterpret_cast<float (*)[kF32Stage * kF32Pitch]>(smem);
  float (*sV)[kF32Stage * kF32Pitch] = sK + 3;
  const F32Tile p = f32_place<CAUSAL>(a);
  const int tid = threadIdx.x, kh = p.kh, hl = p.hl, l32 = p.l32;
  const float *K = p.K, *V = p.V;
  const int n_units = p.n_units;

  // Q: 32 floats (head dims 32h .. 32h + 31) of this lane's query, pre-scaled by c.
  float qreg[32];
  {
    const float* qp = p.Q + (int64_t)min(p.q_me, a.Lq - 1) * a.qs[2] + 32 * hl;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const f32x4 v = __builtin_bit_cast(f32x4, load16(qp + 4 * i));
#pragma unroll
      for (int e = 0; e < 4; ++e) qreg[4 * i + e] = v[e] * a.c;
    }
  }

  // Tile staging: thread t moves 16-byte pieces t and t + 512 of the 64 x 64 K and V tiles.
  u32x4 rk[2], rv[2];
  auto gload = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int piece = tid + i * kF32Threads;
      const int key = min(st * kF32Stage + (piece >> 4), a.Lk - 1);
      const int col = (piece & 15) * 4;
      rk[i] = load16(K + (int64_t)key * a.ks[2] + col);
      rv[i] = load16(V + (int64_t)key * a.vs[2] + col);
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int piece = tid + i * kF32Threads;
      const int off = (piece >> 4) * kF32Pitch + (piece & 15) * 4;
      *reinterpret_cast<u32x4*>(&sK[buf][off]) = rk[i];
      *reinterpret_cast<u32x4*>(&sV[buf][off]) = rv[i];
    }
  };

  f32x16 acc_o[2];  // [db]: O^T rows d = 32 db + 8j + 4h + r, column = query
#pragma unroll
  for (int x = 0; x < 16; ++x) acc_o[0][x] = acc_o[1][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // S^T of step st (K tile in buffer buf), two accumulator chains summed at the end
  auto scores = [&](int buf, f32x16& out) __attribute__((always_inline)) {
    f32x16 sa, sb;
#pragma unroll
    for (int x = 0; x < 16; ++x) sa[x] = sb[x] = 0.f;
    const float* kr = &sK[buf][(kh * kF32BS + l32) * kF32Pitch + 32 * hl];
#pragma unroll
    for (int kq = 0; kq < 8; ++kq) {
      const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + 4 * kq);
      sa = mfma_f32(kv[0], qreg[4 * kq + 0], sa);
      sb = mfma_f32(kv[1], qreg[4 * kq + 1], sb);
      sa = mfma_f32(kv[2], qreg[4 * kq + 2], sa);
      sb = mfma_f32(kv[3], qreg[4 * kq + 3], sb);
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) out[x] = sa[x] + sb[x];
  };
  // O^T += V^T P^T: instruction i uses key 8(i>>2) + 4h + (i&3) in K slot h
  auto pv = [&](int buf, const f32x16& pr) __attribute__((always_inline)) {
    const float* vr = &sV[buf][(kh * kF32BS + 4 * hl) * kF32Pitch + l32];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float* row = vr + (8 * (i >> 2) + (i & 3)) * kF32Pitch;
      acc_o[0] = mfma_f32(row[0], pr[i], acc_o[0]);
      acc_o[1] = mfma_f32(row[32], pr[i], acc_o[1]);
    }
  };

  // Stages of 64 keys (the two halves' steps) go two stages ahead into three buffers: at the top
  // of stage u, stages u and u+1 are visible, so S of the wavefront's step in stage u+1 is
  // issued before its softmax of stage u and the matrix pipe has work while the softmax runs.
  gload(0);
  lstore(0);
  if (n_units > 1) {
    gload(1);
    lstore(1);
  }
  if (n_units > 2) gload(2);
  __syncthreads();
  auto live = [&](int u) { return (2 * u + kh) * kF32BS < p.k_lim_w; };  // causal: keys end earlier
  f32x16 s_cur, s_nxt;
  if (live(0)) scores(0, s_cur);
  auto unit = [&](int u, f32x16& cur, f32x16& nxt) __attribute__((always_inline)) {
    if (live(u)) {
      if (u + 1 < n_units && live(u + 1)) scores((u + 1) % 3, nxt);
      f32_softmax<CAUSAL>(a, p, 2 * u + kh, cur, m_run, l_run, acc_o);
      pv(u % 3, cur);
    }
    // Buffer (u+2)%3 last held stage u-1, whose reads (K in stage u-2, V in stage u-1) came
    // before the previous barrier.
    if (u + 2 < n_units) {
      lstore((u + 2) % 3);
      if (u + 3 < n_units) gload(u + 3);
    }
    __syncthreads();
  };
  int u = 0;
  for (; u + 1 < n_units; u += 2) {
    unit(u, s_cur, s_nxt);
    unit(u + 1, s_nxt, s_cur);
  }
  if (u < n_units) unit(u, s_cur, s_nxt);

  f32_merge_store(a, p, smem, m_run, l_run, acc_o);
}

// ---- the tile on the bf16 matrix cores, operands split in three -----------------------------------
// One 64-key stage in LDS: three bf16 planes of K rows [key][dim] and of V transposed [dim][key].
// The pitches keep the 16-byte operand reads of K and the 8-byte ones of V^T conflict-free.
constexpr int kSpKPitch = kHeadDim + 8;
constexpr int kSpVPitch = kF32Stage + 4;
struct SplitStage {
  uint16_t k[3][kF32Stage][kSpKPitch];
  uint16_t v[3][kHeadDim][kSpVPitch];
};

// x and y as three bf16 pairs (packed x | y << 16) whose sums are x and y exactly.
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&w)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    w[i] = pack_bf16x2(x, y);
    x -= bf16_lo(w[i]);
    y -= bf16_hi(w[i]);
  }
}

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Returns true in lanes that saw operands or results which the split does not serve.
template <bool CAUSAL>
__device__ __forceinline__ bool split_tile(const DenseArgs& a, SplitStage* stage) {
  const F32Tile p = f32_place<CAUSAL>(a);
  const int tid = threadIdx.x, kh = p.kh, hl = p.hl, l32 = p.l32;
  const float *K = p.K, *V = p.V;
  const int n_units = p.n_units;

  // Q, pre-scaled by c: plane i, instruction kk holds head dims 16 kk + 8h .. + 7 of this lane's query
  u32x4 qop[3][4];
  float q_hi = 0.f;     // the largest |q| and, as bits 2 |q| - 1, the smallest that is not zero
  uint32_t q_lo = ~0u;
  {
    const float* qp = p.Q + (int64_t)min(p.q_me, a.Lq - 1) * a.qs[2] + 8 * hl;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f32x4 v = __builtin_bit_cast(f32x4, load16(qp + 16 * kk + 4 * j));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          q_hi = fmaxf(q_hi, fabsf(v[e]));
          q_lo = min(q_lo, (__float_as_uint(v[e]) << 1) - 1);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          uint32_t w[3];
          split_pair(v[2 * e] * a.c, v[2 * e + 1] * a.c, w);
#pragma unroll
          for (int i = 0; i < 3; ++i) qop[i][kk][2 * j + e] = w[i];
        }
      }
  }
  // (all zero: q_lo's float is NaN)
  const bool q_range = q_hi * fabsf(a.c) > kHugeQ || __uint_as_float(q_lo >> 1) * fabsf(a.c) < kTinyQ;

  // Staging: thread t moves dims 4 (t % 16) .. + 3 of the keys 2 (t / 16) and + 1 of a stage, so that
  // V^T's key pairs are packed in one thread.
  const int col = (tid & 15) * 4, kp = (tid >> 4) * 2;
  f32x4 rk[2], rv[2];
  auto gload = [&](int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = min(st * kF32Stage + kp + i, a.Lk - 1);
      rk[i] = __builtin_bit_cast(f32x4, load16(K + (int64_t)key * a.ks[2] + col));
      rv[i] = __builtin_bit_cast(f32x4, load16(V + (int64_t)key * a.vs[2] + col));
    }
  };
  auto lstore = [&](int buf) __attribute__((always_inline)) {
    SplitStage& s = stage[buf];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t lo[3], hi[3];
      split_pair(rk[i][0], rk[i][1], lo);
      split_pair(rk[i][2], rk[i][3], hi);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<u32x2*>(&s.k[pl][kp + i][col]) = u32x2{lo[pl], hi[pl]};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t w[3];
      split_pair(rv[0][e], rv[1][e], w);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<uint32_t*>(&s.v[pl][col + e][kp]) = w[pl];
    }
  };

  f32x16 acc_o[2];  // [db]: O^T rows d = 32 db + 8j + 4h + r, column = query
#pragma unroll
  for (int x = 0; x < 16; ++x) acc_o[0][x] = acc_o[1][x] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // S^T of this wavefront's step in buffer buf: two chains, each from its smallest terms up
  auto scores = [&](int buf, f32x16& out) __attribute__((always_inline)) {
    f32x16 sa, sb;
#pragma unroll
    for (int x = 0; x < 16; ++x) sa[x] = sb[x] = 0.f;
    const SplitStage& s = stage[buf];
    const int key = kh * kF32BS + l32;
    u32x4 k[3][4];
#pragma unroll
    for (int pl = 2; pl >= 0; --pl)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) k[pl][kk] = *reinterpret_cast<const u32x4*>(&s.k[pl][key][16 * kk + 8 * hl]);
#pragma unroll
    for (int pl = 2; pl >= 0; --pl)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        sa = mfma_bf16(k[pl][kk], qop[0][kk], sa);                                    // K2 Q0, K1 Q0, K0 Q0
        sb = mfma_bf16(k[pl == 1 ? 1 : 0][kk], qop[pl == 0 ? 1 : pl][kk], sb);        // K0 Q2, K1 Q1, K0 Q1
      }
#pragma unroll
    for (int x = 0; x < 16; ++x) out[x] = sa[x] + sb[x];
  };
  // O^T += V^T P^T: instruction kk takes accumulators 8 kk .. + 7 as they are, i.e. in the lane half's K
  // slots the keys 16 kk + 4h .. + 3 and 16 kk + 8 + 4h .. + 3, and V^T in that order
  auto pv = [&](int buf, const f32x16& pr) __attribute__((always_inline)) {
    const SplitStage& s = stage[buf];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      u32x4 pop[3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t w[3];
        split_pair(pr[8 * kk + 2 * j], pr[8 * kk + 2 * j + 1], w);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) pop[pl][j] = w[pl];
      }
      u32x4 v[2][3];
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
          const uint16_t* row = &s.v[pl][32 * db + l32][kh * kF32BS + 16 * kk + 4 * hl];
          const u32x2 lo = *reinterpret_cast<const u32x2*>(row), hi = *reinterpret_cast<const u32x2*>(row + 8);
          v[db][pl] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
#pragma unroll
      for (int t = 0; t < 6; ++t) {  // smallest terms first
        constexpr int kV[6] = {2, 0, 1, 1, 0, 0}, kP[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int db = 0; db < 2; ++db) acc_o[db] = mfma_bf16(v[db][kV[t]], pop[kP[t]], acc_o[db]);
      }
    }
  };

  // the same stage schedule as f32_tile
  gload(0);
  lstore(0);
  if (n_units > 1) {
    gload(1);
    lstore(1);
  }
  if (n_units > 2) gload(2);
  __syncthreads();
  auto live = [&](int u) { return (2 * u + kh) * kF32BS < p.k_lim_w; };  // causal: keys end earlier
  f32x16 s_cur, s_nxt;
  if (live(0)) scores(0, s_cur);
  auto unit = [&](int u, f32x16& cur, f32x16& nxt) __attribute__((always_inline)) {
    // The two wavefronts of a SIMD split and store their share of stage u + 2 at opposite ends of the
    // stage, so that one's VALU work runs beside the other's MFMAs (with the priority below, 74.3 ->
    // 70.4 us a layer). The buffer last held stage u - 1, whose reads came before the last barrier.
    if (kh == 1 && u + 2 < n_units) {
      lstore((u + 2) % 3);
      if (u + 3 < n_units) gload(u + 3);
    }
    if (live(u)) {
      __builtin_amdgcn_s_setprio(1);
      if (u + 1 < n_units && live(u + 1)) scores((u + 1) % 3, nxt);
      __builtin_amdgcn_s_setprio(0);
      f32_softmax<CAUSAL>(a, p, 2 * u + kh, cur, m_run, l_run, acc_o);
      pv(u % 3, cur);
    }
    if (kh == 0 && u + 2 < n_units) {
      lstore((u + 2) % 3);
      if (u + 3 < n_units) gload(u + 3);
    }
    __syncthreads();
  };
  int u = 0;
  for (; u + 1 < n_units; u += 2) {
    unit(u, s_cur, s_nxt);
    unit(u + 1, s_nxt, s_cur);
  }
  if (u < n_units) unit(u, s_cur, s_nxt);
  return f32_merge_store(a, p, reinterpret_cast<float*>(stage), m_run, l_run, acc_o) || q_range;
}

template <bool CAUSAL>
__global__ __launch_bounds__(kF32Threads) void dense_f32_kernel(DenseArgs a) {
  __shared__ __align__(16) SplitStage stage[3];
  static_assert(sizeof(stage) >= 6 * sizeof(float) * kF32Stage * kF32Pitch, "f32_tile's stages");
  __shared__ int again;
  if (threadIdx.x == 0) again = 0;
  // (many barriers lie between this store and the ones below)
  if (split_tile<CAUSAL>(a, stage)) again = 1;
  __syncthreads();
  if (again) f32_tile<CAUSAL>(a, reinterpret_cast<float*>(stage));
}

}  // namespace

hipError_t launch_dense_f32(const DenseArgs& a, hipStream_t stream) {
  const int n_qblk = (a.Lq + kF32BM - 1) / kF32BM;
  const int64_t n = (int64_t)a.B * a.H * n_qblk;
  if (n <= 0) return hipSuccess;
  if (n > 0x7fffffff) return hipErrorInvalidValue;
  if (a.causal)
    hipLaunchKernelGGL((dense_f32_kernel<true>), dim3((unsigned)n), dim3(kF32Threads), 0, stream, a);
  else
    hipLaunchKernelGGL((dense_f32_kernel<false>), dim3((unsigned)n), dim3(kF32Threads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace wdrz
