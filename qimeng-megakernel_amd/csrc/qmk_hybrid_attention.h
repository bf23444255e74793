// Prefill attention of bf16 portions.
#pragma once

#include "qmk_hybrid_gemm.h"

namespace qmk {
namespace hybrid {

// Keys of an attention: key j of key head h at at[j * pitch + h * head]; heads_per query heads share a key head.
template <class T>
struct Keys {
  const T* at;
  int pitch, head, heads_per;
};

__device__ const uint32_t kZeroUnit[4] = {0u, 0u, 0u, 0u};

// Maximum over the four lanes of a query, 16 apart: rows, then halves, exchanged between two registers that hold the same.
__device__ __forceinline__ float max_of_quarters(float v) {
  const uint32_t a = __float_as_uint(v);
  const auto rows = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const uint32_t b = __float_as_uint(fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1])));
  const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
}

// Windowed causal attention over expanded keys: 64 queries of one head a workgroup (16 a wave), KEYS keys a stage, QT 32-column steps of a query,
// at most VT 16-row tiles of a value.  Scores are computed transposed (keys x queries), so a lane holds eight weights of ONE query in exactly the shape
// the value product's second operand wants.  A query takes its keys 32 at a time in their order, as bf16 portions have to (qmk_hybrid_tiles.h);
// 32 keys that no query of a wave sees are left out, which changes nothing but that a value among them that is not finite stays out of the sums (0 x inf).
//
// What bounds it is the chain of 32 keys in a wave (fragments, scores, maximum over the lanes, weights, values; about 700 instructions' time), with two waves a
// SIMD at 2048 queries of 16 heads.  So both halves of 64 keys take their scores together, all fragments are asked for at once (asked for
// where they are used, every pair is waited for: 1.5 times as long), stages go from memory to LDS without registers or branches, and weights
// are scaled down only where a maximum has moved.  us, through registers with 32 keys a step -> now: 2048 queries behind 2048 keys, 16 heads
// of 128 | 128 212 -> 90; 1531 queries of 192 | 128, window 1024, 72 -> 33; 43 behind 400 27.7 -> 15.  Stages of 32 keys 124, 42, 16.6; of 128, 179 (one workgroup a CU);
// 128 queries a workgroup, 32 a wave: 160, 60, 25; on eight waves 119, 42, 17.5.
//
// SHARED, for few workgroups: 16 queries a workgroup, its waves share a stage's work.  Each takes the scores of 16 of 64 keys, everybody the weights of all of them, and each
// a quarter of a value's tiles: the same sums in the same order, a third of the fragments to read (us, 43 queries of 192 | 128 behind 400, 16 heads: 16.2 -> 13.4; with three stages
// 13.9, so it is not the loads; three stages for 64 queries 18.7).
struct AttentionArgs {
  const u16* q;
  Keys<u16> keys;
  const u16 *rows, *v_t, *gate;
  QmkHybridLayer layer;
  int first, position, M, keys_cap;
  u16* out;
};
template <int QT, int VT, int KEYS, int STAGES, bool SHARED>
constexpr int kAttentionLds = STAGES * (KEYS * QT * 4 + VT * 2 * KEYS) + (SHARED ? KEYS * 16 / 4 : 0);
// Workgroup `block` of `blocks`.
template <int QT, int VT, int KEYS, int STAGES, bool SHARED>
__device__ __forceinline__ void attend_rows(const AttentionArgs& a, int block, int blocks, v4u* lds) {
  const u16 *q = a.q, *rows = a.rows, *v_t = a.v_t, *gate = a.gate;
  u16* out = a.out;
  const Keys<u16>& keys = a.keys;
  const QmkHybridLayer& l = a.layer;
  const int first = a.first, position = a.position, M = a.M, keys_cap = a.keys_cap;
  constexpr int kRowK = QT * 4, kRowV = KEYS / 8;      // units of 16 bytes
  constexpr int kUnitsK = KEYS * kRowK, kUnits = kUnitsK + VT * 16 * kRowV;
  constexpr int kLoadsK = kUnitsK / kPfThreads, kLoads = kUnits / kPfThreads, kAhead = STAGES - 1, kSubs = KEYS / 32;
  constexpr int kWaves = kPfThreads / 64, kQueries = SHARED ? 16 : 64, kTiles = SHARED ? VT / kWaves : VT;      // tiles of a value: of this wave
  static_assert(kLoadsK * kPfThreads == kUnitsK && kLoads * kPfThreads == kUnits, "every thread stages the same number of units");
  static_assert(!SHARED || (KEYS == kWaves * 16 && VT % kWaves == 0), "a wave has 16 keys and whole tiles");
  static_assert(kAttentionLds<QT, VT, KEYS, STAGES, SHARED> == STAGES * kUnits + (SHARED ? KEYS * 16 / 4 : 0), "its stages and shared scores");
  using Lds = __attribute__((address_space(3))) v4u;
  Lds* const buffers = (Lds*)lds;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, col = lane & 15;
  // The longest rows of keys first, and the workgroups of one key head on one XCD where there are eight of them, so that they share its keys.
  const int kv_heads = l.heads / keys.heads_per, order = block % l.heads, kv = order % kv_heads, head = kv * keys.heads_per + order / kv_heads;
  const int q0 = (blocks / l.heads - 1 - block / l.heads) * kQueries;
  const int dq = l.q_stride, width = l.rank + l.rot_dim;
  const int lo = max(first, position + q0 + 1 - l.window);      // the first key any of these queries sees
  const int hi = min(position + q0 + kQueries, position + M);          // behind the last one
  const int begin = first + ((lo - first) & ~31), count = (hi - begin + KEYS - 1) / KEYS;

  // Staging: a thread has fixed places in a stage, keys first; a row's units are exchanged by its number.
  auto exchange_v = [](int r) { return kRowV == 8 ? r & 7 : (r >> 1) & 3; };
  const u16* at[kLoads];
  long long at_row[kLoadsK];      // from one key to the next
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int u = (i < kLoadsK ? i : i - kLoadsK) * kPfThreads + tid;
    if (i < kLoadsK) {
      const int r = u / kRowK, c = ((u % kRowK) ^ (r & 7)) * 8;
      if (c < l.head_dim) {
        at_row[i] = keys.pitch;
        at[i] = keys.at + static_cast<size_t>(begin - first + r) * keys.pitch + kv * keys.head + c;
      } else if (rows != nullptr && c < l.head_dim + l.rot_dim) {
        at_row[i] = width;
        at[i] = rows + static_cast<size_t>(begin - first + r) * width + l.rank + c - l.head_dim;
      } else {      // columns behind the rotated part
        at_row[i] = 0;
        at[i] = reinterpret_cast<const u16*>(kZeroUnit);
      }
    } else {
      const int r = u / kRowV, c = ((u % kRowV) ^ exchange_v(r)) * 8;
      at[i] = v_t + static_cast<size_t>(kv * l.v_dim + min(r, l.v_dim - 1)) * keys_cap + begin - first + c;
    }
  }
  auto load = [&](const u16* from, int buf, int i) {
    const auto* src = (const __attribute__((address_space(1))) uint32_t*)from;
    auto* dst = (__attribute__((address_space(3))) uint32_t*)(buffers + buf * kUnits + i * kPfThreads + wave * 64);
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
  };
  auto issue = [&](int stage, int buf) {
    const int base = begin + stage * KEYS;
    if (base + KEYS <= hi) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        load(at[i], buf, i);
        at[i] += i < kLoadsK ? at_row[i < kLoadsK ? i : 0] * KEYS : KEYS;
      }
    } else {      // the last stage: keys behind the last one are that one again, values behind its 32 keys are theirs again; neither is used
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int u = (i < kLoadsK ? i : i - kLoadsK) * kPfThreads + tid;
        if (i < kLoadsK) load(at[i] - max(base + u / kRowK - (hi - 1), 0) * at_row[i < kLoadsK ? i : 0], buf, i);
        else load(at[i] - max(base - first + (((u % kRowV) ^ exchange_v(u / kRowV)) * 8 & ~31) - ((hi - 1 - first) & ~31), 0), buf, i);
      }
    }
  };
  const int own_q = SHARED ? 0 : wave * 16, own_tile = SHARED ? wave * kTiles : 0, m = q0 + own_q + col;
  Frag<u16> fq[QT];
#pragma unroll
  for (int s = 0; s < QT; ++s) {
    fq[s] = Frag<u16>{};
    if (s < dq / 32) fq[s] = load_frag(q + static_cast<size_t>(min(m, M - 1)) * l.heads * dq + head * dq + s * 32 + g * 8);
  }
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
    if (s < count) issue(s, s);
  f32x4 acc[kTiles] = {};
  float top = -INFINITY, sum = 0.f;
  const float scale = l.scale * kLog2e;
  const int first_pos = position + q0 + own_q, last_pos = first_pos + 15, window = l.window;      // this wave's queries
  // A stage of keys base .. base + KEYS - 1.  MASKED: some query does not see some of them.
  auto take = [&](auto masked, int base, const Lds* sk, const Lds* sv) {
    constexpr bool MASKED = decltype(masked)::value;
    Frag<u16> fv[kSubs][kTiles];
    f32x4 d[kSubs][2] = {};
    auto values = [&] {
#pragma unroll
      for (int sub = 0; sub < kSubs; ++sub)
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
          const int r = (own_tile + t) * 16 + col;
          fv[sub][t] = Frag<u16>{__builtin_bit_cast(bf16x8_t, sv[r * kRowV + ((sub * 4 + g) ^ exchange_v(r))])};
        }
    };
    auto key = [&](int r, int s) { return Frag<u16>{__builtin_bit_cast(bf16x8_t, sk[r * kRowK + ((s * 4 + g) ^ (r & 7))])}; };
    if constexpr (SHARED) {
      Lds* const scores = buffers + STAGES * kUnits;
      Frag<u16> fk[QT];
#pragma unroll
      for (int s = 0; s < QT; ++s) fk[s] = key(wave * 16 + col, s);
      values();
      f32x4 own = {};
#pragma unroll
      for (int s = 0; s < QT; ++s) own = mma(fk[s], fq[s], own);
      scores[wave * 64 + lane] = __builtin_bit_cast(v4u, own);
      wait_known<63>();      // (not for the next stage, as __syncthreads would; the scores are read before its barrier)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int sub = 0; sub < kSubs; ++sub)
#pragma unroll
        for (int t = 0; t < 2; ++t) d[sub][t] = __builtin_bit_cast(f32x4, scores[(sub * 2 + t) * 64 + lane]);
    } else {
      Frag<u16> fk[kSubs][2][QT];
#pragma unroll
      for (int s = 0; s < QT; ++s)
#pragma unroll
        for (int sub = 0; sub < kSubs; ++sub)
#pragma unroll
          for (int t = 0; t < 2; ++t) fk[sub][t][s] = key(sub * 32 + t * 16 + col, s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int sub = 0; sub < kSubs; ++sub)
#pragma unroll
        for (int s = 0; s < QT; ++s)
#pragma unroll
          for (int t = 0; t < 2; ++t) d[sub][t] = mma(fk[sub][t][s], fq[s], d[sub][t]);
      values();
    }
#pragma unroll
    for (int sub = 0; sub < kSubs; ++sub, base += 32) {
      if (MASKED && (base >= hi || base > last_pos || first_pos - (base + 31) >= window)) continue;      // 32 keys that no query of this wave sees
      float w[8], best = top, step_sum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = d[sub][j >> 2][j & 3] * scale;
      if constexpr (MASKED) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int dist = position + m - (base + (j >> 2) * 16 + g * 4 + (j & 3));
          if (dist < 0 || dist >= window) w[j] = -INFINITY;
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) best = fmaxf(best, w[j]);
      best = max_of_quarters(best);
      const float ref = best == -INFINITY ? 0.f : best;      // no key of this query yet
      const float shrink = exp2_fast(top - ref);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w[j] = exp2_fast(w[j] - ref);
        step_sum += w[j];
      }
      v4u pairs;
#pragma unroll
      for (int j = 0; j < 4; ++j) pairs[j] = f2bf2(w[2 * j], w[2 * j + 1]);
      const Frag<u16> fp{__builtin_bit_cast(bf16x8_t, pairs)};
      sum = sum * shrink + step_sum;
      top = best;
      if (!__all(shrink == 1.f)) {
#pragma unroll
        for (int t = 0; t < kTiles; ++t) acc[t] = acc[t] * shrink;
      }
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        Frag<u16> f = fv[sub][t];
        if (MASKED && base + 32 > hi) {      // whatever the buffer holds behind the last key must not enter a sum
          v4u bits = __builtin_bit_cast(v4u, f.v);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = base + (j >> 1) * 16 + g * 4 + (j & 1) * 2;
            bits[j] &= (key < hi ? 0xffffu : 0u) | (key + 1 < hi ? 0xffff0000u : 0u);
          }
          f = Frag<u16>{__builtin_bit_cast(bf16x8_t, bits)};
        }
        acc[t] = mma(f, fp, acc[t]);
      }
    }
  };
  int buf = 0;
  for (int stage = 0; stage < count; ++stage) {
    // This stage has landed; the barrier makes that true of every wave's part, and says that the buffer filled next is no longer read.
    if (stage + kAhead - 1 < count) wait_outstanding<(kAhead - 1) * kLoads>();
    else wait_outstanding<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (stage + kAhead < count) issue(stage + kAhead, buf == 0 ? STAGES - 1 : buf - 1);
    const int base = begin + stage * KEYS, behind = base + KEYS;
    const Lds *sk = buffers + buf * kUnits, *sv = sk + kUnitsK;
    if (behind - 1 <= first_pos && last_pos - base < window && behind <= hi) take(std::false_type{}, base, sk, sv);
    else if (base <= last_pos && first_pos - (behind - 1) < window) take(std::true_type{}, base, sk, sv);
    buf = buf + 1 == STAGES ? 0 : buf + 1;
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  if (m >= M) return;
  const float inv = 1.f / sum;
  const size_t o = static_cast<size_t>(m) * l.heads * l.v_dim + head * l.v_dim;
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const int at = (own_tile + t) * 16 + g * 4;
    if (at < l.v_dim) store4(out + o + at, acc[t] * inv * read4(gate + o + at));
  }
}
template <int QT, int VT, int KEYS, int STAGES, int WAVES_PER_SIMD, bool SHARED = false>
__global__ __launch_bounds__(kPfThreads, WAVES_PER_SIMD) void attention_rows(const AttentionArgs a) {
  __shared__ __align__(16) v4u lds[kAttentionLds<QT, VT, KEYS, STAGES, SHARED>];
  attend_rows<QT, VT, KEYS, STAGES, SHARED>(a, blockIdx.x, gridDim.x, lds);
}

}  // namespace hybrid
}  // namespace qmk
