// Prefill kernels of the hybrid route: a portion of M tokens, one launch per fused operation.
//
// Element type T (bf16 or fp32) is that of the activations between kernels; sums, norms, angles, scores, gates,
// recurrences and the residual streams are fp32 in both.  Weights are bf16 in memory in both; in fp32 mode a product's
// activations are cut into three bf16 parts on their way to the matrix instructions (qmk_hybrid_gemm.h), and attention and the
// recurrences use the fp32 ones.
#pragma once

#include "qmk_hybrid_attention.h"

namespace qmk {
namespace hybrid {

__device__ __forceinline__ float pf_block_sum(float v, float* scratch) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return scratch[0] + scratch[1] + scratch[2] + scratch[3];
}

// x = the token's embedding in every stream, u = what the first sublayer reads.
__global__ __launch_bounds__(kPfThreads) void embed_tokens(const u16* table, const int64_t* tokens, int vocab, const float* hc_in, int S, int D,
                                                           float* x, float* u) {
  const int m = blockIdx.x;
  long long t = tokens[m];
  if (t < 0 || t >= vocab) t = 0;
  const float g = weight_sum(hc_in, S);
  for (int i = threadIdx.x; i < D; i += kPfThreads) {
    const float e = bf2f(table[t * D + i]);
    for (int s = 0; s < S; ++s) x[(static_cast<size_t>(m) * S + s) * D + i] = e;
    u[static_cast<size_t>(m) * D + i] = e * g;
  }
}

// h = norm(u[row]); row = want[blockIdx.x] where given
template <class T>
__global__ __launch_bounds__(kPfThreads) void norm_rows(const float* u, const float* weight, const int32_t* want, int limit, int D, int true_width, float eps, Operand<T> h) {
  __shared__ float scratch[4];
  const int m = blockIdx.x;
  int from = want != nullptr ? want[m] : m;
  from = from < 0 || from >= limit ? 0 : from;
  const float* row = u + static_cast<size_t>(from) * D;
  float sq = 0.f;
  for (int i = threadIdx.x * 4; i < D; i += kPfThreads * 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(row + i);
    sq += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
  }
  const float inv = 1.f / sqrtf(pf_block_sum(sq, scratch) / true_width + eps);
  for (int i = threadIdx.x * 4; i < D; i += kPfThreads * 4)
    put4(h, static_cast<size_t>(m) * D + i, *reinterpret_cast<const f32x4*>(row + i) * inv * *reinterpret_cast<const f32x4*>(weight + i));
}

// The five mixes of a token's normed input with the previous token's; the last token leaves its own for the next portion.  What the first columns need is asked for
// at once: with few tokens it is a chain of trips to memory (us, element by element, again behind the sums -> now: 43 x 2048 9.2 -> 4.4, 1531 x 2048 19.0 -> 11.8, 2048 x 2048 23.2 -> 15.2).
template <class T>
__global__ __launch_bounds__(kPfThreads) void shift_mix(const float* u, QmkHybridLayer l, int slot, int flip, int M, int rows_cap, int D, int true_width, float eps, Operand<T> out) {
  __shared__ float scratch[4];
  const int m = blockIdx.x;
  const float* row = u + static_cast<size_t>(m) * D;
  const float* prev = row - D;
  const float* before = l.shift + (static_cast<size_t>(slot) * 2 + flip) * D;
  float* after = l.shift + (static_cast<size_t>(slot) * 2 + 1 - flip) * D;
  const float* last = m > 0 ? prev : before;
  constexpr int kHeld = 2;
  struct Columns {
    f32x4 row, last, norm, mix[5];
  } held[kHeld];
  auto at = [&](int j) { return (j * kPfThreads + static_cast<int>(threadIdx.x)) * 4; };
  auto ask = [&](Columns& c, int i) {
    c.row = read4(row + i);
    c.last = read4(last + i);
    c.norm = read4(l.norm1 + i);
#pragma unroll
    for (int q = 0; q < 5; ++q) c.mix[q] = read4(l.vec2 + q * D + i);
  };
  float sq = 0.f, sp = 0.f;
  auto add = [&](f32x4 v, f32x4 p) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sq = fmaf(v[e], v[e], sq);
      sp = fmaf(p[e], p[e], sp);
    }
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (at(j) < D) ask(held[j], at(j));
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (at(j) < D) add(held[j].row, held[j].last);
  for (int i = at(kHeld); i < D; i += kPfThreads * 4) add(read4(row + i), read4(last + i));
  const float inv = 1.f / sqrtf(pf_block_sum(sq, scratch) / true_width + eps);
  const float inv_p = 1.f / sqrtf(pf_block_sum(sp, scratch) / true_width + eps);
  auto put = [&](const Columns& c, int i) {
    const f32x4 h = c.row * inv * c.norm, d = (m > 0 ? c.last * inv_p * c.norm : c.last) - h;      // (the portion before leaves its last token normed)
    if (m == M - 1) store4(after + i, h);
#pragma unroll
    for (int q = 0; q < 5; ++q) put4(out, (static_cast<size_t>(q) * rows_cap + m) * D + i, h + d * c.mix[q]);
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (at(j) < D) put(held[j], at(j));
  for (int i = at(kHeld); i < D; i += kPfThreads * 4) {
    Columns c;
    ask(c, i);
    put(c, i);
  }
}

// u[m] = causal convolution of x (zeros or the previous portion's last inputs before it), four channels a thread.
template <class T>
__global__ __launch_bounds__(kPfThreads) void causal_conv(const T* x, QmkHybridLayer l, int slot, int flip, int M, T* out) {
  const int W = l.mix_width, quads = W / 4, n = l.taps;
  const long long id = static_cast<long long>(blockIdx.x) * kPfThreads + threadIdx.x;
  if (id >= static_cast<long long>(M) * quads) return;
  const int m = static_cast<int>(id / quads), c = static_cast<int>(id % quads) * 4;
  const float* old = l.shift + (static_cast<size_t>(slot) * 2 + flip) * (n - 1) * W;
  float* now = l.shift + (static_cast<size_t>(slot) * 2 + 1 - flip) * (n - 1) * W;
  auto input = [&](int t) {   // t >= -(n - 1)
    return t >= 0 ? read4(x + static_cast<size_t>(t) * W + c) : *reinterpret_cast<const f32x4*>(old + static_cast<size_t>(t + n - 1) * W + c);
  };
  f32x4 acc = *reinterpret_cast<const f32x4*>(l.vec1 + c);
  for (int j = 0; j < n; ++j) acc += *reinterpret_cast<const f32x4*>(l.vec2 + static_cast<size_t>(j) * W + c) * input(m - (n - 1) + j);
  store4(out + static_cast<size_t>(m) * W + c, acc);
  if (m == M - 1)
    for (int j = 0; j < n - 1; ++j) *reinterpret_cast<f32x4*>(now + static_cast<size_t>(j) * W + c) = input(M - (n - 1) + j);
}

// S_t = a_t S_{t-1} + b_t, out = S y: sixteen channels a workgroup, the portion cut into 64 runs of tokens.
constexpr int kScanChannels = 16, kScanRuns = 64;
template <class T>
__global__ __launch_bounds__(kScanChannels * kScanRuns) void lru_scan(const float* a, const float* b, const T* y, QmkHybridLayer l, int slot, int M, Operand<T> out) {
  __shared__ float sa[kScanRuns][kScanChannels], sb[kScanRuns][kScanChannels];
  const int W = l.mix_width, ch = threadIdx.x % kScanChannels, run = threadIdx.x / kScanChannels;
  const int c = blockIdx.x * kScanChannels + ch;
  const int per = (M + kScanRuns - 1) / kScanRuns, lo = min(run * per, M), hi = min(lo + per, M);
  float pa = 1.f, pb = 0.f;
#pragma unroll 4
  for (int t = lo; t < hi; ++t) {
    const size_t at = static_cast<size_t>(t) * W + c;
    const float av = a[at];
    pa *= av;
    pb = fmaf(av, pb, b[at]);
  }
  sa[run][ch] = pa;
  sb[run][ch] = pb;
  __syncthreads();
  float* st = l.state + static_cast<size_t>(slot) * W + c;
  if (run == 0) {
    float s = *st;
    for (int r = 0; r < kScanRuns; ++r) {
      const float e = fmaf(sa[r][ch], s, sb[r][ch]);
      sb[r][ch] = s;      // the state the run starts from
      s = e;
    }
    *st = s;
  }
  __syncthreads();
  float s = sb[run][ch];
#pragma unroll 4
  for (int t = lo; t < hi; ++t) {
    const size_t at = static_cast<size_t>(t) * W + c;
    s = fmaf(a[at], s, b[at]);
    put1(out, at, s * to_f32(y[at]));
  }
}

// Keys first .. position + M - 1 side by side: new rows normed and rotated (and stored in the cache), old ones copied.
template <class T>
__global__ __launch_bounds__(kPfThreads) void latent_rows(const float* raw, QmkHybridLayer l, int slot, int first, int position, float eps, T* rows) {
  __shared__ float scratch[4];
  const int width = l.rank + l.rot_dim, pos = first + blockIdx.x;
  T* row = static_cast<T*>(l.cache) + (static_cast<size_t>(slot) * l.ring + pos % l.ring) * width;
  T* out = rows + static_cast<size_t>(blockIdx.x) * width;
  if (pos < position) {
    for (int i = threadIdx.x; i < width; i += kPfThreads) out[i] = row[i];
    return;
  }
  const float* c = raw + static_cast<size_t>(pos - position) * width;
  float sq = 0.f;
  for (int i = threadIdx.x; i < l.rank; i += kPfThreads) sq = fmaf(c[i], c[i], sq);
  const float inv = 1.f / sqrtf(pf_block_sum(sq, scratch) / l.rank_true + eps);
  for (int i = threadIdx.x * 2; i < width; i += kPfThreads * 2) {
    float a = c[i], b = c[i + 1];
    if (i < l.rank) {
      a = a * inv * l.vec0[i];
      b = b * inv * l.vec0[i + 1];
    } else {
      rotate(l, pos, i - l.rank, a, b);
    }
    row[i] = out[i] = from_f32<T>(a);
    row[i + 1] = out[i + 1] = from_f32<T>(b);
  }
}

// The same as attention_rows for fp32 portions, values in the order of their keys, 32 keys a step through registers.
// GROUPS = 2: two groups of four waves take the 32-key steps in turn, for the same queries, and meet at the end: a step is a chain (keys into LDS, scores, maximum
// over the lanes, weights, values), and a CU that holds one or two workgroups of four waves mostly waits for it (us, one group -> two: 200 queries of 16 heads of 192 | 128 34 -> 29).
template <int QT, int VT, int GROUPS>   // most 32-column steps of a query, most 16-row tiles of a value
__global__ __launch_bounds__(kPfThreads * GROUPS) void window_attention(const float* q, Keys<float> keys, const float* rows, const float* v_t, const float* gate, QmkHybridLayer l,
                                                               int first, int position, int M, int keys_cap, Operand<float> out) {
  constexpr int kKeys = 32, kU = 4;      // keys a step; a unit of 16 bytes, which also sets rows apart
  struct Step {
    float k[kKeys][QT * 32 + kU];
    float v[VT * 16][kKeys + kU];
  };
  __shared__ __align__(16) Step stage[GROUPS];
  const int tid = threadIdx.x % kPfThreads, lane = tid & 63, wave = tid >> 6, g = lane >> 4, col = lane & 15;
  const int part = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kPfThreads);
  auto& sk = stage[part].k;
  auto& sv = stage[part].v;
  // Later queries see more keys where no window ends.  Workgroups 256 apart share a CU: every other such run of heads takes
  // its queries from the far end, so that a CU gets long and short ones.
  const bool mirrored = (blockIdx.y * gridDim.x >> 8 & 1) == 0;
  const int head = blockIdx.y, kv = head / keys.heads_per, q0 = (mirrored ? gridDim.x - 1 - blockIdx.x : blockIdx.x) * 64;
  const int dq = l.q_stride, steps = dq / 32, vt = l.v_dim / 16, width = l.rank + l.rot_dim;
  const int m = q0 + wave * 16 + col, pos = position + m;
  Frag<float> fq[QT];
#pragma unroll
  for (int s = 0; s < QT; ++s)
    if (s < steps) fq[s] = load_frag(q + static_cast<size_t>(min(m, M - 1)) * l.heads * dq + head * dq + s * 32 + g * 8);
  f32x4 acc[VT] = {};
  float top = -INFINITY, sum = 0.f;
  const float scale = l.scale * kLog2e;
  const int lo = max(first, position + q0 + 1 - l.window);      // the first key any of the 64 queries sees
  const int hi = min(position + q0 + 64, position + M);          // behind the last one
  // Staging: each thread has fixed places in a tile of keys and of transposed values; the next tile is in flight while
  // this one is used.
  constexpr int kKLoads = kKeys * QT * 32 / kU / kPfThreads, kVLoads = VT * 16 * kKeys / kU / kPfThreads;
  static_assert(kKLoads * kPfThreads * kU == kKeys * QT * 32 && kVLoads * kPfThreads * kU == VT * 16 * kKeys, "every thread stages the same number of units");
  const int begin = first + ((lo - first) & ~(kKeys - 1)), base0 = begin + part * kKeys;
  const float* k_at[kKLoads];
  int k_step[kKLoads];
  v4u rk[kKLoads], rv[kVLoads];
#pragma unroll
  for (int i = 0; i < kKLoads; ++i) {
    const int id = i * kPfThreads + tid, r = id / (QT * 32 / kU), c = id % (QT * 32 / kU) * kU, row = base0 + r - first;
    k_at[i] = nullptr;                 // columns behind the rotated part: zeros
    k_step[i] = 0;
    if (c < l.head_dim) {
      k_at[i] = keys.at + static_cast<size_t>(row) * keys.pitch + kv * keys.head + c;
      k_step[i] = GROUPS * kKeys * keys.pitch;
    } else if (c < l.head_dim + l.rot_dim) {
      k_at[i] = rows + static_cast<size_t>(row) * width + l.rank + c - l.head_dim;
      k_step[i] = GROUPS * kKeys * width;
    }
  }
  auto fetch = [&](int base) {
#pragma unroll
    for (int i = 0; i < kKLoads; ++i) {
      const int r = (i * kPfThreads + tid) / (QT * 32 / kU);
      rk[i] = v4u{0u, 0u, 0u, 0u};
      if (k_at[i] != nullptr && base + r < hi) rk[i] = *reinterpret_cast<const v4u*>(k_at[i]);
      k_at[i] = k_at[i] == nullptr ? nullptr : k_at[i] + k_step[i];
    }
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const int id = i * kPfThreads + tid, r = id / (kKeys / kU), c = id % (kKeys / kU) * kU;
      rv[i] = v4u{0u, 0u, 0u, 0u};
      if (r < l.v_dim && base + c < hi) rv[i] = *reinterpret_cast<const v4u*>(v_t + static_cast<size_t>(kv * l.v_dim + r) * keys_cap + base - first + c);
      if (base + c + kU > hi) {   // keys behind the last one: whatever the buffer holds there must not enter a sum
        float* e = reinterpret_cast<float*>(&rv[i]);
#pragma unroll
        for (int j = 0; j < kU; ++j)
          if (base + c + j >= hi) e[j] = 0.f;
      }
    }
  };
  fetch(base0);
  const int first_pos = position + q0 + wave * 16;       // this wave's queries: first_pos .. first_pos + 15
  for (int base = base0; base - part * kKeys < hi; base += GROUPS * kKeys) {      // (the groups share the barriers)
#pragma unroll
    for (int i = 0; i < kKLoads; ++i) {
      const int id = i * kPfThreads + tid;
      *reinterpret_cast<v4u*>(&sk[id / (QT * 32 / kU)][id % (QT * 32 / kU) * kU]) = rk[i];
    }
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const int id = i * kPfThreads + tid;
      *reinterpret_cast<v4u*>(&sv[id / (kKeys / kU)][id % (kKeys / kU) * kU]) = rv[i];
    }
    __syncthreads();
    if (base + GROUPS * kKeys < hi) fetch(base + GROUPS * kKeys);
    if (base < hi) {
      f32x4 d[2] = {};
#pragma unroll
      for (int s = 0; s < QT; ++s)
        if (s < steps) {
#pragma unroll
          for (int t = 0; t < 2; ++t) d[t] = mma(load_frag(&sk[t * 16 + col][s * 32 + g * 8]), fq[s], d[t]);
        }
      float w[8];
      float best = top;
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = d[j >> 2][j & 3] * scale;
      if (base + kKeys - 1 > first_pos || first_pos + 15 - base >= l.window) {   // some query does not see some key
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int key = base + (j >> 2) * 16 + g * 4 + (j & 3), dist = pos - key;
          if (dist < 0 || dist >= l.window) w[j] = -INFINITY;
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) best = fmaxf(best, w[j]);
      best = fmaxf(best, __shfl_xor(best, 16));
      best = fmaxf(best, __shfl_xor(best, 32));
      const float ref = best == -INFINITY ? 0.f : best;      // no key of this query yet
      const float shrink = exp2_fast(top - ref);
      float step_sum = 0.f;
      Frag<float> fp;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w[j] = exp2_fast(w[j] - ref);
        step_sum += w[j];
        fp.set(j, w[j]);
      }
      sum = sum * shrink + step_sum;
      top = best;
#pragma unroll
      for (int t = 0; t < VT; ++t)
        if (t < vt) {
          Frag<float> fv;
          const float* r = &sv[t * 16 + col][0];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            fv.set(j, r[g * 4 + j]);
            fv.set(4 + j, r[16 + g * 4 + j]);
          }
          acc[t] = mma(fv, fp, acc[t] * shrink);
        }
    }
    __syncthreads();
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  if constexpr (GROUPS == 2) {      // the second group's maximum, sum and values of every lane's query onto the first one's
    float* box = reinterpret_cast<float*>(stage) + tid;
    static_assert(sizeof(stage) >= sizeof(float) * (VT * 4 + 2) * kPfThreads, "the giving group's states");
    if (part == 1) {
      box[0] = top;
      box[kPfThreads] = sum;
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) box[(2 + t * 4 + i) * kPfThreads] = acc[t][i];
    }
    __syncthreads();
    if (part == 1) return;
    const float other = box[0], most = fmaxf(top, other), ref = most == -INFINITY ? 0.f : most, mine = exp2_fast(top - ref), theirs = exp2_fast(other - ref);
    sum = sum * mine + box[kPfThreads] * theirs;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][i] = acc[t][i] * mine + box[(2 + t * 4 + i) * kPfThreads] * theirs;
  }
  if (m >= M) return;
  const float inv = 1.f / sum;
  const size_t at = static_cast<size_t>(m) * l.heads * l.v_dim + head * l.v_dim;
#pragma unroll
  for (int t = 0; t < VT; ++t)
    if (t < vt) put4(out, at + t * 16 + g * 4, acc[t] * inv * read4(gate + at + t * 16 + g * 4));
}

// The same for few workgroups: 16 queries of a head, whose four waves take the 32-key steps in turn and meet at the end.  A step's keys and values have one reader, so they go from
// memory to its registers, the next step's keys behind the scores and its values behind the sums; what bounds it is the fp32 matrix instruction, 160 a step of 192 | 128 (us,
// 16 heads, 64 queries a workgroup -> now: 200 of 192 | 128 30.0 -> 20.7, behind 400 keys 69.5 -> 45.6).
template <int QT, int VT>
__global__ __launch_bounds__(kPfThreads, 1) void few_attention(const float* q, Keys<float> keys, const float* rows, const float* v_t, const float* gate, QmkHybridLayer l, int first,
                                                               int position, int M, int keys_cap, Operand<float> out) {
  constexpr int kKeys = 32, kWaves = kPfThreads / 64, kTiles = VT / kWaves;      // tiles of a value a wave finishes
  static_assert(VT % kWaves == 0, "whole tiles");
  __shared__ f32x4 box[kWaves][VT][64];
  __shared__ float tops[kWaves][64], sums[kWaves][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, col = lane & 15;
  const int head = blockIdx.y, kv = head / keys.heads_per, q0 = blockIdx.x * 16, m = q0 + col, pos = position + m;
  const int dq = l.q_stride, steps = dq / 32, vt = l.v_dim / 16, width = l.rank + l.rot_dim;
  const int lo = max(first, position + q0 + 1 - l.window), hi = min(position + q0 + 16, position + M);      // keys that any of these queries sees
  const int begin = first + ((lo - first) & ~(kKeys - 1));
  const float* zeros = reinterpret_cast<const float*>(kZeroUnit);
  f32x4 k[2][QT][2], v[VT][2];
  auto load_keys = [&](int base) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = min(base + t * 16 + col, hi - 1) - first;      // (keys behind the last one are that one again, and masked)
      const float* at = keys.at + static_cast<size_t>(row) * keys.pitch + kv * keys.head;
      const float* turned = rows + static_cast<size_t>(row) * width + l.rank - l.head_dim;
#pragma unroll
      for (int s = 0; s < QT; ++s)
        if (s < steps) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int c = s * 32 + g * 8 + u * 4;
            k[t][s][u] = read4(c < l.head_dim ? at + c : rows != nullptr && c < l.head_dim + l.rot_dim ? turned + c : zeros);
          }
        }
    }
  };
  auto load_values = [&](int base) {
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vt) {
        const float* at = v_t + static_cast<size_t>(kv * l.v_dim + t * 16 + col) * keys_cap - first;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int key = base + u * 16 + g * 4;
          v[t][u] = read4(key < hi ? at + key : zeros);
        }
      }
  };
  Frag<float> fq[QT];
#pragma unroll
  for (int s = 0; s < QT; ++s)
    if (s < steps) fq[s] = load_frag(q + static_cast<size_t>(min(m, M - 1)) * l.heads * dq + head * dq + s * 32 + g * 8);
  f32x4 acc[VT] = {};
  float top = -INFINITY, sum = 0.f;
  const float scale = l.scale * kLog2e;
  const int own = begin + wave * kKeys;
  if (own < hi) {
    load_keys(own);
    load_values(own);
  }
  for (int base = own; base < hi; base += kWaves * kKeys) {
    f32x4 d[2] = {};
#pragma unroll
    for (int s = 0; s < QT; ++s)
      if (s < steps) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          Frag<float> f;
#pragma unroll
          for (int j = 0; j < 8; ++j) f.set(j, k[t][s][j >> 2][j & 3]);
          d[t] = mma(f, fq[s], d[t]);
        }
      }
    const int next = base + kWaves * kKeys;
    if (next < hi) load_keys(next);
    float w[8], best = top;
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = d[j >> 2][j & 3] * scale;
    if (base + kKeys - 1 > position + q0 || position + q0 + 15 - base >= l.window) {   // some query does not see some key
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int dist = pos - (base + (j >> 2) * 16 + g * 4 + (j & 3));
        if (dist < 0 || dist >= l.window) w[j] = -INFINITY;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) best = fmaxf(best, w[j]);
    best = fmaxf(best, __shfl_xor(best, 16));
    best = fmaxf(best, __shfl_xor(best, 32));
    const float ref = best == -INFINITY ? 0.f : best;      // no key of this query yet
    const float shrink = exp2_fast(top - ref);
    float step_sum = 0.f;
    Frag<float> fp;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      w[j] = exp2_fast(w[j] - ref);
      step_sum += w[j];
      fp.set(j, w[j]);
    }
    sum = sum * shrink + step_sum;
    top = best;
    const bool last = base + kKeys > hi;
#pragma unroll
    for (int t = 0; t < VT; ++t)
      if (t < vt) {
        Frag<float> f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {      // keys behind the last one: whatever the buffer holds there must not enter a sum
          const float x = v[t][j >> 2][j & 3];
          f.set(j, last && base + (j >> 2) * 16 + g * 4 + (j & 3) >= hi ? 0.f : x);
        }
        acc[t] = mma(f, fp, acc[t] * shrink);
      }
    if (next < hi) load_values(next);
  }
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  tops[wave][lane] = top;
  sums[wave][lane] = sum;
#pragma unroll
  for (int t = 0; t < VT; ++t) box[wave][t][lane] = acc[t];
  __syncthreads();
  if (m >= M) return;
  float most = -INFINITY, part[kWaves], total = 0.f;
#pragma unroll
  for (int p = 0; p < kWaves; ++p) most = fmaxf(most, tops[p][lane]);
  const float ref = most == -INFINITY ? 0.f : most;
#pragma unroll
  for (int p = 0; p < kWaves; ++p) {
    part[p] = exp2_fast(tops[p][lane] - ref);
    total += sums[p][lane] * part[p];
  }
  const float inv = 1.f / total;
  const size_t at = static_cast<size_t>(m) * l.heads * l.v_dim + head * l.v_dim;
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    const int t = wave * kTiles + i;
    if (t >= vt) continue;
    f32x4 o = {};
#pragma unroll
    for (int p = 0; p < kWaves; ++p) o += box[p][t][lane] * part[p];
    put4(out, at + t * 16 + g * 4, o * inv * read4(gate + at + t * 16 + g * 4));
  }
}

// Per-head norm, weight and gate behind the recurrence: one wave per (token, head).
template <class T>
__global__ __launch_bounds__(kPfThreads) void wkv_out(const float* o, const T* gate, QmkHybridLayer l, int M, float eps, Operand<T> out) {
  const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (id >= M * l.heads) return;
  const int n = l.head_dim, m = id / l.heads, head = id % l.heads;
  const size_t at = static_cast<size_t>(m) * l.heads * n + head * n;
  float sq = 0.f;
  for (int i = lane; i < n; i += 64) sq = fmaf(o[at + i], o[at + i], sq);
  const float inv = 1.f / sqrtf(wave_sum(sq) / l.head_dim_true + eps);
  for (int i = lane; i < n; i += 64) put1(out, at + i, o[at + i] * inv * l.vec0[head * n + i] * to_f32(gate[at + i]));
}

__global__ __launch_bounds__(kPfThreads) void sum_streams(const float* x, int S, int D, float* out) {
  const int m = blockIdx.x;
  for (int i = threadIdx.x; i < D; i += kPfThreads) {
    float t = 0.f;
    for (int s = 0; s < S; ++s) t += x[(static_cast<size_t>(m) * S + s) * D + i];
    out[static_cast<size_t>(m) * D + i] = t;
  }
}

}  // namespace hybrid
}  // namespace qmk
