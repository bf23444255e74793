// Prefill kernels of the hybrid route's plain residual: the residual and its norms, values of the full attention, what lies behind the gated recurrences
// (qmk_hybrid_chunks.h).
#pragma once

#include "qmk_hybrid_prefill.h"

namespace qmk {
namespace hybrid {

// Row m of the residual (row want[m] where given): x, or the token's embedding where x is not there yet, plus the normed
// outputs of two branches.  Leaves the sum in x (unless `want`), a copy in `dump`, and in h its norm, or [x; embedding].
struct ResidualArgs {
  float* x;
  const float *a, *b, *wa, *wb;   // branches, or NULL
  const u16* table;               // embedding
  const int64_t* tokens;
  const int32_t* want;
  const float* weight;            // of the norm; NULL: [x; embedding]
  float* dump;
  int embed, vocab, M, D, width, norm;
  float scale, eps;
};
template <class T>
__global__ __launch_bounds__(kPfThreads) void residual_rows(const ResidualArgs g, Operand<T> h) {
  __shared__ float scratch[4];
  const int D = g.D;
  int m = g.want != nullptr ? g.want[blockIdx.x] : blockIdx.x;
  m = m < 0 || m >= g.M ? 0 : m;
  long long token = g.tokens[m];
  if (token < 0 || token >= g.vocab) token = 0;
  const u16* e = g.table + token * D;
  float* x = g.x + static_cast<size_t>(m) * D;
  const float *a = g.a + static_cast<size_t>(m) * D, *b = g.b + static_cast<size_t>(m) * D;
  float sa = 0.f, sb = 0.f;
  const bool two = g.a != nullptr;
  if (two) {
    for (int i = threadIdx.x * 4; i < D; i += kPfThreads * 4) {
      const f32x4 u = read4(a + i), v = read4(b + i);
      sa += u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + u[3] * u[3];
      sb += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    sa = g.scale / sqrtf(pf_block_sum(sa, scratch) / g.width + g.eps);
    sb = g.scale / sqrtf(pf_block_sum(sb, scratch) / g.width + g.eps);
  }
  auto value = [&](int i) {
    f32x4 v = g.embed ? read4(e + i) : read4(x + i);
    if (two) v += read4(a + i) * read4(g.wa + i) * sa + read4(b + i) * read4(g.wb + i) * sb;
    return v;
  };
  constexpr int kHeld = 4;
  f32x4 held[kHeld];
  float total = 0.f;
  auto take = [&](int i, f32x4 v) {
    total += v[0] + v[1] + v[2] + v[3];
    if (g.dump != nullptr) store4(g.dump + static_cast<size_t>(m) * D + i, v);
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    const int i = (j * kPfThreads + static_cast<int>(threadIdx.x)) * 4;
    held[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < D) take(i, held[j] = value(i));
  }
  for (int i = (kHeld * kPfThreads + threadIdx.x) * 4; i < D; i += kPfThreads * 4) take(i, value(i));
  const size_t out = static_cast<size_t>(blockIdx.x) * D * (g.weight == nullptr ? 2 : 1);
  float mean = 0.f, inv = 0.f;
  auto centred = [&](int i, f32x4 v) {
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = i + c < g.width ? v[c] - mean : 0.f;
    return v;
  };
  if (g.weight != nullptr) {
    if (g.norm == QMK_NORM_LAYER) mean = pf_block_sum(total, scratch) / g.width;
    float sq = 0.f;
    auto add = [&](int i, f32x4 v) {
      v = centred(i, v);
      sq += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    };
#pragma unroll
    for (int j = 0; j < kHeld; ++j) add((j * kPfThreads + threadIdx.x) * 4, held[j]);
    for (int i = (kHeld * kPfThreads + threadIdx.x) * 4; i < D; i += kPfThreads * 4) add(i, value(i));
    inv = 1.f / sqrtf(pf_block_sum(sq, scratch) / g.width + g.eps);
  }
  const bool keep = g.want == nullptr && (g.embed || two);
  auto put = [&](int i, f32x4 v) {
    if (keep) store4(x + i, v);
    if (g.weight != nullptr) {
      put4(h, out + i, centred(i, v) * inv * read4(g.weight + i));
    } else {
      put4(h, out + i, v);
      put4(h, out + D + i, read4(e + i));
    }
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    const int i = (j * kPfThreads + static_cast<int>(threadIdx.x)) * 4;
    if (i < D) put(i, held[j]);
  }
  for (int i = (kHeld * kPfThreads + threadIdx.x) * 4; i < D; i += kPfThreads * 4) put(i, value(i));
}

// v_t[key head][value][key] of keys 0 .. keys - 1 out of the cache (bf16: keys where value_place puts them), 64 keys x 64 columns a workgroup, in units
// of 16 bytes on both sides (4096 keys of 8 heads of 128 values, us: element by element 12.7, now 5.7).
template <class T>
__global__ __launch_bounds__(kPfThreads) void transpose_values(const T* cache, int pitch, int row, int value_at, int v_dim, int keys, int cap, T* out) {
  constexpr int kUnit = 16 / sizeof(T), kRow = 64 / kUnit;
  __shared__ __align__(16) T tile[64][64 + kUnit];
  const int key0 = blockIdx.x * 64, col0 = blockIdx.y * 64, kv = blockIdx.z;
  for (int id = threadIdx.x; id < 64 * kRow; id += kPfThreads) {
    const int r = id / kRow, c = id % kRow * kUnit;
    if (key0 + r < keys && col0 + c < v_dim)
      *reinterpret_cast<v4u*>(&tile[r][c]) = *reinterpret_cast<const v4u*>(cache + static_cast<size_t>(key0 + r) * pitch + kv * row + value_at + col0 + c);
  }
  __syncthreads();
  for (int id = threadIdx.x; id < 64 * kRow; id += kPfThreads) {      // (a row of `out` has room for whole units)
    const int c = id / kRow, r = id % kRow * kUnit;
    if (key0 + (sizeof(T) == 2 ? r & ~31 : r) >= keys || col0 + c >= v_dim) continue;
    v4u unit;
    T* e = reinterpret_cast<T*>(&unit);
#pragma unroll
    for (int j = 0; j < kUnit; ++j) e[j] = tile[sizeof(T) == 2 ? (r & ~31) + (j >> 2) * 16 + (r & 31) / 8 * 4 + (j & 3) : r + j][c];
    *reinterpret_cast<v4u*>(out + (static_cast<size_t>(kv) * v_dim + col0 + c) * cap + key0 + r) = unit;
  }
}

// The convolution's last inputs of a portion, for the next one.
__global__ __launch_bounds__(kPfThreads) void keep_inputs(const float* x, QmkHybridLayer l, int W, int slot, int flip, int M) {
  const int c = blockIdx.x * kPfThreads + threadIdx.x, n = l.taps - 1;
  if (c >= W) return;
  const float* old = l.shift + (static_cast<size_t>(slot) * 2 + flip) * n * W;
  float* now = l.shift + (static_cast<size_t>(slot) * 2 + 1 - flip) * n * W;
  for (int j = 0; j < n; ++j) {
    const int t = M - n + j;
    now[static_cast<size_t>(j) * W + c] = t >= 0 ? x[static_cast<size_t>(t) * W + c] : old[static_cast<size_t>(t + n) * W + c];
  }
}

// Per-head norm, weight and gate behind the recurrence: one wave per (token, head).
template <class T>
__global__ __launch_bounds__(kPfThreads) void state_out(const float* o, const T* gate, QmkHybridLayer l, int M, float eps, Operand<T> out) {
  const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (id >= M * l.heads) return;
  const int n = l.v_dim;
  const size_t at = static_cast<size_t>(id) * n;
  float sq = 0.f;
  for (int i = lane; i < n; i += 64) sq = fmaf(o[at + i], o[at + i], sq);
  const float inv = 1.f / sqrtf(wave_sum(sq) / l.v_true + eps);
  for (int i = lane; i < n; i += 64) put1(out, at + i, o[at + i] * inv * l.vec0[i] * to_f32(gate[at + i]));
}

}  // namespace hybrid
}  // namespace qmk
