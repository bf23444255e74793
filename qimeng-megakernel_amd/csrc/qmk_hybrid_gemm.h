// Matrix products of the hybrid route's prefill: out[m][n] = sum_k a[m][k] w[n][k], tokens x weight rows, with everything
// element-wise done in the epilogue.
#pragma once

#include <type_traits>

#include "qmk_hybrid_ops.h"
#include "qmk_hybrid_tiles.h"

namespace qmk {
namespace hybrid {

constexpr int kPfThreads = 256;

enum : int {
  EPI_STORE = 0,        // out T [m][ldo]
  EPI_STORE_VALUES,     // the same, columns where value_place puts them
  EPI_RGLRU_IN,         // gelu of the y half, bias on both
  EPI_LRU_GATES,        // (r, i) pairs -> decay a and input b of the recurrence
  EPI_LATENT_IN,        // rotation of q, sigmoid of the gate, raw latent
  EPI_RESIDUAL,         // all streams of the residual and the next sublayer's input (residual_quads)
  EPI_GEGLU,            // (gate, up) pairs
  EPI_WKV_IN,           // r, k, v fp32; silu gate; tanh
  EPI_WKV_DECAY,        // exp(-exp(. + w0))
  EPI_LOGITS,
  EPI_CAPPED_LOGITS,    // logits times a constant, softly capped
  EPI_ADD,              // onto the fp32 residual
  EPI_ATTENTION_IN,     // rotation of q and k, k and v into the cache, sigmoid of the gate
  EPI_DELTA_IN,         // q, k, v fp32; raw ranks; sigmoid of the step sizes
  EPI_DELTA_DECAY,
  EPI_SIGMOID,
  EPI_GLA_IN,           // q, k, v fp32; silu gate; raw rank
  EPI_GLA_DECAY,
};

// An fp32 value is the sum of three bf16 values of its sign: its upper half, the upper half of what that leaves, and the rest, which has eight
// bits at most.  Both remainders are exact, so the sum is, from 2^-110 on (below, what is smaller than bf16's smallest value, 2^-133, is cut off).  A
// product of two bf16 values is exact in fp32: three bf16 instructions add up the same products as the eight fp32 ones of the same
// columns, in a fifth of their time.  Values that are not finite stay whole in the first part; infinite values on the other side: resolve_undefined.
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ float behind_upper_half(float v) { return v - __uint_as_float(__float_as_uint(v) & 0xffff0000u); }
__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u; }
// Two neighbouring values -> their parts.
__device__ __forceinline__ void split2(float x, float y, uint32_t (&part)[3]) {
  part[0] = upper_halves(x, y);
  const float x1 = behind_upper_half(x), y1 = behind_upper_half(y);
  part[1] = upper_halves(x1, y1);
  part[2] = upper_halves(behind_upper_half(x1), behind_upper_half(y1));
  if (__builtin_expect(not_finite(x) | not_finite(y), 0)) {
    const float v[2] = {x, y};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (not_finite(v[e])) {
        const uint32_t keep = e ? 0x0000ffffu : 0xffff0000u, top = v[e] != v[e] ? 0x7fc0u : __float_as_uint(v[e]) >> 16;
        part[0] = (part[0] & keep) | (e ? top << 16 : top);
        part[1] &= keep;
        part[2] &= keep;
      }
    }
  }
}

// fp32 mode: the rows a projection reads next (normed input, mixed heads, gated rows) are left as three bf16 parts, `part`
// elements from one to the next, by the kernel that makes them, so that their tiles go from memory to LDS as they are and by
// themselves, instead of through the registers of the workgroups that read them.  part = 0: they stay whole.
template <class T>
struct Operand {
  T* at;
  size_t part;
  __device__ __forceinline__ u16* parts() const { return reinterpret_cast<u16*>(at); }
};
template <class T>
__device__ __forceinline__ void store4(T* at, f32x4 v);
template <class T>
__device__ __forceinline__ void put4(const Operand<T>& to, size_t i, f32x4 v) {
  if constexpr (sizeof(T) == 4) {
    if (to.part != 0) {
      uint32_t a[3], b[3];
      split2(v[0], v[1], a);
      split2(v[2], v[3], b);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(to.parts() + q * to.part + i) = make_uint2(a[q], b[q]);
      return;
    }
  }
  store4(to.at + i, v);
}
template <class T>
__device__ __forceinline__ void put2(const Operand<T>& to, size_t i, float x, float y) {
  if constexpr (sizeof(T) == 4) {
    if (to.part != 0) {
      uint32_t a[3];
      split2(x, y, a);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint32_t*>(to.parts() + q * to.part + i) = a[q];
      return;
    }
    *reinterpret_cast<float2*>(to.at + i) = make_float2(x, y);
  } else {
    *reinterpret_cast<uint32_t*>(to.at + i) = f2bf2(x, y);
  }
}
template <class T>
__device__ __forceinline__ void put1(const Operand<T>& to, size_t i, float x) {
  if constexpr (sizeof(T) == 4) {
    if (to.part != 0) {
      uint32_t a[3];
      split2(x, 0.f, a);
#pragma unroll
      for (int q = 0; q < 3; ++q) to.parts()[q * to.part + i] = static_cast<u16>(a[q]);
      return;
    }
  }
  to.at[i] = from_f32<T>(x);
}

// Where key k lies in a row of transposed values of a bf16 portion: of every 32 keys, the eight that a lane of the value product takes (4g .. 4g+3 and
// 16+4g .. 16+4g+3) side by side, one read of 16 bytes.
__host__ __device__ constexpr int value_place(int k) { return (k & ~31) | ((k & 12) << 1) | ((k & 16) >> 2) | (k & 3); }

struct GemmArgs {
  const void* a;         // TA [M][lda]
  const void* w;         // TW [N][ldw]
  int M, N, K, lda, ldw, groups, last_n;   // group g: a + g a_step, w + g w_step, N rows (the last: last_n)
  long long a_step, w_step;
  int epi;
  void* out;             // meaning by epilogue
  void* out2;
  float* f0;
  float* f1;
  const void* src;
  int ldo;
  QmkHybridLayer layer;
  int down, first, position, streams, width, rows_cap, slot;
  float logit_scale, logit_softcap;
  const float* next;
  float* partial;        // sums of the parts of a product that is cut along K, and a zero per tile
  int32_t* tickets;
  int splits;
  size_t a_part;         // Operand::part of a (last: the bf16 mode reads neither, and its first cache lines stay as they are)
  size_t out_part;       // EPI_GEGLU: Operand::part of out
};

template <class T>
__device__ __forceinline__ void store4(T* at, f32x4 v) {
  if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<uint2*>(at) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
  } else {
    *reinterpret_cast<f32x4*>(at) = v;
  }
}
template <class T>
__device__ __forceinline__ f32x4 read4(const T* at) {
  if constexpr (sizeof(T) == 2) {
    const uint2 t = *reinterpret_cast<const uint2*>(at);
    return f32x4{bf_lo(t.x), bf_hi(t.x), bf_lo(t.y), bf_hi(t.y)};
  } else {
    return *reinterpret_cast<const f32x4*>(at);
  }
}

// Eight values side by side.
template <class T>
__device__ __forceinline__ void store8(T* at, f32x4 lo, f32x4 hi) {
  if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<v4u*>(at) = v4u{f2bf2(lo[0], lo[1]), f2bf2(lo[2], lo[3]), f2bf2(hi[0], hi[1]), f2bf2(hi[2], hi[3])};
  } else {
    store4(at, lo);
    store4(at + 4, hi);
  }
}
template <class F>
__device__ __forceinline__ f32x4 each(f32x4 v, F&& f) { return f32x4{f(v[0]), f(v[1]), f(v[2]), f(v[3])}; }

// Eight consecutive outputs n .. n+7 of a token (sizes of storage are multiples of sixteen, so they are of one kind).  What depends on the columns alone
// is worked out once, ahead of the tokens; four pairs' angles of a rotation are read together (us, 2048 x 6144 x 2048 into an attention, inside a portion, pair by pair with
// places worked out for every token -> so: 79 -> 70; 1531 x 5696 x 2048 into a latent one 58 -> 56).
struct Angles {
  f32x4 cos, sin;
};
template <class T, int EPI>
struct Epilogue {
  const GemmArgs& g;
  const int group, n;
  f32x4 b[2] = {};       // constants of the eight outputs
  int dim = -1;          // rotated dimensions: the first of the eight (-1: none is)
  int place = 0;         // keys and values of an attention: where they lie in a cache row

  __device__ __forceinline__ Epilogue(const GemmArgs& args, int group_, int n_) : g(args), group(group_), n(n_) {
    const QmkHybridLayer& l = g.layer;
    const float* from = EPI == EPI_RGLRU_IN ? l.in_b + n
                        : EPI == EPI_LRU_GATES ? l.mid_b + static_cast<size_t>(group) * 2 * l.block_dim + n
                        : EPI == EPI_WKV_DECAY || EPI == EPI_DELTA_DECAY || EPI == EPI_GLA_DECAY ? l.mid_b + n : nullptr;
    if constexpr (EPI == EPI_RGLRU_IN || EPI == EPI_LRU_GATES || EPI == EPI_WKV_DECAY || EPI == EPI_DELTA_DECAY || EPI == EPI_GLA_DECAY) {
      b[0] = read4(from);
      b[1] = read4(from + 4);
    }
    if constexpr (EPI == EPI_LATENT_IN) {
      if (n < l.heads * l.q_stride) dim = max(n % l.q_stride - l.head_dim, -1);
    } else if constexpr (EPI == EPI_ATTENTION_IN) {
      const int c = n - l.heads * l.q_stride, width = l.head_dim + l.v_dim, k_rows = l.kv_heads * l.head_dim;
      if (c < 0) {
        dim = n % l.q_stride;
      } else if (c < k_rows) {
        dim = c % l.head_dim;
        place = c / l.head_dim * width + dim;
      } else {
        place = (c - k_rows) / l.v_dim * width + l.head_dim + (c - k_rows) % l.v_dim;
      }
    }
    if (dim >= l.rot_true) dim = -1;
  }

  __device__ __forceinline__ Angles angles(int m) const {
    const QmkHybridLayer& l = g.layer;
    Angles t{};
    if (dim < 0) return t;
    const size_t at = static_cast<size_t>(g.position + m) * (l.rot_true / 2) + (dim >> 1);
    if (l.rot_true % 8 == 0) {
      t.cos = read4(l.rope_cos + at);
      t.sin = read4(l.rope_sin + at);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const size_t pair = at + min(i, (l.rot_true - dim) / 2 - 1);
        t.cos[i] = l.rope_cos[pair];
        t.sin[i] = l.rope_sin[pair];
      }
    }
    return t;
  }

  // Pairs (dim, dim + 1) .. (dim + 6, dim + 7) of a head turned to their position.
  __device__ __forceinline__ void turn(const Angles& t, f32x4& lo, f32x4& hi) const {
    float e[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (dim + 2 * i >= g.layer.rot_true) continue;
      const float x = e[2 * i] * t.cos[i] - e[2 * i + 1] * t.sin[i];
      e[2 * i + 1] = e[2 * i + 1] * t.cos[i] + e[2 * i] * t.sin[i];
      e[2 * i] = x;
    }
    lo = f32x4{e[0], e[1], e[2], e[3]};
    hi = f32x4{e[4], e[5], e[6], e[7]};
  }

  __device__ __forceinline__ void operator()(int m, f32x4 lo, f32x4 hi) const {
    const QmkHybridLayer& l = g.layer;
    T *out = static_cast<T*>(g.out), *out2 = static_cast<T*>(g.out2);
    const auto gate = [](float x) { return sigmoid(x); };
    const auto silu = [](float x) { return x * sigmoid(x); };
    const auto gelu = [](float x) { return gelu_tanh(x); };
    const size_t row = static_cast<size_t>(m);
    if constexpr (EPI == EPI_STORE) {
      store8(out + row * g.ldo + n, lo, hi);
    } else if constexpr (EPI == EPI_STORE_VALUES) {
      store4(out + row * g.ldo + value_place(n), lo);
      store4(out + row * g.ldo + value_place(n + 4), hi);
    } else if constexpr (EPI == EPI_RGLRU_IN) {
      lo += b[0];
      hi += b[1];
      if (n < l.mix_width) store8(out + row * l.mix_width + n, each(lo, gelu), each(hi, gelu));
      else store8(out2 + row * l.mix_width + n - l.mix_width, lo, hi);
    } else if constexpr (EPI == EPI_LRU_GATES) {
      const int c = group * l.block_dim + n / 2;
      const size_t at = row * l.mix_width + c;
      const f32x4 v[2] = {lo + b[0], hi + b[1]}, u = read4(static_cast<const T*>(g.src) + at), rate = read4(l.vec0 + c);
      f32x4 decay, input;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float la = sigmoid(v[i >> 1][i * 2 & 3]) * rate[i];
        decay[i] = expf(la);
        input[i] = sqrtf(-expm1f(2.f * la)) * sigmoid(v[i >> 1][(i * 2 & 3) + 1]) * u[i];
      }
      store4(g.f0 + at, decay);
      store4(g.f1 + at, input);
    } else if constexpr (EPI == EPI_LATENT_IN) {
      const int q_rows = l.heads * l.q_stride, g_rows = l.heads * l.v_dim;
      if (n < q_rows) {
        if (dim >= 0) turn(angles(m), lo, hi);
        store8(out + row * q_rows + n, lo, hi);
      } else if (n < q_rows + g_rows) {
        store8(out2 + row * g_rows + n - q_rows, each(lo, gate), each(hi, gate));
      } else {
        store8(g.f0 + row * (l.rank + l.rot_dim) + n - q_rows - g_rows, lo, hi);
      }
    } else if constexpr (EPI == EPI_GEGLU) {
      const f32x4 a = {lo[0], lo[2], hi[0], hi[2]}, up = {lo[1], lo[3], hi[1], hi[3]};
      put4(Operand<T>{out, g.out_part}, row * l.ff + n / 2, (l.act == QMK_ACT_SILU ? each(a, silu) : each(a, gelu)) * up);
    } else if constexpr (EPI == EPI_WKV_IN) {
      const int N = l.heads * l.head_dim;
      if (group < 3) {
        store8(g.f0 + (static_cast<size_t>(group) * g.rows_cap + m) * N + n, lo, hi);
      } else if (group == 3) {
        store8(out + row * N + n, each(lo, silu), each(hi, silu));
      } else {
        const auto bound = [](float x) { return tanhf(x); };
        store8(out2 + row * l.rank + n, each(lo, bound), each(hi, bound));
      }
    } else if constexpr (EPI == EPI_WKV_DECAY) {
      const auto decay = [](float x) { return expf(-expf(x)); };
      store8(g.f0 + row * g.ldo + n, each(lo + b[0], decay), each(hi + b[1], decay));
    } else if constexpr (EPI == EPI_CAPPED_LOGITS) {
      const auto cap = [&](float x) { return soft_cap(x * g.logit_scale, g.logit_softcap); };
      store8(g.f0 + row * g.ldo + n, each(lo, cap), each(hi, cap));
    } else if constexpr (EPI == EPI_ADD) {
      float* x = g.f0 + row * g.ldo + n;
      store8(x, read4(x) + lo, read4(x + 4) + hi);
    } else if constexpr (EPI == EPI_ATTENTION_IN) {
      const int q_rows = l.heads * l.q_stride, kv_rows = l.kv_heads * (l.head_dim + l.v_dim), pos = g.position + m;
      if (dim >= 0) turn(angles(m), lo, hi);
      if (n < q_rows) {
        store8(out + row * q_rows + n, lo, hi);
      } else if (n < q_rows + kv_rows) {
        const int ring = pos < l.ring ? pos : pos % l.ring;
        store8(static_cast<T*>(l.cache) + (static_cast<size_t>(g.slot) * l.ring + ring) * kv_rows + place, lo, hi);
      } else {
        store8(out2 + row * l.mix_width + n - q_rows - kv_rows, each(lo, gate), each(hi, gate));
      }
    } else if constexpr (EPI == EPI_DELTA_IN) {
      const int channels = conv_channels(l), ranks = l.rank + l.gate_rank;
      if (n < channels) store8(g.f1 + row * channels + n, lo, hi);
      else if (n < channels + ranks) store8(out2 + row * ranks + n - channels, lo, hi);
      else store8(g.f0 + row * g.ldo + n - channels - ranks, each(lo, gate), each(hi, gate));
    } else if constexpr (EPI == EPI_DELTA_DECAY) {
      const int head = n / l.head_dim;
      const auto decay = [&](float x) { return delta_decay(l, head, x); };
      store8(g.f0 + row * g.ldo + n, each(lo + b[0], decay), each(hi + b[1], decay));
    } else if constexpr (EPI == EPI_SIGMOID) {
      store8(out + row * g.ldo + n, each(lo, gate), each(hi, gate));
    } else if constexpr (EPI == EPI_GLA_IN) {
      const int qkv = 2 * l.heads * l.head_dim + l.mix_width;
      if (n < qkv) store8(g.f0 + row * qkv + n, lo, hi);
      else if (n < qkv + l.mix_width) store8(out + row * l.mix_width + n - qkv, each(lo, silu), each(hi, silu));
      else store8(out2 + row * l.rank + n - qkv - l.mix_width, lo, hi);
    } else if constexpr (EPI == EPI_GLA_DECAY) {
      const auto decay = [&](float x) { return gla_decay(l, x); };
      store8(g.f0 + row * g.ldo + n, each(lo + b[0], decay), each(hi + b[1], decay));
    } else {
      static_assert(EPI == EPI_LOGITS, "every epilogue has its place");
      store8(g.f0 + row * g.ldo + n, lo, hi);
    }
  }
};

// ---- tiles ----
// A tile is BM tokens x BN weight rows, BK columns a step; a wave owns WM x WN of it and takes all columns, one after the other.
// LOADERS: waves besides that request stages and multiply nothing.
template <int BM_, int BN_, int BK_, int WM_, int WN_, int WAVES_, int STAGES_, int LOADERS_ = 0>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, kStages = STAGES_, kLoaders = LOADERS_, kThreadCount = (WAVES_ + LOADERS_) * 64;
  static constexpr int kWavesM = BM / WM, kWavesN = BN / WN;
  static constexpr int kTm = WM / 16, kTn = WN / 16;     // a wave's fragments
  static constexpr int kRow = BK / 8;                                           // a row of a step: units of 16 bytes
  static constexpr int kUnits = (BM + BN) * kRow;
  static constexpr bool kSplits = kTn * kTm <= 12;                              // may be cut along K, with an fp32 side
  static constexpr int kSteps = BK / 32;                                        // matrix steps of a step
  static constexpr int kOutUnits = BM * BN / 4, kPasses = kOutUnits > kStages * kUnits ? 2 : 1;
  static constexpr int kLds = kStages * kUnits > kOutUnits / kPasses ? kStages * kUnits : kOutUnits / kPasses;
  static_assert(kUnits % 64 == 0 && kSteps >= 1 && kTm % kPasses == 0 && kLds * 16 < 160 * 1024, "a tile's sizes");
  static_assert(kWavesM * kWavesN == WAVES_, "the waves cover the tile");
};

// Workgroups go to the XCDs in turn; here an XCD gets a run of neighbouring tiles, which share rows through its L2.
__device__ __forceinline__ int xcd_order(int id, int total) {
  const int per = total >> 3, rest = total & 7, xcd = id & 7;
  return xcd * per + min(xcd, rest) + (id >> 3);
}

// Of a product cut along K every part leaves its sums; the part that arrives last adds them up in their order and goes on
// (true), the others are done.  `sums`: COUNT quads a thread.
template <int COUNT, int THREADS>
__device__ __forceinline__ bool sum_parts(const GemmArgs& g, int tile, int part, f32x4 (&sums)[COUNT], int* last) {
  const int tid = threadIdx.x;
  // Device-coherent units of 16 bytes (sc1); a line is read once in a launch, behind its writer's ticket.
  constexpr int kCoherent = 16;
  float* all = g.partial + static_cast<size_t>(tile) * g.splits * COUNT * THREADS * 4;
  const auto unit = __builtin_amdgcn_make_buffer_rsrc(all, 0, -1, 0x00027000);
  auto at = [&](int p, int i) { return ((p * COUNT + i) * THREADS + tid) * 16; };
#pragma unroll
  for (int i = 0; i < COUNT; ++i) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, sums[i]), unit, at(part, i), 0, kCoherent);
  release_stores();
  __syncthreads();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(g.tickets + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = before == g.splits - 1;
    if (before == g.splits - 1) st_shared32(g.tickets + tile, 0);       // for the next product
  }
  __syncthreads();
  if (!*last) return false;
#pragma unroll
  for (int i = 0; i < COUNT; ++i) sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int kBatch = COUNT <= 8 ? 4 : 2;      // parts asked for together
  for (int p = 0; p < g.splits; p += kBatch) {
    v4u r[kBatch][COUNT];
#pragma unroll
    for (int b = 0; b < kBatch; ++b)
#pragma unroll
      for (int i = 0; i < COUNT; ++i) r[b][i] = __builtin_amdgcn_raw_buffer_load_b128(unit, at(min(p + b, g.splits - 1), i), 0, kCoherent);
#pragma unroll
    for (int b = 0; b < kBatch; ++b)
      if (p + b < g.splits)
#pragma unroll
        for (int i = 0; i < COUNT; ++i) sums[i] += __builtin_bit_cast(f32x4, r[b][i]);
  }
  return true;
}

// The first launch of a portion whose products are cut: a workspace may have held something else since the one before, and a ticket that is not
// zero would leave a product without its last part.
__global__ __launch_bounds__(kPfThreads) void clear_tickets(int32_t* tickets, int count) {
  for (int i = threadIdx.x; i < count; i += kPfThreads) tickets[i] = 0;
}

// All streams of the residual for quads id, id + step, .. of a tile, `BATCH` at a time: the next batch's streams are asked for before this one's are mixed, the first
// one's (`begin`) ahead of the products' exchange where registers allow.  Few workgroups make it a chain of trips to memory, many are bound by its bytes (us, one
// quad at a time with coefficients read among the stores -> now: 200 x 2048 x 64 on tiles of 64 x 128 in fp32 22.5 -> 14.9; 1531 x 2048 x 2048 on Turns96 45 -> 34).
template <int BATCH, int STREAMS>
struct ResidualQuads {
  const GemmArgs& g;
  f32x4 old[BATCH][STREAMS];

  template <class At>
  __device__ __forceinline__ void load(f32x4 (&to)[BATCH][STREAMS], int id, int total, int step, At&& at) const {
    const int S = g.streams, D = g.width;
#pragma unroll
    for (int b = 0; b < BATCH; ++b) {
      int m, n;
      if (id + b * step >= total || !at(id + b * step, m, n)) continue;
      const float* x = g.f0 + static_cast<size_t>(m) * S * D + n;
#pragma unroll
      for (int s = 0; s < STREAMS; ++s)
        if (s < S) to[b][s] = read4(x + static_cast<size_t>(s) * D);
    }
  }
  template <class At>
  __device__ __forceinline__ void begin(int id, int total, int step, At&& at) { load(old, id, total, step, at); }
  template <class At, class Value>
  __device__ __forceinline__ void run(int id, int total, int step, At&& at, Value&& value) {
    const QmkHybridLayer& l = g.layer;
    const int S = g.streams, D = g.width;
    // (Said to be constant: read among the stores, a coefficient would wait for all stores before it.)
    ConstFloat *hc = (ConstFloat*)(l.hc + (g.down ? S * (S + 2) : 0)), *next = (ConstFloat*)g.next;
#pragma unroll 1
    for (; id < total; id += BATCH * step) {
      f32x4 ahead[BATCH][STREAMS];
      load(ahead, id + BATCH * step, total, step, at);
#pragma unroll
      for (int b = 0; b < BATCH; ++b) {
        int m, n;
        if (id + b * step < total && at(id + b * step, m, n)) {
          const f32x4 v = value(id + b * step);
          float* x = g.f0 + static_cast<size_t>(m) * S * D + n;
          f32x4 u = {};
#pragma unroll
          for (int t = 0; t < STREAMS; ++t) {
            if (t < S) {
              f32x4 now = v * hc[S + t];
#pragma unroll
              for (int s = 0; s < STREAMS; ++s)
                if (s < S) now += old[b][s] * hc[2 * S + s * S + t];
              store4(x + static_cast<size_t>(t) * D, now);
              u += now * next[t];
            }
          }
          store4(g.f1 + static_cast<size_t>(m) * D + n, u);
        }
      }
#pragma unroll
      for (int b = 0; b < BATCH; ++b)
#pragma unroll
        for (int s = 0; s < STREAMS; ++s) old[b][s] = ahead[b][s];
    }
  }
};

// A wave's accumulators -> epilogue, through its own part of LDS (quads of a row exchanged by its number): a lane then has eight neighbouring outputs of one
// token, the same eight of every token it takes, and the lanes of a token write side by side (us, four outputs at a time with their columns worked out for each, by the whole
// workgroup -> so: 2048 x 16384 x 2048 with gate and up 151 -> 141, 1531 x 16384 x 2048 129 -> 119).  Unit LDS of the array is one word beside it.  (A kernel has one LDS
// array: with two, this compiler waits for all requests before every read of the main loop, which costs half of the rate.)
template <class T, class S, int LDS, int BATCH = 1>
__device__ __forceinline__ void finish_tile(const GemmArgs& g, int group, int tile, int part, int m0, int n0, int N, v4u* lds, f32x4 (&acc)[S::kTn][S::kTm]) {
  constexpr int kQuads = S::WN / 4, kPassM = S::WM / S::kPasses, kTm = S::kTm, kGroups = S::WN / 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % S::kWavesM, wn = wave / S::kWavesM;
  f32x4 sums[S::kTn * kTm];
  constexpr int kRowQuads = S::BN / 4, kRows = S::BM / S::kPasses, kFewStreams = BATCH == 1 ? kMaxStreams : 4;
  auto residual_at = [&](int pass) {
    return [=, &g](int id, int& m, int& n) {
      const int r = id / kRowQuads;
      m = m0 + r / kPassM * S::WM + pass * kPassM + r % kPassM;
      n = n0 + id % kRowQuads * 4;
      return m < g.M && n < N;
    };
  };
  // (The first batch ahead of the sums, where registers allow.)
  constexpr bool kEarly = BATCH >= 4;
  ResidualQuads<BATCH, kFewStreams> early{g};
  const bool few_streams = g.epi == EPI_RESIDUAL && g.streams <= kFewStreams;
  if (kEarly && few_streams) early.begin(tid, kRows * kRowQuads, S::kThreadCount, residual_at(0));
  const bool multiplies = S::kLoaders == 0 || wave < S::kWavesM * S::kWavesN;
  __syncthreads();
#pragma unroll
  for (int c = 0; c < S::kTn * kTm; ++c) sums[c] = acc[c / kTm][c % kTm];
  if constexpr (S::kSplits && sizeof(T) == 4)
    if (g.splits > 1 && !sum_parts<S::kTn * kTm, S::kThreadCount>(g, tile, part, sums, reinterpret_cast<int*>(lds + LDS))) return;
  f32x4 *all = reinterpret_cast<f32x4*>(lds), *out = all + wave * kPassM * kQuads;
  auto place = [](int r, int quad) { return r * kQuads + (quad ^ (r & ((kQuads & -kQuads) - 1) & 15)); };      // (within a power of two that divides a row)
  const int column = n0 + wn * S::WN;
  // (Epilogues that together grow much longer keep this compiler from unrolling the passes, which costs a third of a product's rate; passes that share their
  // code cost 2 to 6 %.)
#pragma unroll
  for (int pass = 0; pass < S::kPasses; ++pass) {
    const int first = m0 + wm * S::WM + pass * kPassM;
#pragma unroll
    for (int i = 0; i < kTm / S::kPasses; ++i)
#pragma unroll
      for (int j = 0; j < S::kTn; ++j) {
        const int r = i * 16 + (lane & 15), quad = j * 4 + (lane >> 4);
        if (multiplies) out[place(r, quad)] = sums[j * kTm + pass * (kTm / S::kPasses) + i];
      }
    __builtin_amdgcn_wave_barrier();
    auto rows = [&](auto epi) {
      constexpr int kEachTime = 64 / kGroups;      // tokens (of 96 columns five, by 60 lanes)
      const int n = column + lane % kGroups * 8;
      if (n >= N || lane >= kEachTime * kGroups || !multiplies) return;
      const Epilogue<T, decltype(epi)::value> put(g, group, n);
      const int end = min(kPassM, g.M - first);
#pragma unroll 2
      for (int r = lane / kGroups; r < end; r += kEachTime) put(first + r, out[place(r, lane % kGroups * 2)], out[place(r, lane % kGroups * 2 + 1)]);
    };
    switch (g.epi) {
      case EPI_RESIDUAL: {      // the streams of a token are long runs: all waves take rows of the whole tile
        auto product = [&](int id) {
          const int r = id / kRowQuads, q = id % kRowQuads, owner = q / kQuads * S::kWavesM + r / kPassM;
          return all[owner * kPassM * kQuads + place(r % kPassM, q % kQuads)];
        };
        __syncthreads();
        if (few_streams) {
          if constexpr (kEarly) {
            if (pass > 0) early.begin(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass));
            early.run(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass), product);
          } else {
            ResidualQuads<BATCH, kFewStreams> few{g};
            few.begin(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass));
            few.run(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass), product);
          }
        } else if constexpr (kFewStreams < kMaxStreams) {
          ResidualQuads<1, kMaxStreams> many{g};
          many.begin(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass));
          many.run(tid, kRows * kRowQuads, S::kThreadCount, residual_at(pass), product);
        }
        __syncthreads();
        break;
      }
#define QMK_EPILOGUE(EPI) case EPI: rows(std::integral_constant<int, EPI>{}); break;
      QMK_EPILOGUE(EPI_STORE)
      QMK_EPILOGUE(EPI_STORE_VALUES)
      QMK_EPILOGUE(EPI_RGLRU_IN)
      QMK_EPILOGUE(EPI_LRU_GATES)
      QMK_EPILOGUE(EPI_LATENT_IN)
      QMK_EPILOGUE(EPI_GEGLU)
      QMK_EPILOGUE(EPI_WKV_IN)
      QMK_EPILOGUE(EPI_WKV_DECAY)
      QMK_EPILOGUE(EPI_LOGITS)
      QMK_EPILOGUE(EPI_CAPPED_LOGITS)
      QMK_EPILOGUE(EPI_ADD)
      QMK_EPILOGUE(EPI_ATTENTION_IN)
      QMK_EPILOGUE(EPI_DELTA_IN)
      QMK_EPILOGUE(EPI_DELTA_DECAY)
      QMK_EPILOGUE(EPI_SIGMOID)
      QMK_EPILOGUE(EPI_GLA_IN)
      QMK_EPILOGUE(EPI_GLA_DECAY)
#undef QMK_EPILOGUE
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Which part of the product a workgroup takes.
struct Place {
  int group, tile, part, m0, n0, N, first, steps;
};
template <class S>
__device__ __forceinline__ Place place_of(const GemmArgs& g) {
  Place p;
  p.group = blockIdx.z;
  p.N = p.group == g.groups - 1 ? g.last_n : g.N;
  const int id = xcd_order(blockIdx.x, gridDim.x), tiles_m = (g.M + S::BM - 1) / S::BM, tile = id / g.splits;
  p.part = id % g.splits;
  p.m0 = tile % tiles_m * S::BM;
  p.n0 = tile / tiles_m * S::BN;
  p.tile = p.group * (gridDim.x / g.splits) + tile;
  const int all = (g.K + S::BK - 1) / S::BK;
  p.first = all * p.part / g.splits;
  p.steps = all * (p.part + 1) / g.splits - p.first;
  return p;
}

// Until at most `n` of this wave's vector-memory requests are outstanding and none of its LDS reads.
template <int n>
__device__ __forceinline__ void wait_outstanding() {
  static_assert(n >= 0 && n < 64, "six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(n) : "memory");
}

// Until at most `n` of this wave's vector-memory requests are outstanding and none of its LDS reads, said with the builtin: the compiler's own waits take account of it.
template <int n>
__device__ __forceinline__ void wait_known() {
  static_assert(n >= 0 && n < 64, "six bits");
  __builtin_amdgcn_s_waitcnt((n & 15) | 7 << 4 | (n >> 4) << 14);
}

// The tiles of a step, bf16: memory -> LDS without passing through registers, kStages buffers deep.  A row's units are exchanged
// by its number on the memory side (the LDS side of such a load is one run of 64 units per wave), so that fragment reads do
// not conflict.  A lane's places are offsets of 32 bits that stay, and one scalar moves on, so that a request is one instruction (with pointers that move on
// it is two more).
template <class S, int PARTS = 1, int ISSUERS = S::kThreadCount>      // PARTS: of the tokens' side; ISSUERS: threads that request
struct Stages {
  static constexpr int kRowsA = S::BM * PARTS, kUnitsA = kRowsA * S::kRow, kUnits = (kRowsA + S::BN) * S::kRow, kLoads = (kUnits + ISSUERS - 1) / ISSUERS;
  static constexpr int kLastWaves = (kUnits - (kLoads - 1) * ISSUERS) / 64;      // waves that take part in a stage's last load
  static_assert(kUnits % 64 == 0 && kUnitsA % 64 == 0, "a wave's loads are whole, and of one side");
  static_assert(PARTS == 1 || S::BM * S::kRow % ISSUERS == 0, "a load is of one part");
  using Lds = __attribute__((address_space(3))) v4u;      // said outright: a pointer kept in a struct may become a generic one
  __amdgpu_buffer_rsrc_t a[PARTS], w;      // from the tile's first rows on: they are far less than 4 GB
  uint32_t from[kLoads], at = 0;           // this thread's places in a stage: unit i * threads + tid, tokens first; columns of the stage
  Lds* lds;
  int wave;

  static __device__ __forceinline__ int exchange(int r) { return S::kRow == 4 ? (r >> 1) & 3 : r & 7; }
  __device__ __forceinline__ Stages(const GemmArgs& g, const Place& p, v4u* buffers, int wave_number) : lds((Lds*)buffers), wave(wave_number) {
    auto rows = [&](const void* base, long long skip, int row, int ld) {
      const u16* first = static_cast<const u16*>(base) + skip + static_cast<size_t>(row) * ld + p.first * S::BK;
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(first), 0, -1, 0x00027000);
    };
#pragma unroll
    for (int part = 0; part < PARTS; ++part) a[part] = rows(g.a, p.group * g.a_step + (PARTS == 1 ? 0 : part * g.a_part), p.m0, g.lda);
    w = rows(g.w, p.group * g.w_step, p.n0, g.ldw);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int u = i * ISSUERS + (ISSUERS == S::kThreadCount ? static_cast<int>(threadIdx.x) : wave * 64 + static_cast<int>(threadIdx.x & 63)), r = u / S::kRow, c = ((u % S::kRow) ^ exchange(r)) * 8;
      from[i] = (r < kRowsA ? min(PARTS == 1 ? r : r % S::BM, g.M - 1 - p.m0) * g.lda + c : min(r - kRowsA, p.N - 1 - p.n0) * g.ldw + c) * 2;
    }
  }
  __device__ __forceinline__ void issue(int buf) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if (i == kLoads - 1 && kLastWaves * 64 < ISSUERS && wave >= kLastWaves) continue;
      auto* dst = (__attribute__((address_space(3))) uint32_t*)(lds + buf * kUnits + i * ISSUERS + wave * 64);
      const bool tokens = (i + 1) * ISSUERS <= kUnitsA || (i * ISSUERS < kUnitsA && i * ISSUERS + wave * 64 < kUnitsA);
      constexpr int kPart = S::BM * S::kRow;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(tokens ? a[PARTS == 1 ? 0 : min(i * ISSUERS / kPart, PARTS - 1)] : w, dst, 16, from[i], at, 0, 0);
    }
    at += S::BK * 2;
  }
  // Until at most `stages` stages of this wave's are outstanding.
  template <int stages>
  __device__ __forceinline__ void wait() const {
    if (kLastWaves * 64 == ISSUERS || wave < kLastWaves) wait_known<stages * kLoads>();
    else wait_known<stages * (kLoads - 1)>();
  }
  __device__ __forceinline__ void fragments(int buf, int q, int wm, int wn, Frag<u16> (&fa)[PARTS][S::kTm], Frag<u16> (&fw)[S::kTn]) const {
    const Lds *la = lds + buf * kUnits, *lw = la + kRowsA * S::kRow;
    const int row = threadIdx.x & 15;
    auto frag = [](const Lds* at) { return Frag<u16>{__builtin_bit_cast(bf16x8_t, *at)}; };
#pragma unroll
    for (int j = 0; j < S::kTn; ++j) {
      const int r = wn * S::WN + j * 16 + row;
      fw[j] = frag(lw + r * S::kRow + (q ^ exchange(r)));
    }
    static_assert(PARTS == 1 || S::BM % 16 == 0, "rows of every part are exchanged alike");
#pragma unroll
    for (int part = 0; part < PARTS; ++part)
#pragma unroll
      for (int i = 0; i < S::kTm; ++i) {
        const int r = part * S::BM + wm * S::WM + i * 16 + row;
        fa[part][i] = frag(la + r * S::kRow + (q ^ exchange(r)));
      }
  }
};

template <class S, int PARTS>
__device__ __forceinline__ void multiply(const Frag<u16> (&fa)[PARTS][S::kTm], const Frag<u16> (&fw)[S::kTn], f32x4 (&acc)[S::kTn][S::kTm]) {
#pragma unroll
  for (int i = 0; i < S::kTm; ++i) {
    if constexpr (PARTS == 1) {
#pragma unroll
      for (int j = 0; j < S::kTn; ++j) acc[j][i] = mma(fw[j], fa[0][i], acc[j][i]);
    } else {      // 32 columns by themselves, small parts first, then one rounded addition
      f32x4 t[S::kTn] = {};
#pragma unroll
      for (int part = PARTS - 1; part >= 0; --part)
#pragma unroll
        for (int j = 0; j < S::kTn; ++j) t[j] = mma(fw[j], fa[part][i], t[j]);
#pragma unroll
      for (int j = 0; j < S::kTn; ++j) acc[j][i] += t[j];
    }
  }
}

// An infinite value on the bf16 side makes products with those parts of a finite value that are zero undefined, where the product with the whole
// value is infinite.  A sum that came out undefined is therefore taken again, of first parts alone, which are zero or not finite where the
// values are; nothing else can have made it so that does not make it so again.  `a`, `w`: fragments of first parts, tile i and 32 columns from k.
template <class S, class A, class W>
__device__ __forceinline__ void resolve_undefined(const Place& p, f32x4 (&acc)[S::kTn][S::kTm], A&& a, W&& w) {
#pragma unroll
  for (int j = 0; j < S::kTn; ++j)
#pragma unroll
    for (int i = 0; i < S::kTm; ++i) {
      f32x4& v = acc[j][i];
      if (__builtin_expect(__any(v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3]), 0)) {
        f32x4 t = {};
#pragma unroll 1
        for (int k = p.first * S::BK; k < (p.first + p.steps) * S::BK; k += 32) t = mma(w(j, k), a(i, k), t);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] != v[e] ? t[e] : v[e];
      }
    }
}

template <class S>
__device__ __forceinline__ void resolve_undefined(const GemmArgs& g, const Place& p, int wm, int wn, f32x4 (&acc)[S::kTn][S::kTm]) {
  const int lane = threadIdx.x & 63;
  const u16 *a = static_cast<const u16*>(g.a) + p.group * g.a_step + (lane >> 4) * 8, *w = static_cast<const u16*>(g.w) + p.group * g.w_step + (lane >> 4) * 8;
  resolve_undefined<S>(
      p, acc, [&](int i, int k) { return load_frag(a + static_cast<size_t>(min(p.m0 + wm * S::WM + i * 16 + (lane & 15), g.M - 1)) * g.lda + k); },
      [&](int j, int k) { return load_frag(w + static_cast<size_t>(min(p.n0 + wn * S::WN + j * 16 + (lane & 15), p.N - 1)) * g.ldw + k); });
}

// out[m][n] = sum_k a[m][k] w[n][k], bf16 x bf16, K a multiple of BK.  The weights are the matrix instruction's first operand,
// so a lane ends up with four consecutive outputs of one token.  Two to eight waves; several workgroups share a CU where LDS has room.
template <class T, class S>
__global__ __launch_bounds__(S::kThreadCount, S::kThreadCount == 512 ? 4 : 1) void gemm_direct(const GemmArgs g) {
  constexpr int kAhead = S::kStages - 1;
  __shared__ __align__(16) v4u lds[S::kLds + 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % S::kWavesM, wn = wave / S::kWavesM;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  Stages<S> stages(g, p, lds, wave);
  f32x4 acc[S::kTn][S::kTm] = {};
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
    if (s < p.steps) stages.issue(s);
  int buf = 0;
  for (int s = 0; s < p.steps; ++s) {
    // Everything up to this step's stage has landed; the barrier makes that true of every wave's part, and says that the
    // buffer filled next is no longer read.
    if (s + kAhead - 1 < p.steps) stages.template wait<kAhead - 1>();
    else wait_outstanding<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + kAhead < p.steps) stages.issue(buf == 0 ? S::kStages - 1 : buf - 1);
#pragma unroll
    for (int kk = 0; kk < S::kSteps; ++kk) {
      Frag<u16> fa[1][S::kTm], fw[S::kTn];
      stages.fragments(buf, kk * 4 + (lane >> 4), wm, wn, fa, fw);
      multiply<S, 1>(fa, fw, acc);
    }
    buf = buf + 1 == S::kStages ? 0 : buf + 1;
  }
  finish_tile<T, S, S::kLds, 2>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}

// The same for the fewest tokens, whose workgroups have few waves that multiply: on their chain of products, fragments and barriers requests for stages take as long
// as the products, so other waves make them.  A stage has landed for everybody behind the barrier that its loaders reach when it has landed for them; fragments of 32
// columns are read while the 32 before are multiplied (us, the mean of 43 x 2048 x 2048 and x 6144 with the residual's streams, inside a portion: 12.0 with two waves that do both -> 10.8; four
// loaders 10.9, three or six stages 11.5 and 11.1; the same with all weights in the last cache, so what is left is not memory's rate).
template <class T, class S>
__global__ __launch_bounds__(S::kThreadCount, 1) void gemm_few(const GemmArgs g) {
  constexpr int kAhead = S::kStages - 1, kMultipliers = S::kWavesM * S::kWavesN;
  __shared__ __align__(16) v4u lds[S::kLds + 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % S::kWavesM, wn = wave / S::kWavesM % S::kWavesN;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  Stages<S, 1, S::kLoaders * 64> stages(g, p, lds, wave - kMultipliers);
  f32x4 acc[S::kTn][S::kTm] = {};
  auto barrier = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  if (wave >= kMultipliers) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (s < p.steps) stages.issue(s);
    int buf = S::kStages - 1;
    for (int s = 0; s < p.steps; ++s) {
      if (s + kAhead - 1 < p.steps) stages.template wait<kAhead - 1>();
      else wait_outstanding<0>();
      barrier();      // stage s has landed, and stage s - 1 is no longer read
      if (s + kAhead < p.steps) stages.issue(buf);
      buf = buf + 1 == S::kStages ? 0 : buf + 1;
    }
  } else {
    struct Fragments {
      Frag<u16> a[1][S::kTm], w[S::kTn];
    } f[2];
    int buf = 0;
    for (int s = 0; s < p.steps; ++s) {
      wait_known<63>();      // (the last fragments of the step before)
      barrier();
      stages.fragments(buf, lane >> 4, wm, wn, f[0].a, f[0].w);
#pragma unroll
      for (int kk = 0; kk < S::kSteps; ++kk) {
        if (kk + 1 < S::kSteps) stages.fragments(buf, (kk + 1) * 4 + (lane >> 4), wm, wn, f[(kk + 1) & 1].a, f[(kk + 1) & 1].w);
        multiply<S, 1>(f[kk & 1].a, f[kk & 1].w, acc);
      }
      buf = buf + 1 == S::kStages ? 0 : buf + 1;
    }
  }
  finish_tile<T, S, S::kLds, 2>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}

// Scheduling of a block of matrix instructions: one LDS read ahead of each of the first, the requests for a stage among the rest.
template <int PRODUCTS, int READS, int REQUESTS>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < READS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    if (i < PRODUCTS) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
  }
  constexpr int kEach = REQUESTS > 0 && PRODUCTS - READS >= 2 * REQUESTS ? 2 : 1;
#pragma unroll
  for (int i = 0; i < REQUESTS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    if (READS + i * kEach < PRODUCTS) __builtin_amdgcn_sched_group_barrier(0x008, kEach, 0);
  }
}

// The same as gemm_direct for larger tiles of bf16, one workgroup a CU or two.  What bounds them is LDS: a tile's rows are read by every wave that shares them,
// 128 bytes a cycle, so waves take 64 x 64 where they can, and no wave may wait for its reads.  32 columns are multiplied while the fragments of the next 32 are
// read into a second set of registers; one barrier a stage lies ahead of the first reads of the next one, where everybody has read the last of this one: its
// buffer is filled again at once, kStages stages ahead.  (Launch bounds of eight waves also for four: with more registers to give away this compiler keeps
// accumulators in the other half of the file and moves them at every step.)
template <class S, int PARTS>
constexpr int kPipeLds = S::kStages * Stages<S, PARTS>::kUnits > S::kLds ? S::kStages * Stages<S, PARTS>::kUnits : S::kLds;
template <class T, class S, int PARTS>
__device__ __forceinline__ void pipe_tile(const GemmArgs& g, v4u* lds) {
  static_assert(S::kSteps % 2 == 0 && S::kStages >= 2, "pairs of matrix steps a stage");
  constexpr int kDeep = S::kStages, kProducts = PARTS * S::kTm * S::kTn, kReads = PARTS * S::kTm + S::kTn, kRequests = Stages<S, PARTS>::kLoads, kLds = kPipeLds<S, PARTS>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % S::kWavesM, wn = wave / S::kWavesM;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  Stages<S, PARTS> stages(g, p, lds, wave);
  auto barrier = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // Products of parts add every other 32 columns to a sum of their own: half as many rounded additions follow one another (error
  // against 64 bits, logits and states, mean of three prompts, with more cuts along K and one sum -> so: 390 tokens of the 1b shape 1.46e-6 -> 1.41e-6, 33 of the 2b shape 3.7e-6 -> 3.5e-6).
  constexpr int kSums = PARTS > 1 ? 2 : 1;
  f32x4 sums[kSums][S::kTn][S::kTm] = {};
  struct Fragments {
    Frag<u16> a[PARTS][S::kTm], w[S::kTn];
  } f[2];
#pragma unroll
  for (int s = 0; s < kDeep; ++s)
    if (s < p.steps) stages.issue(s);
  if (kDeep <= p.steps) stages.template wait<kDeep - 1>();
  else wait_known<0>();
  barrier();
  stages.fragments(0, lane >> 4, wm, wn, f[0].a, f[0].w);
  int buf = 0;
  auto step = [&](auto more) {
    constexpr bool MORE = decltype(more)::value;
    wait_known<63>();      // (the first fragments)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk + 1 < S::kSteps; ++kk) {
      Fragments &now = f[kk & 1], &next = f[(kk + 1) & 1];
      if (kk > 0) {
        wait_known<63>();
        __builtin_amdgcn_sched_barrier(0);
      }
      stages.fragments(buf, (kk + 1) * 4 + (lane >> 4), wm, wn, next.a, next.w);
      multiply<S, PARTS>(now.a, now.w, sums[kk % kSums]);
      if constexpr (MORE) interleave<kProducts, kReads, 0>();
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MORE) stages.template wait<kDeep - 2>();
    else wait_known<0>();
    barrier();
    const int next = buf + 1 == S::kStages ? 0 : buf + 1;
    stages.fragments(next, lane >> 4, wm, wn, f[0].a, f[0].w);      // (behind the last stage: of a buffer that is there, for nobody)
    if constexpr (MORE) stages.issue(buf);
    multiply<S, PARTS>(f[1].a, f[1].w, sums[kSums - 1]);
    if constexpr (MORE) interleave<kProducts, kReads, kRequests>();
    __builtin_amdgcn_sched_barrier(0);
    buf = next;
  };
  int s = 0;
  for (; s + kDeep < p.steps; ++s) step(std::true_type{});
  for (; s < p.steps; ++s) step(std::false_type{});
  auto& acc = sums[0];
  if constexpr (PARTS > 1) {
#pragma unroll
    for (int j = 0; j < S::kTn; ++j)
#pragma unroll
      for (int i = 0; i < S::kTm; ++i) acc[j][i] += sums[kSums - 1][j][i];
    resolve_undefined<S>(g, p, wm, wn, acc);
  }
  finish_tile<T, S, kLds, 4>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}
template <class T, class S, int PARTS = 1>
__global__ __launch_bounds__(512, 2) void gemm_pipe(const GemmArgs g) {
  __shared__ __align__(16) v4u lds[kPipeLds<S, PARTS> + 1];
  pipe_tile<T, S, PARTS>(g, lds);
}
// Two products that need nothing of each other.
struct GemmPair {
  GemmArgs g[2];
};
template <class T, class S>
__global__ __launch_bounds__(512, 2) void gemm_pipe_pair(const GemmPair pair) {
  __shared__ __align__(16) v4u lds[kPipeLds<S, 1> + 1];
  pipe_tile<T, S, 1>(pair.g[blockIdx.y], lds);
}

// The same with eight waves, one workgroup a CU.  Two waves share a SIMD's matrix unit, and the halves of the workgroup take
// turns: while one multiplies, the other reads its next fragments; a barrier ends each turn, and the second half starts one
// turn late.
template <class T, class S>
__global__ __launch_bounds__(512, 2) void gemm_turns(const GemmArgs g) {
  static_assert(S::kThreadCount == 512 && S::kStages >= 3, "one turn a step, the next stage has landed before it");
  constexpr int kAhead = S::kStages - 1;
  __shared__ __align__(16) v4u lds[S::kLds + 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % S::kWavesM, wn = wave / S::kWavesM;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  Stages<S> stages(g, p, lds, wave);
  auto barrier = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  f32x4 acc[S::kTn][S::kTm] = {};
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
    if (s < p.steps) stages.issue(s);
  if (kAhead - 1 < p.steps) stages.template wait<kAhead - 1>();
  else wait_outstanding<0>();
  barrier();                       // stage 0 is there
  if (wave >= 4) barrier();
  int buf = 0;
  for (int s = 0; s < p.steps; ++s) {
    // The buffer filled here was read in step s - 1: by this half a turn ago, by the other one before the last barrier.
    if (s + kAhead < p.steps) stages.issue(buf == 0 ? S::kStages - 1 : buf - 1);
    Frag<u16> fa[S::kSteps][1][S::kTm], fw[S::kSteps][S::kTn];
#pragma unroll
    for (int kk = 0; kk < S::kSteps; ++kk) stages.fragments(buf, kk * 4 + (lane >> 4), wm, wn, fa[kk], fw[kk]);
    // Stage s + 1 has landed: a barrier lies between this wait and either half's reads of it.
    if (s + kAhead < p.steps) stages.template wait<kAhead - 1>();
    else wait_outstanding<0>();
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < S::kSteps; ++kk) multiply<S, 1>(fa[kk], fw[kk], acc);
    __builtin_amdgcn_s_setprio(0);
    barrier();
    buf = buf + 1 == S::kStages ? 0 : buf + 1;
  }
  if (wave < 4) barrier();
  finish_tile<T, S, S::kLds>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}

// ---- products with an fp32 side, and bf16 ones of any K ----
template <class T>
constexpr int kPlanes = sizeof(T) == 2 ? 1 : 3;

// BN weight rows x BM tokens a workgroup, four waves as 2 x 2, 64 columns a step, through registers.  LDS holds
// 16-byte units of bf16, planes one after the other, a row's units exchanged by its number.
template <class TA, class TW, class T, int BM_, int BN_, int BUFFERS>
__global__ __launch_bounds__(kPfThreads) void gemm(const GemmArgs g) {
  using S = Tile<BM_, BN_, 64, BM_ / 2, BN_ / 2, 4, 2>;
  constexpr int BM = S::BM, BN = S::BN, kBK = S::BK, kTm = S::kTm, kTn = S::kTn;
  constexpr int kPa = kPlanes<TA>, kPw = kPlanes<TW>, kUnitsA = BM * 8, kUnitsW = BN * 8;
  constexpr int kRunsA = kUnitsA / kPfThreads, kRunsW = kUnitsW / kPfThreads;       // runs of eight columns a thread stages
  constexpr int kStage = kPa * kUnitsA + kPw * kUnitsW, kLds = BUFFERS * kStage > S::kOutUnits ? BUFFERS * kStage : S::kOutUnits;
  __shared__ __align__(16) v4u lds[kLds + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  const TA* a = static_cast<const TA*>(g.a) + p.group * g.a_step;
  const TW* w = static_cast<const TW*>(g.w) + p.group * g.w_step;

  v4u ra[kRunsA][sizeof(TA) / 2], rw[kRunsW][sizeof(TW) / 2];
  auto fetch = [&](int k0) {
    auto side = [&](auto* base, auto& r, int runs, int row0, int rows, long long ld) {
      constexpr int kUnit = 16 / sizeof(*base), kEach = 8 / kUnit;
#pragma unroll
      for (int i = 0; i < runs; ++i) {
        const int id = i * kPfThreads + tid, k = k0 + id % 8 * 8;
        const auto* from = base + static_cast<size_t>(min(row0 + id / 8, rows - 1)) * ld + k;
#pragma unroll
        for (int e = 0; e < kEach; ++e)
          r[i][e] = k + e * kUnit < g.K ? *reinterpret_cast<const v4u*>(from + e * kUnit) : v4u{0u, 0u, 0u, 0u};
      }
    };
    side(a, ra, kRunsA, p.m0, g.M, g.lda);
    side(w, rw, kRunsW, p.n0, p.N, g.ldw);
  };
  auto stash = [&](int buf) {
    auto side = [&](auto tag, auto& r, int runs, v4u* to, int units) {
      using E = decltype(tag);
#pragma unroll
      for (int i = 0; i < runs; ++i) {
        const int id = i * kPfThreads + tid, row = id / 8, place = row * 8 + (id % 8 ^ (row & 7));
        if constexpr (sizeof(E) == 2) {
          to[place] = r[i][0];
        } else {
          v4u plane[3];
          const uint32_t bits[8] = {r[i][0].x, r[i][0].y, r[i][0].z, r[i][0].w, r[i][1].x, r[i][1].y, r[i][1].z, r[i][1].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            uint32_t t[3];
            split2(__uint_as_float(bits[2 * e]), __uint_as_float(bits[2 * e + 1]), t);
#pragma unroll
            for (int q = 0; q < 3; ++q) plane[q][e] = t[q];
          }
#pragma unroll
          for (int q = 0; q < 3; ++q) to[q * units + place] = plane[q];
        }
      }
    };
    side(TA{}, ra, kRunsA, lds + buf * kStage, kUnitsA);
    side(TW{}, rw, kRunsW, lds + buf * kStage + kPa * kUnitsA, kUnitsW);
  };
  f32x4 acc[kTn][kTm] = {};
  if (p.steps > 0) {
    fetch(p.first * kBK);
    stash(0);
  }
  __syncthreads();
  for (int s = 0; s < p.steps; ++s) {
    const v4u *la = lds + (BUFFERS == 2 ? s & 1 : 0) * kStage, *lw = la + kPa * kUnitsA;
    if (s + 1 < p.steps) fetch((p.first + s + 1) * kBK);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int q = kk * 4 + (lane >> 4);
      Frag<u16> fa[kPa][kTm], fw[kPw][kTn];
#pragma unroll
      for (int pl = 0; pl < kPa; ++pl)
#pragma unroll
        for (int i = 0; i < kTm; ++i) {
          const int r = wm * S::WM + i * 16 + (lane & 15);
          fa[pl][i] = load_frag(reinterpret_cast<const u16*>(la + pl * kUnitsA + r * 8 + (q ^ (r & 7))));
        }
#pragma unroll
      for (int pl = 0; pl < kPw; ++pl)
#pragma unroll
        for (int j = 0; j < kTn; ++j) {
          const int r = wn * S::WN + j * 16 + (lane & 15);
          fw[pl][j] = load_frag(reinterpret_cast<const u16*>(lw + pl * kUnitsW + r * 8 + (q ^ (r & 7))));
        }
      static_assert(kPa == 1 || kPw == 1, "one side is bf16");
#pragma unroll
      for (int j = 0; j < kTn; ++j)
#pragma unroll
        for (int i = 0; i < kTm; ++i) {
          if constexpr (kPa * kPw == 1) {
            acc[j][i] = mma(fw[0][j], fa[0][i], acc[j][i]);
          } else {      // 32 columns by themselves, small parts first, then one rounded addition
            f32x4 t = {};
#pragma unroll
            for (int pl = 2; pl >= 0; --pl) t = mma(fw[kPw == 1 ? 0 : pl][j], fa[kPa == 1 ? 0 : pl][i], t);
            acc[j][i] += t;
          }
        }
    }
    if (BUFFERS == 1) __syncthreads();
    if (s + 1 < p.steps) stash(BUFFERS == 2 ? (s + 1) & 1 : 0);
    __syncthreads();
  }
  if constexpr (kPa * kPw > 1) {
    auto first_part = [&](auto* base, int row, int rows, long long ld, int k) {      // (K is a multiple of the units a row is read in)
      constexpr int kUnit = 16 / sizeof(*base);
      const auto* from = base + static_cast<size_t>(min(row, rows - 1)) * ld;
      k += (lane >> 4) * 8;
      v4u unit = {0u, 0u, 0u, 0u};
      if constexpr (kUnit == 8) {
        if (k < g.K) unit = *reinterpret_cast<const v4u*>(from + k);
      } else {
#pragma unroll
        for (int e = 0; e < 2; ++e)
          if (k + e * kUnit < g.K) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(from + k + e * kUnit);
            uint32_t lo[3], hi[3];
            split2(x[0], x[1], lo);
            split2(x[2], x[3], hi);
            unit[2 * e] = lo[0];
            unit[2 * e + 1] = hi[0];
          }
      }
      return Frag<u16>{__builtin_bit_cast(bf16x8_t, unit)};
    };
    resolve_undefined<S>(
        p, acc, [&](int i, int k) { return first_part(a, p.m0 + wm * S::WM + i * 16 + (lane & 15), g.M, g.lda, k); },
        [&](int j, int k) { return first_part(w, p.n0 + wn * S::WN + j * 16 + (lane & 15), p.N, g.ldw, k); });
  }
  finish_tile<T, S, kLds>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}

// At most 64 columns with an fp32 side: one step, where the fp32 instruction is no slower than three parts (5.1 us against 5.6 for
// 64 x 64 x 64; both are a launch and its loads).
template <class TA, class TW, class T>
__global__ __launch_bounds__(kPfThreads) void gemm_short(const GemmArgs g) {
  using S = Tile<64, 64, 64, 32, 32, 4, 4>;
  constexpr int kUnitA = 16 / sizeof(TA), kUnitW = 16 / sizeof(TW), kRowA = 64 / kUnitA, kRowW = 64 / kUnitW;
  __shared__ __align__(16) v4u lds[S::kLds + 1];
  static_assert(64 * (kRowA + kRowW) <= S::kLds, "both tiles");
  v4u *la = lds, *lw = lds + 64 * kRowA;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  const Place p = place_of<S>(g);
  if (p.n0 >= p.N) return;
  auto place = [](int r, int unit, int row_units) { return r * row_units + (unit ^ ((r & 7) * (row_units / 8))); };
  auto stage = [&](auto* from, v4u* to, int row_units, int unit, int row0, int rows, long long ld) {
    for (int id = tid; id < 64 * row_units; id += kPfThreads) {
      const int r = id / row_units, k = id % row_units * unit;
      to[place(r, id % row_units, row_units)] =
          k < g.K ? *reinterpret_cast<const v4u*>(from + static_cast<size_t>(min(row0 + r, rows - 1)) * ld + k) : v4u{0u, 0u, 0u, 0u};
    }
  };
  stage(static_cast<const TA*>(g.a) + p.group * g.a_step, la, kRowA, kUnitA, p.m0, g.M, g.lda);
  stage(static_cast<const TW*>(g.w) + p.group * g.w_step, lw, kRowW, kUnitW, p.n0, p.N, g.ldw);
  __syncthreads();
  f32x4 acc[S::kTn][S::kTm] = {};
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int q = kk * 4 + (lane >> 4);
    Frag<TA> fa[S::kTm];
#pragma unroll
    for (int i = 0; i < S::kTm; ++i) fa[i] = load_frag(reinterpret_cast<const TA*>(&la[place(wm * S::WM + i * 16 + (lane & 15), q * (kRowA / 8), kRowA)]));
#pragma unroll
    for (int j = 0; j < S::kTn; ++j) {
      const Frag<TW> fw = load_frag(reinterpret_cast<const TW*>(&lw[place(wn * S::WN + j * 16 + (lane & 15), q * (kRowW / 8), kRowW)]));
#pragma unroll
      for (int i = 0; i < S::kTm; ++i) acc[j][i] = mma(fw, fa[i], acc[j][i]);
    }
  }
  finish_tile<T, S, S::kLds>(g, p.group, p.tile, p.part, p.m0, p.n0, p.N, lds, acc);
}

// ---- which tiles ----
// (Figures here are of single launches one after another, weights from memory; inside a portion they differ by up to a fifth, qmk_hybrid_tiles.h.)
// Few tokens: weight rows of a workgroup, deep steps, since a step's barrier and reads are most of its time (us, M x N x K, 64 x 16 in steps of 64 columns, of
// 128, 32 x 16 in steps of 256: 43 x 2048 x 2048 with the residual's streams 12.2, 10.1, 9.5; 43 x 2048 x 6144 with them 26.4, 19.9, 17.3; the last one now 7.9 and 14.9, and with waves that only load a tenth less).
using Few32 = Tile<32, 16, 256, 16, 16, 2, 4, 2>;
using Few64 = Tile<64, 16, 128, 16, 16, 4, 3>;
using Wide64 = Tile<128, 64, 64, 32, 32, 8, 3>;
// Below with gemm_pipe (us, M x N x K, before -> with it: 512 x 2048 x 2048 Tiles64 14.5 -> 11.8; 43 x 5696 x 2048 Tiles32 10.7 -> 9.0; 2048 x 2048 x 2048 and x 8192 Turns128, halves of the workgroup in turns, 28.5
// and 88 -> 22.6 and 73, on four waves of 64 x 64 26 and 76; 1536 x 4096 x 8192 Tall192 119 -> 95, 2048 x 4096 x 8192 Tall256 139 -> 122).
using Tiles32 = Tile<64, 32, 64, 32, 16, 4, 6>;
using Tiles64 = Tile<64, 64, 64, 32, 32, 4, 4>;
using Turns96 = Tile<96, 128, 64, 48, 32, 8, 4>;
using Turns128 = Tile<128, 128, 64, 32, 64, 8, 4>;
// Three stages where four do not fit.
using Tall192 = Tile<192, 128, 64, 48, 64, 8, 3>;
using Tall256 = Tile<256, 128, 64, 64, 64, 8, 3>;
using Wide256 = Tile<128, 256, 64, 64, 64, 8, 3>;
// With gemm_turns: accumulators leave no registers for a second set of fragments of 64 columns, and with steps of 32 the turns are as fast (2048 x 16384 x 2048 141, gemm_pipe 143).
using Turns192 = Tile<192, 256, 32, 96, 64, 8, 4>;
using Turns256 = Tile<256, 256, 32, 128, 64, 8, 4>;
// The tokens' side in three parts, with gemm_pipe: it is what fills LDS (us, 32 x 128 in two stages without a second set of fragments -> the kind that is taken: 200 x
// 2048 x 6144 with the streams 43 -> 34, 200 x 12288 x 2048 65 -> 40, 200 x 5696 x 2048 33 -> 26, 20 x 12288 x 2048 21 -> 16).
using Parts32 = Tile<32, 128, 64, 16, 64, 4, 3>;
using Parts64 = Tile<64, 128, 64, 32, 64, 4, 3>;
using PartsWide = Tile<64, 192, 64, 32, 96, 4, 3>;

}  // namespace hybrid
}  // namespace qmk
