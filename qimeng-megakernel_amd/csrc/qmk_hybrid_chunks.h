// Recurrences of prefill that keep a state [keys][values] a head: wkv, gated linear attention, gated delta rule, in chunks of sixteen tokens on the matrix cores.
//
// Recurrence of one head, state S, decay g_t per key channel:
//   S <- g_t S,  u_t = beta_t (v_t - S^T k_t),  S <- S + k_t u_t^T,  o_t = S^T q_t        (gla: u_t = v_t)
//   wkv: o_t = (S + diag(bonus) k_t v_t^T)^T r_t ahead of S <- g_t S + k_t v_t^T
// Over a chunk that starts from S, with G_t = g_1 .. g_t and D_ts = g_{s+1} .. g_t (products, never quotients: a decay may
// be small enough for its inverse to overflow):
//   u = T v - W S,  W = T (G k)^T,  T = (I + diag(beta) A)^-1 diag(beta),  A_ts = sum_i k_t D_ts k_s  (s < t)
//   o_t = (G_t q_t)^T S + sum_{s <= t} B_ts u_s,  B_ts = sum_i q_t D_ts k_s               (wkv: G_{t-1}, D_{t-1,s}, B_tt = sum_i r_t bonus k_t)
//   S  <- G_16 S + sum_s (D_16,s k_s) u_s^T
// chunk_prepare works out everything that no state enters, for all chunks at once.  Where u is v a chunk's state is a sum that may be cut anywhere: segments of
// eight chunks are walked side by side, once from nothing for what they leave (segment_scan<.., false>), then, from the states that segment_starts puts
// together, for the outputs.  Segments lie where they do from the portion's start on whatever its length, so a token's bits do not depend on it.  The delta rule's
// chunks are walked one after the other (chunk_scan).
#pragma once

#include "qmk_hybrid_prefill.h"

namespace qmk {
namespace hybrid {

constexpr int kChunkTokens = 16;
constexpr int kChunkWaves = 4;
constexpr int kSegmentChunks = 8, kShortChunks = 16;
// Chunks of a segment.  In fp32, where orders may depend on the length, up to kShortChunks are one segment: walking them twice in halves takes longer (us, 200 tokens
// of 32 heads of 64: prepared and walked once 21.0, in halves 23.5).
template <class T>
__host__ __device__ constexpr int segment_chunks(int tokens) { return sizeof(T) == 4 && tokens <= kShortChunks * kChunkTokens ? kShortChunks : kSegmentChunks; }
// Up to so many segments put their own starts together (the same sums in the same order; a launch less, but every segment reads all before it).
constexpr int kOwnStarts = 4;

// Tiles of sixteen key channels of a head, the last ones zeros.
__host__ __device__ constexpr int chunk_tiles(int head_dim) { return head_dim <= 64 ? 4 : head_dim <= 128 ? 8 : 16; }
// Floats of one (chunk, head): per tile the fragments of G q, W and D k and the decays G over the whole chunk, then B.  A fragment is in the order the
// matrix instruction takes it: [lane][4].
__host__ __device__ constexpr int chunk_floats(int head_dim) { return chunk_tiles(head_dim) * (3 * 256 + 16) + 256; }
__host__ __device__ constexpr int chunks_of(int tokens) { return (tokens + kChunkTokens - 1) / kChunkTokens; }
__host__ __device__ constexpr int segments_of(int tokens, int chunks) { return (chunks_of(tokens) + chunks - 1) / chunks; }

enum : int { CHUNK_GLA, CHUNK_DELTA, CHUNK_WKV };
struct ChunkArgs {
  QmkHybridLayer layer;
  const float *q, *k;    // [M][ld]; delta: q alone, q, k, v ahead of the convolution
  const float* decay;    // [M][heads * dim]
  const float* beta;     // delta: [M][beta_ld]
  float* chunks;         // [chunk][head][chunk_floats]
  float* values;         // [M][value_ld] at value_at; delta: T v, [chunk][head][n / 16] fragments, written here
  float* out;            // [M][heads * n]
  float* starts;         // [segment][head][dim][n]: what the segment before leaves, then the state the segment starts from
  float* fades;          // [segment][head][dim]: decays over the segment before
  int M, heads, dim, n, ld, beta_ld, value_ld, value_at, slot, flip, segment;      // segment: chunks of one
};

// One workgroup per (chunk, head).  delta: convolution, silu and unit norm of the head's q and k, convolution and silu of its v.
// A lane holds one token's four channels of every tile of its wave.  Pairs s < t differ first in some bit h of their numbers: with the decays of t from the last
// multiple of h on and those behind s up to it, each of them at most one, all pairs of that bit are one matrix product over the channels; the products of decays
// over blocks of h tokens become those of 2h by one exchange between lanes of a row.  So four levels of products replace sixteen running keys a pair of threads
// (us, 2048 tokens: 8 heads of 128 of gated linear attention 29 -> 13, 16 of 128 | 128 of the delta rule 71 -> 54).  What is left is memory: it writes 27 KB a chunk and head of 128 channels.
// Three workgroups a CU for the delta rule's largest heads: left alone the compiler takes 180 registers there, which hold two (us, 1531 tokens of 8 heads of 256 | 256: 54 -> 42).
template <int KIND, int TILES>      // of a wave
__global__ __launch_bounds__(kPfThreads, KIND == CHUNK_DELTA && TILES == 4 ? 3 : 1) void chunk_prepare(const ChunkArgs g) {
  constexpr int C = kChunkTokens, kSums = KIND == CHUNK_DELTA ? 2 : 1;
  __shared__ f32x4 sums[kSums][kChunkWaves][64];
  __shared__ double diagonal[kChunkWaves][C];
  __shared__ float norms[2][kChunkWaves][C], step[C];
  __shared__ __align__(16) float turned[kChunkWaves][C][C + 4];
  __shared__ __align__(16) float sa[C][C];
  __shared__ f32x4 st[KIND == CHUNK_DELTA ? 64 : 1];      // T as a fragment
  const QmkHybridLayer& l = g.layer;
  const int head = blockIdx.y, chunk = blockIdx.x, m0 = chunk * C, count = min(C, g.M - m0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), t = lane & 15, quad = lane >> 4;
  const size_t row = min(m0 + t, g.M - 1);
  const bool real = t < count;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};

  // One 16 x 16 matrix turned, through this wave's part of LDS: four columns of a row -> four rows of a column.
  auto turn = [&](f32x4 v) {
    store4(&turned[wave][t][quad * 4], v);
    __builtin_amdgcn_wave_barrier();
    const f32x4 out = {turned[wave][quad * 4][t], turned[wave][quad * 4 + 1][t], turned[wave][quad * 4 + 2][t], turned[wave][quad * 4 + 3][t]};
    __builtin_amdgcn_wave_barrier();
    return out;
  };
  // delta: four channels from `ch` on at this lane's token, behind convolution and silu.
  auto convolved = [&](int ch) {
    const int W = conv_channels(l), taps = l.taps;
    const float* old = l.shift + (static_cast<size_t>(g.slot) * 2 + g.flip) * (taps - 1) * W;
    constexpr int kFew = 4;
    auto input = [&](int back) {      // tokens behind the portion are not used
      const int at = min(m0 + t - back, g.M - 1);
      return read4((at >= 0 ? g.q + static_cast<size_t>(at) * W : old + static_cast<size_t>(at + taps - 1) * W) + ch);
    };
    f32x4 v = zero;
    if (taps <= kFew) {
      f32x4 in[kFew], weight[kFew];
#pragma unroll
      for (int j = 0; j < kFew; ++j) {
        const bool there = j >= kFew - taps;
        in[j] = input(there ? kFew - 1 - j : 0);
        weight[j] = there ? read4(l.vec2 + static_cast<size_t>(j - kFew + taps) * W + ch) : zero;
      }
#pragma unroll
      for (int j = 0; j < kFew; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = j >= kFew - taps ? fmaf(weight[j][i], in[j][i], v[i]) : v[i];
    } else {
      for (int j = 0; j < taps; ++j) {
        const f32x4 in = input(taps - 1 - j), weight = read4(l.vec2 + static_cast<size_t>(j) * W + ch);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaf(weight[i], in[i], v[i]);
      }
    }
    return each(v, [](float x) { return x * sigmoid(x); });
  };
  // Its values' tile `tile`, the head's last one again behind it.
  auto value_tile = [&](int tile) {
    const f32x4 v = convolved(2 * l.kv_heads * g.dim + head * g.n + min(tile * 16, g.n - 16) + quad * 4);
    return real ? v : zero;
  };
  constexpr int kValues = 2;      // tiles of values that a wave holds until T is there
  f32x4 q[TILES], k[TILES], w[TILES], held[KIND == CHUNK_DELTA ? kValues : 1];
  double dot = 0.;      // of this token's q and k: at a first token, or behind strong decays, it is all of an output, whose norm may leave little but its sign
  if constexpr (KIND == CHUNK_DELTA) {
    const int kv = head / (l.heads / l.kv_heads), keys = l.kv_heads * g.dim;
    float nq = 0.f, nk = 0.f;
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int c = (wave * TILES + j) * 16 + quad * 4;
      q[j] = k[j] = zero;
      if ((wave * TILES + j) * 16 < g.dim) {
        q[j] = convolved(kv * g.dim + c);
        k[j] = convolved(keys + kv * g.dim + c);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        nq = fmaf(q[j][i], q[j][i], nq);
        nk = fmaf(k[j][i], k[j][i], nk);
        dot = fma(static_cast<double>(q[j][i]), static_cast<double>(k[j][i]), dot);
      }
    }
#pragma unroll
    for (int j = 0; j < kValues; ++j) held[j] = value_tile(wave + j * kChunkWaves);
    if (tid < count) step[tid] = g.beta[static_cast<size_t>(m0 + tid) * g.beta_ld + head];
    nq += __shfl_xor(nq, 16);
    nk += __shfl_xor(nk, 16);
    nq += __shfl_xor(nq, 32);
    nk += __shfl_xor(nk, 32);
    if (quad == 0) {
      norms[0][wave][t] = nq;
      norms[1][wave][t] = nk;
    }
    __syncthreads();
    nq = nk = 0.f;
#pragma unroll
    for (int i = 0; i < kChunkWaves; ++i) {
      nq += norms[0][i][t];
      nk += norms[1][i][t];
    }
    const float iq = l.q_scale / sqrtf(nq + 1e-6f), ik = 1.f / sqrtf(nk + 1e-6f);      // unit vectors
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      q[j] *= iq;
      k[j] *= ik;
    }
    dot = real ? dot * iq * ik : 0.;
  } else {
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int c = head * g.dim + min((wave * TILES + j) * 16, g.dim - 16) + quad * 4;
      q[j] = read4(g.q + row * g.ld + c);
      k[j] = read4(g.k + row * g.ld + c);
      if constexpr (KIND == CHUNK_GLA) q[j] *= l.q_scale;
    }
  }
#pragma unroll
  for (int j = 0; j < TILES; ++j) {
    const bool there = (wave * TILES + j) * 16 < g.dim;
    const int c = head * g.dim + min((wave * TILES + j) * 16, g.dim - 16) + quad * 4;
    w[j] = read4(g.decay + row * g.heads * g.dim + c);
    q[j] = there && real ? q[j] : zero;
    k[j] = there && real ? k[j] : zero;
    w[j] = there && real ? w[j] : one;
    const f32x4 bonus = KIND == CHUNK_WKV ? read4(l.vec1 + c) : one;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if constexpr (KIND != CHUNK_DELTA) dot = fma(static_cast<double>(q[j][i]) * bonus[i], static_cast<double>(k[j][i]), dot);
  }
  dot += __shfl_xor(dot, 16);
  dot += __shfl_xor(dot, 32);
  if (quad == 0) diagonal[wave][t] = dot;

  // Products of decays within this token's block of h: ahead of it, behind it, all; from now on q (delta: and k') with its own decay but for wkv.
  f32x4 ahead[TILES], behind[TILES], all[TILES], key[KIND == CHUNK_DELTA ? TILES : 1];
#pragma unroll
  for (int j = 0; j < TILES; ++j) {
    ahead[j] = behind[j] = one;
    all[j] = w[j];
    if constexpr (KIND != CHUNK_WKV) q[j] *= w[j];
    if constexpr (KIND == CHUNK_DELTA) key[j] = k[j] * w[j];
  }
  f32x4 pairs[kSums] = {};
  auto level = [&](auto size, auto exchange) {
    constexpr int h = decltype(size)::value;
    const bool later = (t & h) != 0;
    f32x4 p[kSums] = {};
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const f32x4 to = later ? q[j] * ahead[j] : zero, from = later ? zero : k[j] * behind[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) p[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(to[i], from[i], p[0], 0, 0, 0);
      if constexpr (KIND == CHUNK_DELTA) {
        const f32x4 also = later ? key[j] * ahead[j] : zero;
#pragma unroll
        for (int i = 0; i < 4; ++i) p[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(also[i], from[i], p[1], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float other = dpp_f32<decltype(exchange)::value>(1.f, all[j][i]);
        ahead[j][i] *= later ? other : 1.f;
        behind[j][i] *= later ? 1.f : other;
        all[j][i] *= other;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {      // row (later token) r, column (earlier one) t: of one block of 2h.  All others are zeros, also where an operand is not finite
      const int r = quad * 4 + i;
      const bool pair = (r ^ t) < 2 * h && (r & ~t & h) != 0;
#pragma unroll
      for (int e = 0; e < kSums; ++e) pairs[e][i] += pair ? p[e][i] : 0.f;
    }
  };
  level(std::integral_constant<int, 1>{}, std::integral_constant<int, kDppQuadXor1>{});
  level(std::integral_constant<int, 2>{}, std::integral_constant<int, kDppQuadXor2>{});
  level(std::integral_constant<int, 4>{}, std::integral_constant<int, kDppHalfMirror>{});
  level(std::integral_constant<int, 8>{}, std::integral_constant<int, 0x140>{});      // row_mirror
#pragma unroll
  for (int e = 0; e < kSums; ++e) sums[e][wave][lane] = pairs[e];

  float* rec = g.chunks + (static_cast<size_t>(chunk) * g.heads + head) * chunk_floats(g.dim);
  constexpr int stored = TILES * kChunkWaves;
  float *rq = rec, *rk = rq + stored * 256, *rd = rk + stored * 256, *rg = rd + stored * 256, *rb = rg + stored * 16;
#pragma unroll
  for (int j = 0; j < TILES; ++j) {
    const int tile = wave * TILES + j;
    store4(rq + tile * 256 + lane * 4, q[j] * ahead[j]);
    if (t == 0) store4(rg + tile * 16 + quad * 4, all[j]);
    store4(rd + tile * 256 + lane * 4, turn(k[j] * behind[j]));
    if constexpr (KIND == CHUNK_DELTA) key[j] = turn(key[j] * ahead[j]);
  }
  if constexpr (KIND == CHUNK_DELTA) {
#pragma unroll
    for (int j = 0; j < kValues; ++j) held[j] = turn(held[j]);
  }
  __syncthreads();
  {
    const int to = (tid >> 2) & 15, from = (tid >> 6) * 4 + (tid & 3), at = (to >> 2) * 16 + from;
    float b = 0.f, a = 0.f;
    double d = 0.;
#pragma unroll
    for (int i = 0; i < kChunkWaves; ++i) {
      b += sums[0][i][at][to & 3];
      d += diagonal[i][to];
      if constexpr (KIND == CHUNK_DELTA) a += sums[1][i][at][to & 3];
    }
    rb[tid] = to == from ? static_cast<float>(d) : b;      // (no pair is on the diagonal)
    if constexpr (KIND == CHUNK_DELTA) sa[to][from] = a;
  }
  if constexpr (KIND == CHUNK_DELTA) {
    __syncthreads();
    if (tid < C) {     // column tid of T
      float col[C];
#pragma unroll
      for (int r = 0; r < C; ++r) {
        float acc = r == tid ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < r; ++j) acc = fmaf(-sa[r][j], col[j], acc);
        col[r] = r < count ? acc * step[r] : 0.f;
        st[(tid >> 2) * 16 + r][tid & 3] = col[r];
      }
    }
    __syncthreads();
    // W and T v: what the scan's chain need not wait for.
    const f32x4 T = st[lane];
    auto product = [](f32x4 a, f32x4 b) {
      f32x4 c = {};
#pragma unroll
      for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
      return c;
    };
#pragma unroll
    for (int j = 0; j < TILES; ++j) store4(rk + (wave * TILES + j) * 256 + lane * 4, product(key[j], T));
    float* values = g.values + (static_cast<size_t>(chunk) * g.heads + head) * (g.n * C) + lane * 4;
#pragma unroll
    for (int j = 0; j < kValues; ++j) {
      const f32x4 v = product(T, held[j]);
      const int tile = wave + j * kChunkWaves;
      if (tile * 16 < g.n) store4(values + tile * 256, v);
    }
#pragma unroll 1
    for (int tile = wave + kValues * kChunkWaves; tile * 16 < g.n; tile += kChunkWaves) store4(values + tile * 256, product(T, turn(value_tile(tile))));
  }
}

// Sixteen value columns a wave, all key channels; one segment and head a workgroup.  A chunk's record goes from memory to LDS by itself while the one before is
// multiplied: the state's tiles are the matrix instruction's accumulators and at the same time the second operand of the products that read them, and nothing is
// exchanged between waves.  OUT: from the segment's start, with outputs, and the last segment leaves the portion's state; otherwise from nothing, for what it
// leaves.  What a chunk adds to a state is summed by itself, so that the state is rounded once a chunk and not with every product (error against 64 bits, the state
// as the products' own accumulator -> so: 640 tokens without decay 2.9e-7 -> 1.1e-7; a first wkv state of the 2b shape behind 200 tokens in fp32, beside token after token, x 1.012 -> x 0.991).
// What bounds it is the fp32 matrix instruction (of eight tiles 68 of 32 cycles a chunk and wave, 32 without outputs) and, where a launch begins, all its workgroups' first loads (12 us of
// 29).  us in whole portions, chunks one after the other with keys split over waves -> three launches side by side: 2048 tokens of 8 heads of 128 | 256 68 -> 29 + 17 + 8, 1531 of 32
// heads of 64 (wkv, before: token by token, with chunk_prepare's 16) 117 -> 17 + 10 + 5 + 16.  Segments of 16 chunks: 33 + 19 + 6 and 20 + 12 + 5.
// (Sums by chunk and the look for values that are not finite are part of it: without them 30.5 + 17.9 where it takes 31.8 + 18.5 with.)
template <int TILES, bool OUT>
__global__ __launch_bounds__(kPfThreads, TILES == 16 ? 1 : 2) void segment_scan(const ChunkArgs g) {
  constexpr int kFirst = OUT ? TILES : 0, kRest = (TILES * 256 + TILES * 16 + (OUT ? 256 : 0) + 255) / 256;      // loads of 1 KB of a record: G q; D k, G and B
  constexpr int kRecord = (kFirst + kRest + 3) / 4, kEach = kRecord + 1;      // loads of a wave: of the record (the last ones twice), its part of the values
  constexpr int kStage = kEach * 4 * 64, kValues = kRecord * 4 * 64, kStages = TILES == 16 ? 2 : 3;
  __shared__ __align__(16) v4u lds[kStages * kStage];
  using Lds = __attribute__((address_space(3))) v4u;
  Lds* const stages = (Lds*)lds;
  const QmkHybridLayer& l = g.layer;
  // (Workgroups of one segment and head, which read the same records, on one XCD.)
  const int dim = g.dim, n = g.n, groups = (n + 63) / 64, id = xcd_order(blockIdx.x, gridDim.x), group = id % groups, head = id / groups % g.heads, segment = id / groups / g.heads;
  const int out_ld = g.heads * n;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, quad = lane >> 4;
  const int column = group * 64, v0 = column + wave * 16, tiles = dim / 16;
  const bool mine = v0 < n;
  const int first = segment * g.segment, chunks = min(chunks_of(g.M) - first, g.segment), segments = segments_of(g.M, g.segment);
  const size_t size = static_cast<size_t>(dim) * n, place = v0 + col;
  float* state = l.state + (static_cast<size_t>(g.slot) * g.heads + head) * size + place;
  f32x4 s[TILES], fade[OUT ? 1 : TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j) {
    s[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (!OUT) fade[j] = f32x4{1.f, 1.f, 1.f, 1.f};
  }
  if constexpr (OUT) {
    const bool own = segments <= kOwnStarts;
    const int from = own ? 0 : segment;
    const float* start = segments == 1 ? state : g.starts + (static_cast<size_t>(from) * g.heads + head) * size + place;
    if (mine) {
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (j < tiles) s[j][i] = start[static_cast<size_t>(j * 16 + quad * 4 + i) * n];
#pragma unroll 1
      for (int before = from; before < segment; ++before) {
        start += g.heads * size;
        const float* fades = g.fades + (static_cast<size_t>(before + 1) * g.heads + head) * dim + quad * 4;
        f32x4 left[TILES];
#pragma unroll
        for (int j = 0; j < TILES; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j < tiles) left[j][i] = start[static_cast<size_t>(j * 16 + quad * 4 + i) * n];
#pragma unroll
        for (int j = 0; j < TILES; ++j)
          if (j < tiles) s[j] = s[j] * read4(fades + j * 16) + left[j];
      }
    }
  }
  // Tokens and columns behind the last ones are that one and the head's last four again: they meet zeros of the record, or nobody reads them.
  auto issue = [&](int c) {
    const int chunk = first + c;
    Lds* to = stages + c % kStages * kStage;
    auto load = [&](const float* from, int place) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)from, (__attribute__((address_space(3))) uint32_t*)(to + place * 64), 16, 0, 0);
    };
    const float* rec = g.chunks + (static_cast<size_t>(chunk) * g.heads + head) * chunk_floats(dim) + lane * 4;
#pragma unroll
    for (int i = 0; i < kRecord; ++i) {
      const int part = min(i * 4 + wave, kFirst + kRest - 1);
      load(rec + (part < kFirst ? part * 256 : TILES * 512 + (part - kFirst) * 256), part);
    }
    const int token = min(chunk * kChunkTokens + wave * 4 + quad, g.M - 1), at = min(column + col * 4, n - 4);
    load(g.values + static_cast<size_t>(token) * g.value_ld + g.value_at + head * n + at, kRecord * 4 + wave);
  };
  auto buffer = [](const float* base, int bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00027000); };
  // Bytes from a chunk's first value (output) to behind its last one, of rows of `ld`: tokens behind the last one are read as zero and not written.
  auto extent = [&](int chunk, int ld) { return ((min(g.M - chunk * kChunkTokens, kChunkTokens) - 1) * ld + 16) * 4; };
  // Until all but the last `later` of this wave's requests are done, and everybody's.
  auto landed = [&](auto later) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(later)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto product = [](f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
    return c;
  };
  constexpr int kAhead = kStages - 1;
#pragma unroll
  for (int c = 0; c < kAhead; ++c)
    if (c < chunks) issue(c);
#pragma unroll 1
  for (int c = 0; c < chunks; ++c) {
    // This chunk's stage has landed, and everybody has read the one that is filled next.  Behind its requests come those of the stages since and, from the second
    // chunk on, at least one chunk's four stores of outputs, which count like loads.
    constexpr int kLater = (kAhead - 1) * kEach;
    if (kLater == 0 || c + kAhead > chunks) landed(std::integral_constant<int, 0>{});
    else if (OUT && mine && c > 0) landed(std::integral_constant<int, kLater + 4>{});
    else landed(std::integral_constant<int, kLater>{});
    if (c + kAhead < chunks) issue(c + kAhead);
    const int chunk = first + c;
    const Lds *q = stages + c % kStages * kStage, *d = q + kFirst * 64, *decay = d + TILES * 64, *b = decay + TILES * 4;
    const auto* value = (const __attribute__((address_space(3))) float*)(stages + c % kStages * kStage + kValues) + wave * 16 + col;
    const f32x4 u = {value[quad * 256], value[quad * 256 + 64], value[quad * 256 + 128], value[quad * 256 + 192]};
    auto fragment = [&](const Lds* at) { return __builtin_bit_cast(f32x4, at[lane]); };
    f32x4 fq[OUT ? TILES : 1], fd[TILES], faded[TILES], fb, o[4] = {}, finite = u;
    bool whole = true;
    if constexpr (OUT) {
#pragma unroll
      for (int j = 0; j < TILES; ++j) fq[j] = fragment(q + j * 64);
      fb = fragment(b);
    }
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      fd[j] = fragment(d + j * 64);
      faded[j] = __builtin_bit_cast(f32x4, decay[j * 4 + quad]);
    }
    __builtin_amdgcn_sched_barrier(0);      // (all fragments are asked for ahead of the products: read between them, they wait for registers)
    if constexpr (OUT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        whole = whole && __builtin_isfinite(u[i]);
        finite[i] = __builtin_isfinite(u[i]) ? u[i] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < TILES; ++j) o[j & 3] = product(fq[j], s[j], o[j & 3]);
      o[0] = ((o[0] + o[1]) + (o[2] + o[3])) + product(fb, finite, f32x4{0.f, 0.f, 0.f, 0.f});
    }
    f32x4 added[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) added[j] = product(fd[j], u, f32x4{0.f, 0.f, 0.f, 0.f});
    if constexpr (!OUT) __builtin_amdgcn_sched_barrier(0);      // (nothing else is left to do while a product is waited for)
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      if constexpr (!OUT) fade[j] *= faded[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[j][i] = fmaf(s[j][i], faded[j][i], added[j][i]);
    }
    if constexpr (OUT) {      // (branches behind all products, which are scheduled together)
      if (!__all(whole)) {      // A value that is not finite reaches its own token and later ones alone: above B's diagonal it would meet zeros.
        const auto* pair = (const __attribute__((address_space(3))) float*)b;
#pragma unroll 1
        for (int from = 0; from < kChunkTokens; ++from) {
          const float v = value[from * 64];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = quad * 4 + i;
            if (from <= t && !__builtin_isfinite(v)) o[0][i] += pair[((from >> 2) * 16 + t) * 4 + (from & 3)] * v;
          }
        }
      }
      if (mine) {
        const auto to = buffer(g.out + static_cast<size_t>(chunk) * kChunkTokens * out_ld + head * n + v0, extent(chunk, out_ld));
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[0][i]), to, ((quad * 4 + i) * out_ld + col) * 4, 0, 0);
      }
    }
  }
  if (!mine) return;
  if (!OUT && segment == 0 && segments <= kOwnStarts) {      // a copy of the portion's state, which the last segment overwrites, for the others to start from
    f32x4 held[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j < tiles) held[j][i] = state[static_cast<size_t>(j * 16 + quad * 4 + i) * n];
    float* copy = g.starts + head * size + place;
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j < tiles) copy[static_cast<size_t>(j * 16 + quad * 4 + i) * n] = held[j][i];
  }
  float* to = OUT ? state : g.starts + (static_cast<size_t>(segment + 1) * g.heads + head) * size + place;
  if (OUT && segment + 1 < segments) return;
#pragma unroll
  for (int j = 0; j < TILES; ++j)
    if (j < tiles) {
#pragma unroll
      for (int i = 0; i < 4; ++i) to[static_cast<size_t>(j * 16 + quad * 4 + i) * n] = s[j][i];
      if constexpr (!OUT)
        if (v0 == 0 && col == 0) store4(g.fades + (static_cast<size_t>(segment + 1) * g.heads + head) * dim + j * 16 + quad * 4, fade[j]);
    }
}

// The state every segment starts from, out of the portion's and what the segments leave: four columns of a key row a thread.
__global__ __launch_bounds__(kPfThreads) void segment_starts(const ChunkArgs g) {
  const int rows = g.heads * g.dim, quads = g.n / 4, id = blockIdx.x * kPfThreads + threadIdx.x, segments = segments_of(g.M, g.segment);
  if (id >= rows * quads) return;
  const int row = id / quads;
  const size_t at = static_cast<size_t>(row) * g.n + id % quads * 4, step = static_cast<size_t>(rows) * g.n;
  f32x4 s = read4(g.layer.state + static_cast<size_t>(g.slot) * step + at);
  store4(g.starts + at, s);      // (the last segment overwrites it where it was)
  constexpr int kBatch = 8;      // segments asked for together: each is read and written in one place
#pragma unroll 1
  for (int first = 1; first < segments; first += kBatch) {
    f32x4 left[kBatch];
    float fade[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int segment = min(first + i, segments - 1);
      left[i] = read4(g.starts + segment * step + at);
      fade[i] = g.fades[static_cast<size_t>(segment) * rows + row];
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (first + i >= segments) break;
      s = s * fade[i] + left[i];
      store4(g.starts + (first + i) * step + at, s);
    }
  }
}

// One head and sixteen value columns a workgroup; a wave holds TILES tiles of sixteen key channels of the state as the
// accumulators of the matrix instruction, which are also the second operand of the products that read it.  Tiles behind the
// last one are zeros and take part: with a branch around each tile's products this compiler has left out the wait between a
// tile's last product and the first use of its result on the path that skips the next tile.  Loads have no branches either,
// so that kAhead chunks are in flight: a chunk behind the last one is the last one again, and is not used; tokens behind the last one are zeros of the record.
// What bounds it is the chain of a chunk: products of the state with W (four instructions of 32 cycles a tile), the waves' sums through LDS, the state's update.
// What only the output needs fills the wait for the sums, is the same for every wave (of B u each takes the columns of one of the four instructions, of the sums the
// tokens of one), and is added up behind the next chunk's barrier; W and T v come from chunk_prepare.  us, 2048 tokens of 16 heads of 128 | 128, beside an
// attention behind nothing and behind 2048 keys, T (v - (Gk)^T S) on the chain and a chunk's outputs by one wave -> so: 140 -> 116, 158 -> 158 (the attention's own time there), for which
// chunk_prepare takes 58 where it took 55.  Error against 64 bits in fp32, beside that: 1b shape, 150 tokens (56 models) states x 0.999 +- 0.001, logits x 1.012 +- 0.007, 331 tokens (30) x 0.998 +- 0.001,
// x 1.006 +- 0.009; one token over and over (12), where v is nearly what the state returns, x 1.10 +- 0.06, x 1.07 +- 0.10.  With B u's part in a sum of its own the launch takes 136 where it takes 120.
template <int WAVES>
constexpr int kScanLds = 4 * WAVES * 64;
// kAhead: chunks in flight, what the registers hold.
template <int TILES, int WAVES, int kAhead = TILES == 4 ? 2 : 3>
__device__ __forceinline__ void scan_chunks(const ChunkArgs& g, int head, int v0, f32x4* lds) {
  static_assert(WAVES == 4, "a wave takes one of four instructions, and four of sixteen tokens");
  auto px = reinterpret_cast<f32x4(*)[WAVES][64]>(lds), po = px + 2;
  const QmkHybridLayer& l = g.layer;
  const int dim = g.dim, n = g.n;
  constexpr int tiles = TILES * WAVES;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, quad = lane >> 4;
  const int tile0 = wave * TILES, mine = min(max(dim / 16 - tile0, 0), TILES);
  const int chunks = (g.M + kChunkTokens - 1) / kChunkTokens, out_ld = l.heads * n;
  float* state = l.state + (static_cast<size_t>(g.slot) * l.heads + head) * dim * n + v0 + col;
  auto buffer = [](const float* base, int bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00027000); };
  // This lane's output of a chunk: token wave * 4 + quad, column col; rows behind the last token are not written.
  const uint32_t out_at = ((wave * 4 + quad) * out_ld + col) * 4;
  const uint32_t fragment_at = tile0 * 1024 + lane * 16, decay_at = tile0 * 64 + quad * 16, pairs_at = lane * 16 + wave * 4, value_at = lane * 16;
  f32x4 s[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) s[j][i] = j < mine ? state[static_cast<size_t>((tile0 + j) * 16 + quad * 4 + i) * n] : 0.f;

  struct Fragments {
    f32x4 q[TILES], w[TILES], d[TILES], g[TILES], v;
    float b;
  };
  // Chunks are fetched in their order; behind the last one it is the last one again.
  const size_t rec_step = static_cast<size_t>(l.heads) * chunk_floats(dim), value_step = static_cast<size_t>(l.heads) * n * kChunkTokens;
  const float *rec = g.chunks + static_cast<size_t>(head) * chunk_floats(dim), *values = g.values + static_cast<size_t>(head) * n * kChunkTokens + v0 * kChunkTokens;
  int fetched = 0;
  auto fetch = [&](Fragments& f) {
    const auto r = buffer(rec, chunk_floats(tiles * 16) * 4), v = buffer(values, 1024);
    auto read = [&](uint32_t at, int first) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, first * 4, 0)); };
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      f.w[j] = read(fragment_at + j * 1024, tiles * 256);
      f.q[j] = read(fragment_at + j * 1024, 0);
      f.d[j] = read(fragment_at + j * 1024, tiles * 512);
      f.g[j] = read(decay_at + j * 64, tiles * 768);
    }
    f.b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, pairs_at, tiles * 784 * 4, 0));
    f.v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(v, value_at, 0, 0));
    const bool more = fetched + 1 < chunks;
    rec += more ? rec_step : 0;
    values += more ? value_step : 0;
    fetched += more;
  };
  auto product = [](f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
    return c;
  };
  // Ahead of a branch's end: this compiler (clang 22 of ROCm 7.2.0) has left out the wait between a product and the move of its result where paths meet.  The rule, for any
  // kernel: an accumulator that lives across the end of a branch with a product in it is settled there if its built code has such a move (tests/test_matrix_waits.py walks every
  // path of every kernel for it).  As built now none has, here neither: it stays for the next change of these loops.
  auto settle = [](f32x4& v) { asm volatile("s_nop 15" : "+v"(v)); };
  auto outputs = [&](int chunk) {      // of chunk 0 on: everybody's sums of its outputs are in LDS
    const auto to = buffer(g.out + static_cast<size_t>(chunk) * kChunkTokens * out_ld + head * n + v0, ((min(g.M - chunk * kChunkTokens, kChunkTokens) - 1) * out_ld + 16) * 4);
    const float* from = reinterpret_cast<const float*>(po[chunk & 1][0]) + (wave * 16 + col) * 4 + quad;
    const float o = (from[0] + from[256]) + (from[512] + from[768]);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), to, out_at, 0, 0);
  };
  auto advance = [&](const Fragments& f, int chunk) {
    const int buf = chunk & 1;
    f32x4 x[2] = {}, o[2] = {};      // (two sums of every other tile: half as many roundings follow one another)
#pragma unroll
    for (int j = 0; j < TILES; ++j) x[j & 1] = product(f.w[j], s[j], x[j & 1]);
    px[buf][wave][lane] = TILES == 1 ? x[0] : x[0] + x[1];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < (TILES + 1) / 2; ++j) o[j & 1] = product(f.q[j], s[j], o[j & 1]);
    wait_known<63>();
    __builtin_amdgcn_s_barrier();      // everybody's W S; the outputs of the chunk before
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    f32x4 part[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) part[w] = px[buf][w][lane];
#pragma unroll
    for (int j = (TILES + 1) / 2; j < TILES; ++j) o[j & 1] = product(f.q[j], s[j], o[j & 1]);
    const f32x4 u = f.v - ((part[0] + part[1]) + (part[2] + part[3]));
#pragma unroll
    for (int j = 0; j < TILES; ++j) s[j] = product(f.d[j], u, s[j] * f.g[j]);
    const float own = wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3];
    o[TILES > 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b, own, o[TILES > 1], 0, 0, 0);
    po[buf][wave][lane] = TILES == 1 ? o[0] : o[0] + o[1];
    if (chunk > 0) outputs(chunk - 1);
  };
  Fragments f[kAhead];
#pragma unroll
  for (int a = 0; a < kAhead; ++a) fetch(f[a]);
  int chunk = 0;
  for (; chunk + kAhead <= chunks; chunk += kAhead) {
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      advance(f[a], chunk + a);
      fetch(f[a]);
    }
  }
#pragma unroll
  for (int a = 0; a < kAhead - 1; ++a)
    if (chunk + a < chunks) {
      advance(f[a], chunk + a);
#pragma unroll
      for (int j = 0; j < TILES; ++j) settle(s[j]);
    }
  __syncthreads();
  outputs(chunks - 1);
#pragma unroll
  for (int j = 0; j < TILES; ++j)
    if (j < mine)
#pragma unroll
      for (int i = 0; i < 4; ++i) state[static_cast<size_t>((tile0 + j) * 16 + quad * 4 + i) * n] = s[j][i];
}
template <int TILES, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 1) void chunk_scan(const ChunkArgs g) {
  __shared__ __align__(16) f32x4 lds[kScanLds<WAVES>];
  scan_chunks<TILES, WAVES>(g, blockIdx.x, blockIdx.y * 16, lds);
}

// The two branches of a run need nothing of each other, and the delta rule's chunks are a chain of instructions on a part of the chip: its workgroups come first, and go first on their SIMDs, an
// attention's fill what is left (us, 2048 tokens of 16 heads of 128 | 128 in either, behind nothing and behind 2048 keys, two launches -> one: 122 + 51 -> 116, 122 + 99 -> 158;
// 530 tokens 34 + 18 -> 31, 200 tokens 15 + 8 -> 14).
template <int TILES, int QT, int VT, int KEYS, int STAGES, bool SHARED>
__global__ __launch_bounds__(kPfThreads, 2) void scan_and_attend(const ChunkArgs c, const AttentionArgs a) {
  constexpr int kUnits = kAttentionLds<QT, VT, KEYS, STAGES, SHARED>;
  static_assert(kUnits >= kScanLds<kChunkWaves>, "one array for either");
  __shared__ __align__(16) v4u lds[kUnits];
  const int scans = c.heads * (c.n / 16), id = blockIdx.x;
  if (id < scans) {
    __builtin_amdgcn_s_setprio(3);
    scan_chunks<TILES, kChunkWaves>(c, id % c.heads, id / c.heads * 16, reinterpret_cast<f32x4*>(lds));
  } else {
    attend_rows<QT, VT, KEYS, STAGES, SHARED>(a, id - scans, gridDim.x - scans, lds);
  }
}

}  // namespace hybrid
}  // namespace qmk
