// Prefill kernels of the hybrid route's plain residual: the residual and its norms, keys and values of the full attention,
// and the gated state recurrences (gated linear attention, gated delta rule) in chunks of sixteen tokens on the matrix cores.
//
// Recurrence of one head, state S [keys][values], decay g_t per key channel:
//   S <- g_t S,  u_t = beta_t (v_t - S^T k_t),  S <- S + k_t u_t^T,  o_t = S^T q_t        (gla: u_t = v_t)
// Over a chunk that starts from S, with G_t = g_1 .. g_t and D_ts = g_{s+1} .. g_t (products, never quotients: a decay may
// be small enough for its inverse to overflow):
//   X_t = (G_t k_t)^T S           u = T (v - X),  T = (I + diag(beta) A)^-1 diag(beta),  A_ts = sum_i k_t D_ts k_s  (s < t)
//   o_t = (G_t q_t)^T S + sum_{s <= t} B_ts u_s,  B_ts = sum_i q_t D_ts k_s
//   S  <- G_16 S + sum_s (D_16,s k_s) u_s^T
// chunk_prepare works out everything that no state enters, for all chunks at once; chunk_scan walks the chunks.
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

constexpr int kChunkTokens = 16;
constexpr int kChunkWaves = 4;      // of chunk_prepare

// Tiles of sixteen key channels of a head, the last ones zeros.
__host__ __device__ constexpr int chunk_tiles(int head_dim) { return head_dim <= 64 ? 4 : head_dim <= 128 ? 8 : 16; }
// Floats of one (chunk, head): per tile the fragments of G q, G k and D k and the decays G over the whole chunk, then B and
// T.  A fragment is in the order the matrix instruction takes it: [lane][4].
__host__ __device__ constexpr int chunk_floats(int head_dim) { return chunk_tiles(head_dim) * (3 * 256 + 16) + 2 * 256; }

struct ChunkArgs {
  QmkHybridLayer layer;
  const float* qkv;      // [M][q, k, v]; delta: ahead of the convolution
  const float* decay;    // [M][heads * head_dim]
  const float* beta;     // delta: [M][beta_ld]
  float* chunks;         // [chunk][head][chunk_floats]
  float* values;         // [M][value_ld] at value_at; delta: written here
  float* out;            // [M][heads * v_dim]
  int M, beta_ld, value_ld, value_at, slot, flip;
};

// One workgroup per (chunk, head).  delta: convolution, silu and unit norm of the head's q and k, convolution and silu of its v.
template <bool DELTA>
__global__ __launch_bounds__(kPfThreads) void chunk_prepare(const ChunkArgs g) {
  constexpr int C = kChunkTokens;
  __shared__ float sq[C][kMaxHeadDim], sk[C][kMaxHeadDim], sg[C][kMaxHeadDim];
  __shared__ __align__(16) float sa[C][C], sb[C][C];
  __shared__ float step[C];
  const QmkHybridLayer& l = g.layer;
  const int dim = l.head_dim, n = l.v_dim, head = blockIdx.y, chunk = blockIdx.x, m0 = chunk * C, count = min(C, g.M - m0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kv = head / (l.heads / l.kv_heads), keys = l.kv_heads * dim;

  // A thread takes a channel of q, k or v down the chunk's tokens.
  for (int id = tid; id < (DELTA ? 2 * dim + n : 2 * dim); id += kPfThreads) {
    const int part = id / dim < 2 ? id / dim : 2, c = id - part * dim;
    float v[C];
    if constexpr (DELTA) {
      const int W = conv_channels(l), taps = l.taps, ch = part == 0 ? kv * dim + c : part == 1 ? keys + kv * dim + c : 2 * keys + head * n + c;
      const float* x = g.qkv + ch;
      const float* old = l.shift + (static_cast<size_t>(g.slot) * 2 + g.flip) * (taps - 1) * W + ch;
      const float* weight = l.vec2 + ch;
      auto inside = [&](int at) { return x[static_cast<size_t>(min(at, g.M - 1)) * W]; };      // tokens behind the portion are not used
      auto input = [&](int at) { return at >= 0 ? inside(at) : old[static_cast<size_t>(at + taps - 1) * W]; };
      constexpr int kFew = 4;
      if (taps <= kFew) {
        float in[C + kFew - 1], w[kFew];
#pragma unroll
        for (int j = 0; j < kFew; ++j) w[j] = j >= kFew - taps ? weight[static_cast<size_t>(j - kFew + taps) * W] : 0.f;
#pragma unroll
        for (int j = 0; j < kFew - 1; ++j) in[j] = j >= kFew - taps ? input(m0 - (kFew - 1) + j) : 0.f;
#pragma unroll
        for (int j = 0; j < C; ++j) in[kFew - 1 + j] = inside(m0 + j);
#pragma unroll
        for (int t = 0; t < C; ++t) {
          v[t] = 0.f;
#pragma unroll
          for (int j = 0; j < kFew; ++j) v[t] = fmaf(w[j], in[t + j], v[t]);
        }
      } else {
#pragma unroll
        for (int t = 0; t < C; ++t) {
          v[t] = 0.f;
          for (int j = 0; j < taps; ++j) v[t] = fmaf(weight[static_cast<size_t>(j) * W], input(m0 + t - (taps - 1) + j), v[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < C; ++t) v[t] *= sigmoid(v[t]);
      if (part == 2) {
        float* to = g.values + static_cast<size_t>(m0) * g.value_ld + g.value_at + head * n + c;
#pragma unroll
        for (int t = 0; t < C; ++t)
          if (t < count) to[static_cast<size_t>(t) * g.value_ld] = v[t];
        continue;
      }
    } else {
      const int ld = 2 * keys + l.heads * n;
      const float* row = g.qkv + static_cast<size_t>(m0) * ld + part * keys + kv * dim + c;
#pragma unroll
      for (int t = 0; t < C; ++t) v[t] = row[static_cast<size_t>(min(t, count - 1)) * ld] * (part == 0 ? l.q_scale : 1.f);
    }
    auto& to = part == 0 ? sq : sk;
#pragma unroll
    for (int t = 0; t < C; ++t) to[t][c] = t < count ? v[t] : 0.f;
  }
  if constexpr (DELTA) {
    if (tid < count) step[tid] = g.beta[static_cast<size_t>(m0 + tid) * g.beta_ld + head];
  }
  for (int c = tid; c < dim; c += kPfThreads) {
    const float* row = g.decay + static_cast<size_t>(m0) * l.heads * dim + head * dim + c;
    float v[C];
#pragma unroll
    for (int t = 0; t < C; ++t) v[t] = row[static_cast<size_t>(min(t, count - 1)) * l.heads * dim];
#pragma unroll
    for (int t = 0; t < C; ++t) sg[t][c] = t < count ? v[t] : 1.f;
  }
  __syncthreads();
  if constexpr (DELTA) {      // unit vectors
    for (int t = wave; t < C; t += kChunkWaves) {
      float nq = 0.f, nk = 0.f;
      for (int c = lane; c < dim; c += 64) {
        nq = fmaf(sq[t][c], sq[t][c], nq);
        nk = fmaf(sk[t][c], sk[t][c], nk);
      }
      const float iq = l.q_scale / sqrtf(wave_sum(nq) + 1e-6f), ik = 1.f / sqrtf(wave_sum(nk) + 1e-6f);
      for (int c = lane; c < dim; c += 64) {
        sq[t][c] *= iq;
        sk[t][c] *= ik;
      }
    }
    __syncthreads();
  }

  float* rec = g.chunks + (static_cast<size_t>(chunk) * l.heads + head) * chunk_floats(dim);
  const int tiles = dim / 16, stored = chunk_tiles(dim);
  float *rq = rec, *rk = rq + stored * 256, *rd = rk + stored * 256, *rg = rd + stored * 256, *rb = rg + stored * 16, *rt = rb + 256;
  for (int i = tiles * 256 + tid; i < stored * 256; i += kPfThreads) rq[i] = rk[i] = rd[i] = 0.f;
  if (tid >= dim && tid < stored * 16) rg[tid] = 0.f;
  if (tid < dim) {
    const int tile = tid >> 4, c = tid & 15;
    float cum = 1.f;
#pragma unroll
    for (int t = 0; t < C; ++t) {
      cum *= sg[t][tid];
      const int at = tile * 256 + ((c >> 2) * 16 + t) * 4 + (c & 3);
      rq[at] = sq[t][tid] * cum;
      if constexpr (DELTA) rk[at] = sk[t][tid] * cum;
    }
    rg[tid] = cum;
    float rest = 1.f;
#pragma unroll
    for (int t = C - 1; t >= 0; --t) {
      rd[tile * 256 + ((t >> 2) * 16 + c) * 4 + (t & 3)] = sk[t][tid] * rest;
      rest *= sg[t][tid];
    }
  }
  // Pairs: sixteen lanes share an s, channels 16 apart each; the decayed key runs down the tokens.
  {
    const int s = tid >> 4, part = tid & 15;
    float run[kMaxHeadDim / 16];
#pragma unroll
    for (int j = 0; j < kMaxHeadDim / 16; ++j) run[j] = 0.f;
    for (int t = 0; t < C; ++t) {
      float da = 0.f, db = 0.f;
#pragma unroll
      for (int j = 0; j < kMaxHeadDim / 16; ++j) {
        if (j < tiles) {
          const int c = j * 16 + part;
          const float kt = sk[t][c];
          run[j] *= sg[t][c];
          da = fmaf(kt, run[j], da);
          if (t == s) run[j] = kt;
          db = fmaf(sq[t][c], run[j], db);
        }
      }
      auto sum16 = [](float v) {
        v += dpp_f32<kDppQuadXor1>(0.f, v);
        v += dpp_f32<kDppQuadXor2>(0.f, v);
        v += dpp_f32<0x124>(0.f, v);        // row_ror:4
        v += dpp_f32<0x128>(0.f, v);        // row_ror:8
        return v;
      };
      db = sum16(db);
      if constexpr (DELTA) da = sum16(da);
      if (part == 0) {
        sb[t][s] = db;                       // zero above the diagonal
        sa[t][s] = da;                       // ... and on it
      }
    }
  }
  __syncthreads();
  if (tid < 256) rb[tid] = sb[(tid >> 2) & 15][(tid >> 6) * 4 + (tid & 3)];
  if constexpr (DELTA) {
    if (tid < C) {     // column tid of T
      float col[C];
#pragma unroll
      for (int t = 0; t < C; ++t) {
        float acc = t == tid ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < t; ++j) acc = fmaf(-sa[t][j], col[j], acc);
        col[t] = t < count ? acc * step[t] : 0.f;
        rt[((tid >> 2) * 16 + t) * 4 + (tid & 3)] = col[t];
      }
    }
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

// One head and sixteen value columns a workgroup; a wave holds TILES tiles of sixteen key channels of the state as the
// accumulators of the matrix instruction, which are also the second operand of the products that read it.  Tiles behind the
// last one are zeros and take part: with a branch around each tile's products this compiler has left out the wait between a
// tile's last product and the first use of its result on the path that skips the next tile.  Loads have no branches either,
// so that kAhead chunks are in flight: a chunk, or token, behind the last one is the last one again, and its value is either
// not used or multiplied by zero.
// What bounds it is the chain of a chunk: products of the state with the keys (four dependent instructions of 32 cycles a tile), the
// waves' sums through LDS, T (v - X), the state's update.  So in fp32 eight waves hold the tiles of a gated linear attention's heads of more than
// 64 channels (bf16 portions keep one order, four waves, qmk_hybrid_tiles.h); and what only the output needs is off the chain: G q S is taken while the sums are on their way, and a chunk's outputs
// are added up and stored behind the next chunk's barrier.
// A wave's instructions are on that chain too, one wave a SIMD: chunks are read and written by buffer accesses (places of 32 bits that stay, bases that move on by
// one scalar addition, tokens behind the last one read as zero and not written).  Without the delta rule launch bounds of eight waves, also for four, keep accumulators where
// vector instructions reach them; with it a chunk has too many registers for that.  us, 2048 tokens, addresses of 64 bits worked out for every access -> now: 16 heads of
// 128 | 128 of the delta rule 134 -> 120, 8 of 128 | 256 of gated linear attention 92 -> 70.  Lines of chunks further ahead asked for into L2: 141 and 88.
template <int TILES, int WAVES, bool DELTA>
__global__ __launch_bounds__(DELTA ? WAVES * 64 : 512, DELTA ? 1 : 2) void chunk_scan(const ChunkArgs g) {
  // Chunks in flight: what the registers hold (us, the two shapes above, with 2, 3 and 4 ahead: 131, 120, 123; 87, 70 and, 12 registers of them spilled, 68; 8 heads of 256 | 256 in
  // fp32, 4000 tokens, a portion of one layer with eight waves: 2 628, 3 597, 4 603).
  constexpr int kAhead = TILES == 1 ? 4 : TILES == 2 ? 3 : 2;
  __shared__ f32x4 px[2][WAVES][64], po[2][WAVES][64];
  const QmkHybridLayer& l = g.layer;
  const int dim = l.head_dim, n = l.v_dim, head = blockIdx.x, v0 = blockIdx.y * 16;
  constexpr int tiles = TILES * WAVES;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, quad = lane >> 4;
  const int tile0 = wave * TILES, mine = min(max(dim / 16 - tile0, 0), TILES);
  const int chunks = (g.M + kChunkTokens - 1) / kChunkTokens, out_ld = l.heads * n;
  float* state = l.state + (static_cast<size_t>(g.slot) * l.heads + head) * dim * n + v0 + col;
  auto buffer = [](const float* base, int bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00027000); };
  // Bytes from a chunk's first value (output) to behind its last one, of rows of `ld`.
  auto extent = [&](int chunk, int ld) { return ((min(g.M - chunk * kChunkTokens, kChunkTokens) - 1) * ld + 16) * 4; };
  uint32_t value_at[4], out_at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    value_at[i] = ((quad * 4 + i) * g.value_ld + col) * 4;
    out_at[i] = ((quad * 4 + i) * out_ld + col) * 4;
  }
  const uint32_t fragment_at = tile0 * 1024 + lane * 16, decay_at = tile0 * 64 + quad * 16, shared_at = lane * 16;
  f32x4 s[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) s[j][i] = j < mine ? state[static_cast<size_t>((tile0 + j) * 16 + quad * 4 + i) * n] : 0.f;

  struct Fragments {
    f32x4 q[TILES], k[TILES], d[TILES], g[TILES], b, t, v;
  };
  // Chunks are fetched in their order; behind the last one it is the last one again.
  const size_t rec_step = static_cast<size_t>(l.heads) * chunk_floats(dim), value_step = static_cast<size_t>(kChunkTokens) * g.value_ld;
  const float *rec = g.chunks + static_cast<size_t>(head) * chunk_floats(dim), *values = g.values + g.value_at + head * n + v0;
  int fetched = 0;
  auto fetch = [&](Fragments& f) {
    const auto r = buffer(rec, chunk_floats(tiles * 16) * 4), v = buffer(values, extent(fetched, g.value_ld));
    auto read = [&](uint32_t at, int first) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, first * 4, 0)); };
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      if constexpr (DELTA) f.k[j] = read(fragment_at + j * 1024, tiles * 256);
      f.q[j] = read(fragment_at + j * 1024, 0);
      f.d[j] = read(fragment_at + j * 1024, tiles * 512);
      f.g[j] = read(decay_at + j * 64, tiles * 768);
    }
    f.b = read(shared_at, tiles * 784);
    if constexpr (DELTA) f.t = read(shared_at, tiles * 784 + 256);
#pragma unroll
    for (int i = 0; i < 4; ++i) f.v[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v, value_at[i], 0, 0));
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
  // Ahead of a branch's end: this compiler (clang 22 of ROCm 7.2.0) has left out the wait between a product and the move of its result where paths meet; without
  // this <1, 4> moves one two instructions behind its product.  The rule, for any kernel: an accumulator that lives across the end of a branch with a product in it is
  // settled there if its built code has such a move (tests/test_matrix_waits.py walks every path of every kernel for it); none but these two places has.
  auto settle = [](f32x4& v) { asm volatile("s_nop 15" : "+v"(v)); };
  f32x4 inner = {};       // B u of the last chunk whose outputs are this wave's
  auto outputs = [&](int chunk) {
    if (chunk < 0 || wave != (chunk & (WAVES - 1))) return;
    f32x4 o = inner;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += po[chunk & 1][w][lane];
    const auto to = buffer(g.out + static_cast<size_t>(chunk) * kChunkTokens * out_ld + head * n + v0, extent(chunk, out_ld));
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[i]), to, out_at[i], 0, 0);
  };
  auto advance = [&](const Fragments& f, int chunk) {
    const int buf = chunk & 1;
    if constexpr (DELTA) {
      f32x4 x = {};
#pragma unroll
      for (int j = 0; j < TILES; ++j) x = product(f.k[j], s[j], x);
      px[buf][wave][lane] = x;
    }
    __syncthreads();      // everybody's X; the chunk before's G q S
    f32x4 u = f.v;
    if constexpr (DELTA) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) u -= px[buf][w][lane];
    }
    f32x4 o = {};
#pragma unroll
    for (int j = 0; j < TILES; ++j) o = product(f.q[j], s[j], o);
    po[buf][wave][lane] = o;
    if constexpr (DELTA) u = product(f.t, u, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int j = 0; j < TILES; ++j) s[j] = product(f.d[j], u, s[j] * f.g[j]);
    outputs(chunk - 1);
    if (wave == (chunk & (WAVES - 1))) {
      inner = product(f.b, u, f32x4{0.f, 0.f, 0.f, 0.f});
      settle(inner);
    }
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
