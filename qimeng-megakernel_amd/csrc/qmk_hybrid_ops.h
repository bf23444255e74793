// Decode ops of the hybrid route: one workgroup executes one instruction of the tensor built by
// decode_schedule_hybrid/instructions/scheduler.py.
//
// A step is a chain of stages; an instruction waits for the units of the stages before that it reads, and only an attention's
// parts are counted in (the per-XCD counters of qmk_device.h).  Activations between stages are fp32 and travel as tagged units
// with device-coherent loads and stores; weights are streamed once, bf16, and multiplied in fp32.  On a plain residual no stage adds to it: the instructions that read it next
// add what the layer run before has left (each for itself, one of them keeps the sum), so a norm over a branch's whole
// output costs no stage of its own.  What does not depend on this step's earlier stages is asked for before an
// instruction waits: its first weight rows, norm weights, recurrent states, old cache rows, the streams it will update.
//
// What bounds a step beside its bytes is the way from a stage's last store to the next one's first products, 3 to 4 us on the average of lusupel-1b's 89 stages:
// the store's way, a look's way, the norm, rows behind the look.  Work that an instruction does ahead of its first look counts in full for the workgroup that
// the others wait for, so its addresses are worked out while the instruction before waits (plan_of).
#pragma once

#include <type_traits>

#include "qmk_device.h"
#include "qmk_hybrid.h"

namespace qmk {
namespace hybrid {

enum : int {
  OP_NOOP = 0,
  OP_IN_PROJECT = 1,      // norm1 + the mixer's input projections, with what can be done per output behind them
  OP_LRU_STEP = 2,        // gates of one block + the recurrence of its channels
  OP_LATENT_ABSORB = 3,   // W_uk^T q per head
  OP_ATTEND = 4,          // one part of the visible keys for 16 heads; the one that holds the step's position appends the cache row
  OP_LATENT_VALUE = 5,    // merge of the parts, W_uv, output gate
  OP_WKV_STEP = 6,        // decay, recurrence, per-head norm and gate of one head
  OP_OUT_PROJECT = 7,     // output (sub 0) or down (sub 1) projection + all streams of the residual
  OP_UP_GATE = 8,         // norm2 + gate/up rows + gelu
  OP_LM_HEAD = 9,         // final norm + vocabulary rows
  OP_STATE_STEP = 10,     // gla, delta: decays and recurrence of some value columns of one head
  OP_ATTEND_MERGE = 11,   // merge of the parts of one head, output gate
  OP_JOIN = 12,           // rows of [x; embedding] -> x
  OP_GATE = 13,           // delta: rows of the output gate
};

constexpr int kMaxStreams = QMK_HYBRID_MAX_STREAMS;
constexpr int kMaxTaps = QMK_HYBRID_MAX_TAPS;
constexpr int kMaxRows = 512;                 // rows of one instruction
constexpr int kMaxOutRows = kThreads / kMaxStreams;   // ... of OP_OUT_PROJECT: a thread per row and stream
constexpr int kChunk = kWaveSize * 8;         // columns one wave covers with one 16-byte load per lane
constexpr int kMaxK = 24576;                  // longest activation vector
constexpr int kAttendFloats = 33792;          // LDS of the attention op: query, key tile, scores
constexpr int kMaxRank = 512;
constexpr int kMaxHeadDim = 256;              // wkv, gla, delta
constexpr int kStateColumns = 64;             // value columns of one OP_STATE_STEP
constexpr int kStateRows = 32;                // key rows of the state one of its threads holds: 256 rows / (512 / 64) threads a column
constexpr int kStateBatch = 8;                // ... taken together, without branches: rows behind the last one count with weights of zero
constexpr int kStateVector = kMaxHeadDim + kStateBatch * kThreads / 16;   // places of q, k and the decays in LDS, zeros behind head_dim
constexpr int kMaxParts = 64;
constexpr int kDepth = 8;                     // weight rows a wave keeps in flight and reduces together
// ... of which so many are asked for ahead of the wait, the others when the vector has come: looks and stores of a hand-over stand behind the requests for rows
// in the memory system's queues (us a step with 2, 4, 6 and 8 ahead: lusupel-1b 760, 749, 761, 767; givopel-1b with 4, 6 and 8 580, 601, 612).
constexpr int kRowsFirst = 4;
constexpr int kFewTaps = 4;                   // taps of a convolution whose inputs and weights a thread holds
constexpr int kStageGroupRows = 54;           // the counter layout of one group of four stages (qmk_device.h)
constexpr int kStageGroupSlots = 48;

struct DecodeParams {
  const int32_t* instructions;
  const QmkHybridLayer* layers;
  int32_t* barriers;
  int32_t* status;
  uint64_t* timeline;
  uint64_t* candidates;
  const u16* embed;
  const u16* head;
  const float* final_norm;
  const int64_t* token_in;
  int64_t* token_out;
  float* logits;
  // units (below), but for the streams
  uint64_t* u;          // [D] input of the next sublayer before its norm
  uint64_t* sums;       // plain: [2][1 + branches + 1][D] a copy of the residual and what the run that has left it adds: branches, feed-forward
  uint64_t* proj;       // outputs of OP_IN_PROJECT
  uint64_t* mix;        // what the output / down projection reads
  uint64_t* absorbed;   // [heads][rank], in bf16 mode pairs of rounded values
  uint64_t* units;      // all of them
  float* x;             // [streams][D], each element's owner alone
  float* part;       // [parts][heads16][rank] unnormalised sums
  float* ml;         // [parts][heads16][2] maximum (log2) and sum
  int32_t num_insts;
  int32_t num_layers;
  int32_t groups;
  int32_t width, width_true, streams;
  int32_t vocab, vocab_rows;
  int32_t slot, position, flip;
  int32_t max_splits;
  int32_t early_units, all_units;      // those that nobody reads any more when the last norm's input has come stand first
  float eps, logit_scale, logit_softcap;
  uint32_t spin_limit;
};

// What the first requests of an instruction that streams rows need, worked out while the instruction before it ends: its rows, the vector that they are
// multiplied with; plain: what makes the residual (x, two branches).
struct Plan {
  const u16* w;
  int rows, columns;           // rows 0: an operand is out of range
  const uint64_t* from;
  int length;
  uint32_t tag;
  const uint64_t* sum[3];
  uint32_t sum_tag[3];
};

// Values that are the same in all lanes, in scalar registers.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(v)); }
template <class P>
__device__ __forceinline__ P* uniform(P* v) {
  const uint64_t bits = reinterpret_cast<uint64_t>(v);
  return reinterpret_cast<P*>(static_cast<uint64_t>(uniform(static_cast<uint32_t>(bits >> 32))) << 32 | uniform(static_cast<uint32_t>(bits)));
}

struct Smem {
  union {
    struct {
      float xs[kMaxK];
      float part[kWaves * kMaxRows];
    };
    float attend[kAttendFloats];
  };
  float aux[3072];
  float scratch[3 * kWaves];
  int32_t inst[2][kInstWords];      // of even and of odd index: this instruction and the one behind it
  Plan plan[2];                     // of an instruction of even and of odd index
  int32_t ctl[4];          // [0] no wait has failed, [1] last to retire, [2] this workgroup has cleared its share of the units
  uint64_t t_wait;
  uint64_t stamps[4];      // timeline only: requests made, vector in LDS, rows multiplied, results stored
  float best_val;
  int32_t best_idx;
};

// The layer table never changes during a launch: read through the constant address space its fields are scalar loads
// that stay valid across barriers.
using LayerRef = const __attribute__((address_space(4))) QmkHybridLayer;
using ConstFloat = const __attribute__((address_space(4))) float;
__device__ __forceinline__ LayerRef& layer_of(const DecodeParams& p, int layer) { return ((LayerRef*)p.layers)[layer]; }

struct Op {                // decoded instruction
  int index, opcode, layer, sub, start, count, wait_stage, wait_count, arrive_stage, extra;
};

// The counter helpers of qmk_device.h read these fields of the other routes' parameter block.
__device__ __forceinline__ Params counters_of(const DecodeParams& p) {
  Params c{};
  c.barriers = p.barriers;
  c.status = p.status;
  c.num_layer_barriers = kStageGroupRows;
  c.barrier_slots = kStageGroupSlots;
  c.flags = QMK_FLAG_XCD_COUNTERS;
  c.spin_limit = p.spin_limit;
  return c;
}

__device__ __forceinline__ bool bad_operand(const DecodeParams& p, const Op& o, int operand) {
  if (threadIdx.x == 0) report_error(counters_of(p), QMK_DEV_BAD_OPERAND, o.index, o.opcode, operand);
  return false;
}

__device__ __forceinline__ void stamp(const DecodeParams& p, Smem& s, int which) {
  if (p.timeline != nullptr && threadIdx.x == 0) s.stamps[which] = wall_clock64();
}

// ---- hand-over ----
// What a workgroup leaves for others of the same launch is 8-byte units {value, tag}, each stored at once: a reader looks at the units it needs until all carry
// the tag of their entry and half of it, so nobody waits for stores to be acknowledged, counts arrivals or fetches behind a count.  Tags grow along the
// model: a unit's next writer depends on all of its readers through the data (an output row needs every product before it), but for rows of padding,
// whose readers may find the next one there already.  What is read is cleared before the launch ends (OP_LM_HEAD, retirement), failed launches included:
// nothing is kept, and a tag is a pattern (a float of 2.3e18) that nothing else that may use the buffer leaves there.  Only the parts of an attention,
// up to 64 KB for each reader, stay on counters: their readers would look at them all through the attention.
// us a step, counters and leaders on every stage -> so: lusupel-1b, 1000 positions 804 -> 745, givopel-1b, 600 positions 605 -> 580.
constexpr uint32_t kTagBase = 0x5e000000u, kTags = 1u << 20;
__device__ __forceinline__ uint32_t tag_of(int entry, int half) { return kTagBase + 2 * static_cast<uint32_t>(entry) + half; }
__device__ __forceinline__ bool has_come(uint64_t unit, uint32_t tag) { return static_cast<uint32_t>(unit >> 32) - tag < kTags; }
__device__ __forceinline__ void put_bits(uint64_t* at, uint32_t bits, uint32_t tag) {
  __hip_atomic_store(at, static_cast<uint64_t>(tag) << 32 | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put_unit(uint64_t* at, float v, uint32_t tag) { put_bits(at, __float_as_uint(v), tag); }
__device__ __forceinline__ float value_of(uint64_t unit) { return __uint_as_float(static_cast<uint32_t>(unit)); }

__device__ __forceinline__ void wait_failed(const DecodeParams& p, Smem& s, const Op& o) {
  if (static_cast<int>(threadIdx.x) == __builtin_amdgcn_readfirstlane(threadIdx.x)) {
    s.ctl[0] = 0;
    report_error(counters_of(p), QMK_DEV_WAIT_TIMEOUT, o.index, o.opcode, o.wait_stage);
  }
}

// Behind a failed wait of this workgroup the others end early.
__device__ __forceinline__ bool out_of_looks(const DecodeParams& p, Smem& s, const Op& o, uint32_t looks) {
  if (looks > p.spin_limit) {
    wait_failed(p, s, o);
    return true;
  }
  return (looks & 63) == 0 && *const_cast<volatile int32_t*>(s.ctl) == 0;
}

// Units first, first + step, .. of v[0 .. end): `ask` makes the first look, `wait` the others.  A wait that runs out of looks leaves what is there, and
// ctl[0] = 0 behind the next barrier.
template <int N>
struct Units {
  uint64_t r[N];
  __device__ __forceinline__ void ask(const uint64_t* v, int first, int step, int end) {
#pragma unroll
    for (int j = 0; j < N; ++j) r[j] = ld_shared64(v + min(first + j * step, end - 1));
  }
  __device__ __forceinline__ void wait(const DecodeParams& p, Smem& s, const Op& o, const uint64_t* v, int first, int step, int end, uint32_t tag) {
    uint32_t looks = 0;
    while (true) {
      bool all = true;
#pragma unroll
      for (int j = 0; j < N; ++j) all = all && has_come(r[j], tag);
      if (__all(all)) return;
      if (out_of_looks(p, s, o, ++looks)) return;
      ask(v, first, step, end);
    }
  }
  __device__ __forceinline__ float operator[](int j) const { return value_of(r[j]); }
};
// The same of units at places of their own.
template <int N>
struct Gather {
  const uint64_t* at[N];
  uint64_t r[N];
  __device__ __forceinline__ void ask() {
#pragma unroll
    for (int j = 0; j < N; ++j) r[j] = ld_shared64(at[j]);
  }
  __device__ __forceinline__ void wait(const DecodeParams& p, Smem& s, const Op& o, uint32_t tag) {
    uint32_t looks = 0;
    while (true) {
      bool all = true;
#pragma unroll
      for (int j = 0; j < N; ++j) all = all && has_come(r[j], tag);
      if (__all(all)) return;
      if (out_of_looks(p, s, o, ++looks)) return;
      ask();
    }
  }
  __device__ __forceinline__ float operator[](int j) const { return value_of(r[j]); }
};
// One unit of every active lane.
__device__ __forceinline__ float unit_of(const DecodeParams& p, Smem& s, const Op& o, const uint64_t* at, uint32_t tag) {
  Units<1> u;
  u.ask(at, 0, 0, 1);
  u.wait(p, s, o, at, 0, 0, 1, tag);
  return u[0];
}

// The attention's parts: counted arrivals of a whole stage.
__device__ __forceinline__ bool wait_stage(const DecodeParams& p, Smem& s, const Op& o) {
  if (o.wait_stage < 0) return true;
  const Params c = counters_of(p);
  if (threadIdx.x < kWaveSize && !wait_edge_xcd(c, o.wait_stage >> 2, 2 + (o.wait_stage & 3), o.wait_count, p.spin_limit)) wait_failed(p, s, o);
  __syncthreads();
  return s.ctl[0] != 0;
}
__device__ __forceinline__ void arrive_stage(const DecodeParams& p, const Op& o) {
  if (threadIdx.x == 0 && o.arrive_stage >= 0) arrive_all(counters_of(p), o.arrive_stage >> 2, 2 + (o.arrive_stage & 3), 1);
}

// exp(z) as one hardware 2^x, relative error |z| 2^-24: for gates and activations.  Decays, which are multiplied up over
// thousands of tokens, take expf.
__device__ __forceinline__ float exp_fast(float z) { return exp2_fast(z * 1.4426950408889634f); }
__device__ __forceinline__ float sigmoid(float z) { return 1.f / (1.f + exp_fast(-z)); }
// 0.5 z (1 + tanh(t)) = z sigmoid(2 t), t = sqrt(2/pi) (z + 0.044715 z^3)
__device__ __forceinline__ float gelu_tanh(float z) { return z * sigmoid(1.5957691216057308f * (z + 0.044715f * z * z * z)); }
template <class T>
__device__ __forceinline__ float to_f32(T v) {
  if constexpr (sizeof(T) == 2) return bf2f(v);
  else return v;
}
template <class T>
__device__ __forceinline__ T from_f32(float v) {
  if constexpr (sizeof(T) == 2) return f2bf(v);
  else return v;
}

// Place of element k of an activation vector in LDS: a lane's eight columns of a chunk lie in two runs of four, each
// run side by side with the other lanes' (16-byte LDS reads without bank conflicts).
__device__ __forceinline__ int xs_at(int k) {
  return (k & ~(kChunk - 1)) + ((k & 4) << 6) + ((k & (kChunk - 8)) >> 1) + (k & 3);
}

// ---- row streaming ----
// Rows [0, n) of w [., ld] times xs.  A wave owns fixed chunks of 512 columns (several waves share a chunk's rows where
// there are fewer than eight chunks, a wave takes every eighth chunk where there are more), so its eight columns of xs
// per lane sit in registers; it walks down the rows, eight in flight, and reduces eight rows' products at once.
// Narrow matrices (128 and 256 columns) are read as rows of 512: 4 or 2 neighbouring rows side by side.
struct RowStream {
  const u16* at;        // next row to load
  long long pitch;      // elements between rows
  int n, chunk, per, lanes, first, waves, total, ld;
  v4u r[kDepth];

  __device__ __forceinline__ int column(int c) const {
    const int col = c * kChunk + static_cast<int>(threadIdx.x & (kWaveSize - 1)) * 8;
    return col < total ? col : 0;      // a lane behind the last column multiplies whatever it reads by zero
  }
  __device__ __forceinline__ void start(const u16* w, int rows, int columns) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize);
    int narrow = 0;                                          // log2 of the rows side by side
    if (columns == 128 && rows % 4 == 0) narrow = 2;
    if (columns == 256 && rows % 2 == 0) narrow = 1;
    per = 1 << narrow;
    lanes = kWaveSize >> narrow;
    ld = columns;
    total = columns << narrow;
    pitch = total;
    rows >>= narrow;
    const unsigned chunks = static_cast<unsigned>(total + kChunk - 1) / kChunk;
    const int share = chunks > 4 ? 0 : chunks > 2 ? 1 : chunks == 2 ? 2 : 3;     // log2 of the waves per chunk
    chunk = wave >> share;
    const int part = wave & ((1 << share) - 1);
    first = (rows * part) >> share;
    n = ((rows * (part + 1)) >> share) - first;
    waves = chunk < static_cast<int>(chunks) ? (chunks - chunk + kWaves - 1) / kWaves : 0;      // chunks of this wave: chunk, chunk + 8, ...
    if (waves == 0) n = 0;
    at = w + first * pitch;
    const u16* top = at + column(chunk);
#pragma unroll
    for (int j = 0; j < kRowsFirst; ++j)
      if (j < n) r[j] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(top + j * pitch));
  }
  // Behind the wait.
  __device__ __forceinline__ void rest() {
    const u16* top = at + column(chunk);
#pragma unroll
    for (int j = kRowsFirst; j < kDepth; ++j)
      if (j < n) r[j] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(top + j * pitch));
  }
  // part[wave][row] += sums; part must be zero, one barrier behind it.
  __device__ __forceinline__ void run(Smem& s) {
    if (n == 0) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWaveSize), lane = threadIdx.x & (kWaveSize - 1);
    float* out = s.part + wave * kMaxRows;
#pragma unroll 1
    for (int q = 0; q < waves; ++q) {
      const int c = chunk + q * kWaves;
      float x[8];
      {
        // (narrow matrices: every run of `lanes` lanes holds the same vector)
        const int k = per == 1 ? lane : (lane & (lanes - 1));
        float4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
        if (c * kChunk + k * 8 < ld) {
          a = *reinterpret_cast<const float4*>(s.xs + c * kChunk + k * 4);
          b = *reinterpret_cast<const float4*>(s.xs + c * kChunk + kChunk / 2 + k * 4);
        }
        x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
        x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
      }
#pragma unroll 1
      for (int base = 0; base < n; base += kDepth) {
        // the group behind this one: further down, or the top of this wave's next chunk
        const bool more = base + kDepth < n;
        const int next_rows = more ? min(n - base - kDepth, kDepth) : (q + 1 < waves ? min(n, kDepth) : 0);
        const u16* next = more ? at + (base + kDepth) * pitch + column(c) : at + column(c + kWaves);
        float v[kDepth];
#pragma unroll
        for (int j = 0; j < kDepth; ++j) {
          const v4u w = r[j];
          float t = bf_lo(w.x) * x[0];
          t = fmaf(bf_hi(w.x), x[1], t);
          t = fmaf(bf_lo(w.y), x[2], t);
          t = fmaf(bf_hi(w.y), x[3], t);
          t = fmaf(bf_lo(w.z), x[4], t);
          t = fmaf(bf_hi(w.z), x[5], t);
          t = fmaf(bf_lo(w.w), x[6], t);
          t = fmaf(bf_hi(w.w), x[7], t);
          v[j] = t;
          if (j < next_rows) r[j] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(next + j * pitch));
        }
        const float t = reduce8(v, lane, lanes);
        const int row = base + (lane & 7);
        if ((lane & (lanes - 1)) < kDepth && row < n) {
          float* o = out + (first + row) * per + (per == 1 ? 0 : lane / lanes);
          *o = q == 0 ? t : *o + t;
        }
      }
    }
  }
  // Eight values per lane -> lane l holds the sum of value l % 8 over its run of `lanes` lanes (16, 32 or 64): three
  // steps that halve the values while they pair lanes, then plain sums.
  static __device__ __forceinline__ float reduce8(const float (&v)[kDepth], int lane, int lanes) {
    const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4;
    float a[4], b[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float keep = b0 ? v[2 * i + 1] : v[2 * i], give = b0 ? v[2 * i] : v[2 * i + 1];
      a[i] = keep + dpp_f32<kDppQuadXor1>(0.f, give);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float keep = b1 ? a[2 * i + 1] : a[2 * i], give = b1 ? a[2 * i] : a[2 * i + 1];
      b[i] = keep + dpp_f32<kDppQuadXor2>(0.f, give);
    }
    const float keep = b2 ? b[1] : b[0], give = b2 ? b[0] : b[1];
    float t = keep + dpp_f32<0x124>(0.f, give);          // row_ror:4
    t += dpp_f32<0x128>(0.f, t);                          // row_ror:8
    if (lanes > 16) t += __shfl_xor(t, 16);
    if (lanes > 32) t += __shfl_xor(t, 32);
    return t;
  }
};

// Three sums over the workgroup at once; `scratch` holds 3 kWaves floats.
__device__ __forceinline__ void block_sum3(float (&v)[3], float* scratch) {
  const int wave = threadIdx.x / kWaveSize;
#pragma unroll
  for (int i = 0; i < 3; ++i) v[i] = wave_sum(v[i]);
  __syncthreads();
  if ((threadIdx.x & (kWaveSize - 1)) == 0)
#pragma unroll
    for (int i = 0; i < 3; ++i) scratch[i * kWaves + wave] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    v[i] = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) v[i] += scratch[i * kWaves + w];
  }
}

__device__ __forceinline__ void clear_part(Smem& s, int rows) {
  if (static_cast<int>(threadIdx.x) < rows)
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s.part[w * kMaxRows + threadIdx.x] = 0.f;
}
__device__ __forceinline__ float row_total(const Smem& s, int row) {
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) t += s.part[w * kMaxRows + row];
  return t;
}

__device__ __forceinline__ float& xs_value(Smem& s, int i) { return s.xs[xs_at(i)]; }

// A thread's elements of a vector: tid, tid + 512, .., the first kHeld of them in registers.
constexpr int kHeld = 4, kHeldSpan = kHeld * kThreads;
using Look = Units<kHeld>;

// Behind a first look at the first kHeldSpan of them: units v[0 .. n) -> xs.
template <class F>
__device__ __forceinline__ void load_vector(const DecodeParams& p, Smem& s, const Op& o, Look& look, const uint64_t* v, int n, uint32_t tag, F&& seen) {
  const int tid = threadIdx.x;
  look.wait(p, s, o, v, tid, kThreads, n, tag);
  seen();
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kThreads < n) xs_value(s, tid + j * kThreads) = look[j];
  constexpr int kBatch = 12;
#pragma unroll 1
  for (int base = kHeldSpan; base < n; base += kBatch * kThreads) {
    Units<kBatch> more;
    more.ask(v, base + tid, kThreads, n);
    more.wait(p, s, o, v, base + tid, kThreads, n, tag);
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (base + tid + j * kThreads < n) xs_value(s, base + tid + j * kThreads) = more[j];
  }
}

__device__ __forceinline__ int token_of(const DecodeParams& p) {
  const long long t = *p.token_in;
  return t < 0 || t >= p.vocab ? 0 : static_cast<int>(t);
}
__device__ __forceinline__ float weight_sum(const float* w, int n) {
  float t = 0.f;
#pragma unroll 1
  for (int i = 0; i < n; ++i) t += w[i];
  return t;
}

// A thread's first elements of a [n] vector that no one writes.
__device__ __forceinline__ void load_ahead(float (&v)[kHeld], const float* from, int n) {
#pragma unroll
  for (int j = 0; j < kHeld; ++j) v[j] = from[min(static_cast<int>(threadIdx.x) + j * kThreads, n - 1)];
}

// RMS norm of the sublayer input -> xs; `ahead`: the thread's first norm weights.  `first`: the input is the embedding seen through the first layer's
// weights (their sum).
template <class F>
__device__ __forceinline__ void norm_to_xs(const DecodeParams& p, Smem& s, const Op& o, Look& look, uint32_t tag, const float* weight, const float (&ahead)[kHeld], bool first,
                                           const float* hc_in, F&& seen) {
  const int D = p.width, tid = threadIdx.x;
  const u16* e = p.embed;
  float g = 0.f;
  if (first) {
    e += static_cast<size_t>(token_of(p)) * D;
    g = weight_sum(hc_in, p.streams);
  } else {
    look.wait(p, s, o, p.u, tid, kThreads, D, tag);
  }
  seen();
  float v[kHeld], sq = 0.f;
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    const int i = tid + j * kThreads;
    v[j] = i < D ? first ? bf2f(e[i]) * g : look[j] : 0.f;
    sq = fmaf(v[j], v[j], sq);
  }
#pragma unroll 1
  for (int base = kHeldSpan; base < D; base += kHeldSpan) {
    Look more;
    if (!first) {
      more.ask(p.u, base + tid, kThreads, D);
      more.wait(p, s, o, p.u, base + tid, kThreads, D, tag);
    }
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const int i = base + tid + j * kThreads;
      if (i < D) {
        const float t = first ? bf2f(e[i]) * g : more[j];
        sq = fmaf(t, t, sq);
        xs_value(s, i) = t;
      }
    }
  }
  const float inv = 1.f / sqrtf(block_sum(sq, s.scratch) / p.width_true + p.eps);
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kThreads < D) xs_value(s, tid + j * kThreads) = v[j] * ahead[j] * inv;
#pragma unroll 1
  for (int i = kHeldSpan + tid; i < D; i += kThreads) xs_value(s, i) = xs_value(s, i) * weight[i] * inv;
}

// A copy of the plain residual and, behind it, what the run that leaves it adds.  (Two of both: a run's first outputs may be ready before the last of the
// workgroups that read the run before has read it.)
__device__ __forceinline__ uint64_t* copy_of(const DecodeParams& p, int copy) { return p.sums + static_cast<size_t>(copy) * (2 + QMK_HYBRID_MAX_BRANCHES) * p.width; }

// First looks at what makes the plain residual.
struct ResidualLook {
  Look x, a, b;
  const uint64_t *x_at, *a_at, *b_at;
  uint32_t x_tag, a_tag, b_tag;
  __device__ __forceinline__ void ask(const DecodeParams& p, const Plan& plan) {
    const int D = p.width, tid = threadIdx.x;
    x_at = uniform(plan.sum[0]);
    a_at = uniform(plan.sum[1]);
    b_at = uniform(plan.sum[2]);
    x_tag = uniform(plan.sum_tag[0]);
    a_tag = uniform(plan.sum_tag[1]);
    b_tag = uniform(plan.sum_tag[2]);
    x.ask(x_at, tid, kThreads, D);
    a.ask(a_at, tid, kThreads, D);
    b.ask(b_at, tid, kThreads, D);
  }
};

// The plain residual as a run (or the model's norm, or a loop's pass) reads it: the copy `x_from` plus what the run `prev`
// left.  normed: its norm under `weight` -> xs (`ahead`: the thread's first weights); otherwise [x; embedding] -> xs.
// keep: also leaves the sum in copy `x_to`.
template <class F>
__device__ __forceinline__ void residual_to_xs(const DecodeParams& p, Smem& s, const Op& o, LayerRef& l, int lead, ResidualLook& look, bool normed, bool keep, const float* weight,
                                               const float (&ahead)[kHeld], F&& seen) {
  const int D = p.width, tid = threadIdx.x;
  const u16* e = p.embed;
  const bool embed = l.x_from < 0, added = l.prev >= 0;
  if (embed || !normed) e += static_cast<size_t>(token_of(p)) * D;
  LayerRef& run = layer_of(p, added ? l.prev : 0);
  const bool two = added && run.branches == 2;
  const float *wa = nullptr, *wb = nullptr;
  if (two) {
    wa = run.out_norm;
    wb = layer_of(p, l.prev + 1).out_norm;
  }
  // x and a lone branch in `v`; two branches in `a` and `b`, their norm weights in `na` and `nb`
  auto fetch = [&](ResidualLook& k, int first, float (&v)[kHeld], float (&a)[kHeld], float (&b)[kHeld], float (&na)[kHeld], float (&nb)[kHeld]) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const int i = min(first + j * kThreads, D - 1);
      v[j] = a[j] = b[j] = na[j] = nb[j] = 0.f;
      if (two) {
        na[j] = wa[i];
        nb[j] = wb[i];
      }
      if (embed) v[j] = bf2f(e[i]);
    }
    if (!embed) k.x.wait(p, s, o, look.x_at, first, kThreads, D, look.x_tag);
    if (added) k.a.wait(p, s, o, look.a_at, first, kThreads, D, look.a_tag);
    if (two) k.b.wait(p, s, o, look.b_at, first, kThreads, D, look.b_tag);
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const bool in = first + j * kThreads < D;
      if (!embed) v[j] = k.x[j];
      if (two) {
        a[j] = in ? k.a[j] : 0.f;
        b[j] = in ? k.b[j] : 0.f;
      } else if (added) {
        v[j] += k.a[j];
      }
      if (!in) v[j] = 0.f;
    }
  };
  auto again = [&](ResidualLook& k, int first) {
    k.x.ask(look.x_at, first, kThreads, D);
    k.a.ask(look.a_at, first, kThreads, D);
    k.b.ask(look.b_at, first, kThreads, D);
  };
  float v[kHeld], a[kHeld], b[kHeld], na[kHeld], nb[kHeld];
  float sum[3] = {0.f, 0.f, 0.f};
  fetch(look, tid, v, a, b, na, nb);
  seen();
  float sa = 0.f, sb = 0.f;
  if (two) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      sum[0] = fmaf(a[j], a[j], sum[0]);
      sum[1] = fmaf(b[j], b[j], sum[1]);
    }
#pragma unroll 1
    for (int base = kHeldSpan; base < D; base += kHeldSpan) {
      Look ma, mb;
      ma.ask(look.a_at, base + tid, kThreads, D);
      mb.ask(look.b_at, base + tid, kThreads, D);
      ma.wait(p, s, o, look.a_at, base + tid, kThreads, D, look.a_tag);
      mb.wait(p, s, o, look.b_at, base + tid, kThreads, D, look.b_tag);
#pragma unroll
      for (int j = 0; j < kHeld; ++j) {
        const bool in = base + tid + j * kThreads < D;
        const float ta = in ? ma[j] : 0.f, tb = in ? mb[j] : 0.f;
        sum[0] = fmaf(ta, ta, sum[0]);
        sum[1] = fmaf(tb, tb, sum[1]);
      }
    }
    block_sum3(sum, s.scratch);
    const float scale = run.out_scale;
    sa = scale / sqrtf(sum[0] / p.width_true + p.eps);
    sb = scale / sqrtf(sum[1] / p.width_true + p.eps);
#pragma unroll
    for (int j = 0; j < kHeld; ++j) v[j] = fmaf(b[j] * nb[j], sb, fmaf(a[j] * na[j], sa, v[j]));
  }
  uint64_t* x_to = copy_of(p, l.x_to);
  const uint32_t kept = tag_of(lead, 0);
  float total = 0.f;
  auto take = [&](int i, float t) {
    total += t;
    if (keep) put_unit(x_to + i, t, kept);
    if (!normed) {
      xs_value(s, i) = t;
      xs_value(s, D + i) = bf2f(e[i]);
    }
  };
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kThreads < D) take(tid + j * kThreads, v[j]);
#pragma unroll 1
  for (int base = kHeldSpan; base < D; base += kHeldSpan) {
    ResidualLook more;
    float t[kHeld], ta[kHeld], tb[kHeld], ua[kHeld], ub[kHeld];
    again(more, base + tid);
    fetch(more, base + tid, t, ta, tb, ua, ub);
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const int i = base + tid + j * kThreads;
      if (i >= D) continue;
      if (two) t[j] = fmaf(tb[j] * ub[j], sb, fmaf(ta[j] * ua[j], sa, t[j]));
      take(i, t[j]);
      if (normed) xs_value(s, i) = t[j];
    }
  }
  if (!normed) return;
  const float mean = l.norm == QMK_NORM_LAYER ? block_sum(total, s.scratch) / p.width_true : 0.f;
  auto centred = [&](int i, float t) { return i < p.width_true ? t - mean : 0.f; };   // storage columns behind the true width stay zero
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    v[j] = centred(tid + j * kThreads, v[j]);
    sq = fmaf(v[j], v[j], sq);
  }
#pragma unroll 1
  for (int i = kHeldSpan + tid; i < D; i += kThreads) {
    const float t = centred(i, xs_value(s, i));
    sq = fmaf(t, t, sq);
    xs_value(s, i) = t;
  }
  const float inv = 1.f / sqrtf(block_sum(sq, s.scratch) / p.width_true + p.eps);
#pragma unroll
  for (int j = 0; j < kHeld; ++j)
    if (tid + j * kThreads < D) xs_value(s, tid + j * kThreads) = v[j] * ahead[j] * inv;
#pragma unroll 1
  for (int i = kHeldSpan + tid; i < D; i += kThreads) xs_value(s, i) = xs_value(s, i) * weight[i] * inv;
}

// What a gla or delta entry left in xs, head by head, a wave each: RMS norm over the head's values, weight, output gate.  The first head's gates are asked for ahead
// of the wait, the others' while the head before is normed.
struct HeadGates {
  static constexpr int kPer = kMaxHeadDim / kWaveSize;
  Units<kPer> g;
  __device__ __forceinline__ static const uint64_t* of(const DecodeParams& p, LayerRef& l, int head) {
    return p.proj + l.proj_at + (l.type == QMK_MIXER_DELTA ? l.in_rows : 2 * l.heads * l.head_dim + l.mix_width) + min(head, l.heads - 1) * l.v_dim;
  }
  __device__ __forceinline__ void ask(const DecodeParams& p, LayerRef& l, int head) { g.ask(of(p, l, head), threadIdx.x & (kWaveSize - 1), kWaveSize, l.v_dim); }
};
__device__ __forceinline__ void norm_heads(const DecodeParams& p, Smem& s, const Op& o, LayerRef& l, HeadGates& gates) {
  constexpr int kPer = HeadGates::kPer;
  const int lane = threadIdx.x & (kWaveSize - 1), wave = uniform(threadIdx.x / kWaveSize), n = l.v_dim;
  __syncthreads();
#pragma unroll 1
  for (int head = wave; head < l.heads; head += kWaves) {
    HeadGates next;
    next.ask(p, l, head + kWaves);
    gates.g.wait(p, s, o, HeadGates::of(p, l, head), lane, kWaveSize, n, tag_of(o.layer, 0));
    float v[kPer], sq = 0.f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = j * kWaveSize + lane;
      v[j] = i < n ? s.xs[xs_at(head * n + i)] : 0.f;
      sq = fmaf(v[j], v[j], sq);
    }
    const float inv = 1.f / sqrtf(wave_sum(sq) / l.v_true + p.eps);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = j * kWaveSize + lane;
      if (i < n) s.xs[xs_at(head * n + i)] = v[j] * inv * (gates.g[j] * l.vec0[i]);
    }
    gates = next;
  }
}

// log(1 + e^z) and the decays of the gated recurrences
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
template <class Layer>
__device__ __forceinline__ float delta_decay(const Layer& l, int head, float z) { return expf(l.vec1[head] * softplus(z)); }
template <class Layer>
__device__ __forceinline__ float gla_decay(const Layer& l, float z) { return expf(-softplus(-z) * l.decay_scale); }
template <class Layer>
__host__ __device__ constexpr int conv_channels(const Layer& l) { return 2 * l.kv_heads * l.head_dim + l.heads * l.v_dim; }
__device__ __forceinline__ float soft_cap(float z, float cap) { return cap > 0.f ? cap * tanhf(z / cap) : z; }

template <class Layer>
__device__ __forceinline__ void rotate(const Layer& l, int position, int d, float& a, float& b) {
  if (d >= l.rot_true) return;
  const size_t at = static_cast<size_t>(position) * (l.rot_true / 2) + (d >> 1);
  const float c = l.rope_cos[at], sn = l.rope_sin[at];
  const float x = a * c - b * sn;
  b = b * c + a * sn;
  a = x;
}

// ---- the ops that stream weight rows: one body, so that the streaming code exists once ----
// rows of the matrix this instruction covers; false: an operand is out of range
struct Rows {
  const u16* w;
  int rows, columns;
};
__device__ __forceinline__ bool rows_of(const DecodeParams& p, LayerRef& l, const Op& o, Rows& g) {
  const int D = p.width;
  auto set = [&](const u16* w, long long row, int rows, int columns) {
    g.w = w + row * columns;
    g.rows = rows;
    g.columns = columns;
    return o.start >= 0 && o.count > 0 && rows <= kMaxRows;
  };
  switch (o.opcode) {
    case OP_IN_PROJECT:
      return o.sub >= 0 && o.sub < 5 && !((o.start | o.count) & 1) && o.start + o.count <= l.in_rows && set(l.in_w, o.start, o.count, D);
    case OP_LRU_STEP:
      return l.type == QMK_MIXER_RGLRU && o.sub >= 0 && o.sub < l.blocks && o.start + o.count <= l.block_dim &&
             set(l.mid_w, static_cast<long long>(o.sub) * 2 * l.block_dim + 2 * o.start, 2 * o.count, l.block_dim);
    case OP_LATENT_ABSORB:
      return l.type == QMK_MIXER_LATENT && o.sub >= 0 && o.sub < l.heads && o.start + o.count <= l.rank &&
             set(l.mid_w, static_cast<long long>(o.sub) * l.rank + o.start, o.count, l.head_dim);
    case OP_LATENT_VALUE:
      return l.type == QMK_MIXER_LATENT && o.sub >= 0 && o.sub < l.heads && o.start + o.count <= l.v_dim && o.extra > 0 &&
             o.extra <= p.max_splits && o.extra <= kMaxParts && set(l.uv_w, static_cast<long long>(o.sub) * l.v_dim + o.start, o.count, l.rank);
    case OP_WKV_STEP:
      return l.type == QMK_MIXER_WKV && o.sub >= 0 && o.sub < l.heads && l.head_dim <= kMaxHeadDim &&
             set(l.mid_w, static_cast<long long>(o.sub) * l.head_dim, l.head_dim, l.rank);
    case OP_OUT_PROJECT:
      if (p.streams > 0 && o.count > kMaxOutRows) return false;
      if (o.sub == 1) return l.has_mlp && o.start + o.count <= D && set(l.down_w, o.start, o.count, l.ff);
      return l.type <= QMK_MIXER_DELTA && o.start + o.count <= D && set(l.o_w, o.start, o.count, l.mix_width);
    case OP_UP_GATE: return l.has_mlp && o.start + o.count <= l.ff && set(l.mlp_w, 2LL * o.start, 2 * o.count, D);
    case OP_STATE_STEP: {
      if ((l.type != QMK_MIXER_GLA && l.type != QMK_MIXER_DELTA) || o.sub < 0 || o.sub >= l.heads || l.head_dim > kMaxHeadDim) return false;
      return o.count <= kStateColumns && o.start + o.count <= l.v_dim && set(l.mid_w, static_cast<long long>(o.sub) * l.head_dim, l.head_dim, l.rank);
    }
    case OP_GATE: return l.type == QMK_MIXER_DELTA && o.start + o.count <= l.mix_width && set(l.gate_w, o.start, o.count, l.gate_rank);
    case OP_JOIN: return l.type == QMK_ENTRY_JOIN && o.start + o.count <= D && set(l.in_w, o.start, o.count, 2 * D);
    case OP_LM_HEAD: return (p.streams > 0 || l.type == QMK_ENTRY_FINAL) && o.start + o.count <= p.vocab_rows && set(p.head, o.start, o.count, D);
    default: return false;
  }
}

// The plan of an instruction, by one wave.
template <bool PLAIN>
__device__ __forceinline__ void plan_of(const DecodeParams& p, Smem& s, int index) {
  const int32_t* words = s.inst[index & 1];
  auto operand = [&](int w) { return static_cast<int>(uniform(words[w])); };
  const Op o{index, operand(0), operand(1), operand(2), operand(3), operand(4), operand(5), operand(6), operand(7), operand(8)};
  Plan t{};
  if (o.opcode != OP_NOOP && o.layer >= 0 && o.layer < p.num_layers) {
    LayerRef& l = layer_of(p, o.layer);
    Rows m{};
    if (rows_of(p, l, o, m)) {
      const int op = o.opcode, D = p.width;
      const bool delta = l.type == QMK_MIXER_DELTA;
      t.w = m.w;
      t.rows = m.rows;
      t.columns = m.columns;
      t.from = p.proj;
      t.length = m.columns;
      t.tag = tag_of(o.layer, 0);
      if (op == OP_OUT_PROJECT) {
        t.from = p.mix + (o.sub == 1 ? l.ff_at : l.mix_at);
        t.tag = tag_of(o.layer, o.sub);
      } else if constexpr (!PLAIN) {
        if (op == OP_IN_PROJECT || op == OP_UP_GATE || op == OP_LM_HEAD) {
          const int before = op == OP_IN_PROJECT ? max(o.layer - 1, 0) : o.layer;
          t.from = p.u;
          t.tag = tag_of(before, op == OP_UP_GATE ? 0 : layer_of(p, before).has_mlp != 0);
        } else if (op == OP_LRU_STEP) {
          t.from = p.proj + l.mix_width + o.sub * l.block_dim;
        } else if (op == OP_LATENT_ABSORB) {
          t.from = p.proj + o.sub * l.q_stride;
          t.length = l.q_stride;      // (with what lies behind the head's query: whoever makes it is waited for too)
        } else if (op == OP_WKV_STEP) {
          t.from = p.proj + 4 * l.heads * l.head_dim;
        } else {      // OP_LATENT_VALUE: merged of parts
          t.length = 1;
        }
      } else if (op == OP_STATE_STEP) {
        t.from = p.proj + l.proj_at + 2 * l.kv_heads * l.head_dim + l.heads * l.v_dim * (delta ? 1 : 2);
      } else if (op == OP_GATE) {
        t.from = p.proj + l.proj_at + conv_channels(l) + l.rank;
      } else {
        const int first = o.layer - l.branch;
        LayerRef& lead = layer_of(p, first);
        const int prev = lead.prev, copy = lead.x_from;
        int writer = first - 1;      // whose lead has left copy x_from: the last one ahead that leaves that copy
        if (copy >= 0) {
#pragma unroll 1
          while (writer > 0 && (layer_of(p, writer).branch != 0 || layer_of(p, writer).x_to != copy)) --writer;
        }
        LayerRef& run = layer_of(p, max(prev, 0));
        uint64_t* out = copy_of(p, prev >= 0 ? run.x_to : 0) + D;
        const bool ff = prev >= 0 && run.has_mlp;      // (the down projection has added x to its rows)
        t.sum[0] = ff ? out + static_cast<size_t>(QMK_HYBRID_MAX_BRANCHES) * D : copy_of(p, max(copy, 0));
        t.sum[1] = out;
        t.sum[2] = out + (prev >= 0 && run.branches == 2 ? D : 0);
        t.sum_tag[0] = ff ? tag_of(prev, 1) : tag_of(writer, 0);
        t.sum_tag[1] = tag_of(prev, 0);
        t.sum_tag[2] = tag_of(prev + 1, 0);
      }
    }
  }
  if ((threadIdx.x & (kWaveSize - 1)) == 0) s.plan[index & 1] = t;
}
// The last wave plans the instruction behind this one while its first requests are on their way.
template <bool PLAIN>
__device__ __forceinline__ void plan_next(const DecodeParams& p, Smem& s, const Op& o) {
  if (uniform(threadIdx.x) >= kThreads - kWaveSize) plan_of<PLAIN>(p, s, o.index + 1);
}
// The last norm's input has come, so everything before it has been read: every workgroup clears its share of those units, once.
__device__ __forceinline__ void clear_units(uint64_t* at, int count, int first, int step) {
#pragma unroll 1
  for (int i = first; i < count; i += step) __hip_atomic_store(at + i, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void clear_share(const DecodeParams& p, Smem& s, int copy) {      // copy: of the plain residual, that the last norm has read
  const int first = blockIdx.x * kThreads + threadIdx.x, step = gridDim.x * kThreads;
  clear_units(p.units, p.early_units, first, step);
  if (copy >= 0) clear_units(copy_of(p, 1 - copy), (2 + QMK_HYBRID_MAX_BRANCHES) * p.width, first, step);
  if (threadIdx.x == 0) s.ctl[2] = 1;
}

// PLAIN: the kernel of a plain residual (its entries, its ops), which holds none of the other kernel's code, nor that of its.
template <class T, bool PLAIN>
__device__ __forceinline__ bool op_rows(const DecodeParams& p, Smem& s, const Op& o) {
  constexpr bool plain = PLAIN;
  constexpr unsigned kOps = 1u << OP_IN_PROJECT | 1u << OP_OUT_PROJECT | 1u << OP_UP_GATE | 1u << OP_LM_HEAD |
                            (plain ? 1u << OP_STATE_STEP | 1u << OP_JOIN | 1u << OP_GATE : 1u << OP_LRU_STEP | 1u << OP_LATENT_ABSORB | 1u << OP_LATENT_VALUE | 1u << OP_WKV_STEP);
  const int op = o.opcode;
  if (!(kOps >> op & 1)) return bad_operand(p, o, o.opcode);
  __builtin_assume(kOps >> op & 1);
  const Plan& plan = s.plan[o.index & 1];
  struct {
    const u16* w;
    int rows, columns;
  } const m{uniform(plan.w), static_cast<int>(uniform(plan.rows)), static_cast<int>(uniform(plan.columns))};
  if (m.rows == 0) return bad_operand(p, o, o.start);
  const int tid = threadIdx.x, D = p.width, S = p.streams;
  const uint32_t tag = tag_of(o.layer, 0);     // of this entry's projections and what its mixer leaves
  const bool normed = op == OP_IN_PROJECT || op == OP_UP_GATE || op == OP_LM_HEAD;
  const bool reads_x = plain && (normed || op == OP_JOIN);
  const bool down = op == OP_OUT_PROJECT && o.sub == 1;
  const bool first = !plain && o.layer == 0 && (op == OP_IN_PROJECT || (op == OP_OUT_PROJECT && o.sub == 0));

  // The first look at the vector, ahead of everything: the last workgroup of a stage finds it there, and has it normed while its rows are on their way.  (A look
  // behind the rows' requests returns behind the rows.)
  const uint64_t* from = uniform(plan.from);
  const int length = uniform(plan.length);
  const uint32_t from_tag = uniform(plan.tag);
  Look look;
  ResidualLook residual;
  if (reads_x) residual.ask(p, plan);
  else look.ask(from, tid, kThreads, length);
  __builtin_amdgcn_sched_barrier(0);
  RowStream g;
  g.start(m.w, m.rows, m.columns);
  clear_part(s, m.rows);
  LayerRef& l = layer_of(p, o.layer);
  const int type = l.type;
  __builtin_assume(plain ? type >= QMK_MIXER_GLA : type <= QMK_MIXER_WKV);
  const int lead_at = o.layer - l.branch;      // the run's first entry
  LayerRef& lead = layer_of(p, lead_at);
  const bool wkv_in = !plain && op == OP_IN_PROJECT && type == QMK_MIXER_WKV;

  // Asked for ahead of the wait: what no one writes in this launch, or this workgroup alone.  Thread r of the workgroup owns row r.  (A variable of its own for
  // everything: where values of several branches meet in one register, this compiler waits for them, and so for all rows ahead of them.)
  const int row = o.start + tid;
  const bool mine = tid < m.rows;
  const float* norm = plain ? lead.norm1 : op == OP_IN_PROJECT ? l.norm1 : op == OP_UP_GATE ? l.norm2 : p.final_norm;
  const int channels = type == QMK_MIXER_DELTA ? conv_channels(l) : l.mix_width;
  const size_t shift_copy = type == QMK_MIXER_WKV ? static_cast<size_t>(D) : static_cast<size_t>(l.taps - 1) * channels;
  const float* shift_old = l.shift + (static_cast<size_t>(p.slot) * 2 + p.flip) * shift_copy;
  float* shift_new = l.shift + (static_cast<size_t>(p.slot) * 2 + 1 - p.flip) * shift_copy;
  const float* mu = l.vec2 + static_cast<size_t>(o.sub) * D;
  float norm_weight[kHeld], before[kHeld], mix_weight[kHeld];
  // OP_IN_PROJECT: a convolution's inputs and weights, the present one's last
  const bool convolves = op == OP_IN_PROJECT && type == (plain ? QMK_MIXER_DELTA : QMK_MIXER_RGLRU);
  const int channel = plain ? row : row - l.mix_width;
  const bool conv_row = convolves && mine && channel >= 0 && channel < channels;
  float in_bias = 0.f, conv_bias = 0.f, conv_in[kFewTaps - 1], conv_weight[kFewTaps - 1], conv_now = 0.f;
  float lru_bias, lru_rate, lru_state;
  float wkv_state[kMaxStreams], wkv_decay, wkv_bonus, wkv_norm;
  float step_bias;
  float mixes[kMaxStreams], streams[kMaxStreams], out_weight, next_weight;
  float held[kStateRows];      // OP_STATE_STEP: this thread's rows of the state
  float* state = nullptr;
  if (normed) load_ahead(norm_weight, norm, D);
  if (wkv_in) {
    load_ahead(before, shift_old, D);
    load_ahead(mix_weight, mu, D);
  }
  if (conv_row) {
    if constexpr (!plain) conv_bias = l.vec1[channel];
#pragma unroll
    for (int j = 0; j < kFewTaps - 1; ++j) {
      if (j < l.taps - 1 && l.taps <= kFewTaps) {
        conv_in[j] = shift_old[static_cast<size_t>(j) * channels + channel];
        conv_weight[j] = l.vec2[static_cast<size_t>(j) * channels + channel];
      }
    }
    conv_now = l.vec2[static_cast<size_t>(l.taps - 1) * channels + channel];
  }
  if (!plain && convolves && mine) in_bias = l.in_b[row];
  if (!plain && op == OP_LRU_STEP && mine) {   // rows (r, i) of a channel: neighbouring threads
    const int c = o.sub * l.block_dim + o.start + (tid >> 1);
    state = l.state + static_cast<size_t>(p.slot) * l.mix_width + c;
    lru_bias = l.mid_b[2 * c + (tid & 1)];
    lru_rate = l.vec0[c];
    lru_state = *state;
  }
  if (!plain && op == OP_WKV_STEP) {
    const int n = l.head_dim, groups = kThreads / n, e = tid % n, group = tid / n;
    state = l.state + (static_cast<size_t>(p.slot) * l.heads + o.sub) * n * n + e;
#pragma unroll
    for (int j = 0; j < kMaxStreams; ++j) wkv_state[j] = state[min(group + j * groups, n - 1) * n];      // (rows behind the last one are not used)
    const int at = o.sub * n + min(tid, n - 1);
    wkv_decay = l.mid_b[at];
    wkv_bonus = l.vec1[at];
    wkv_norm = l.vec0[at];
  }
  if (plain && op == OP_STATE_STEP) {
    const int n = o.count, groups = kThreads / n, e = tid % n, group = tid / n;
    state = l.state + (static_cast<size_t>(p.slot) * l.heads + o.sub) * l.head_dim * l.v_dim + o.start + e;
#pragma unroll
    for (int j0 = 0; j0 < kStateRows; j0 += kStateBatch) {
      if (j0 * groups < l.head_dim) {
#pragma unroll
        for (int j = j0; j < j0 + kStateBatch; ++j) held[j] = state[static_cast<size_t>(min(group + j * groups, l.head_dim - 1)) * l.v_dim];
      }
    }
    static_assert(3 * kStateVector + kStateColumns <= 3072 && kStateVector <= 2 * kThreads, "q, k, decays and values in aux");
#pragma unroll
    for (int i = 0; i < 3; ++i)
      for (int at = l.head_dim + tid; at < kStateVector; at += kThreads) s.aux[i * kStateVector + at] = 0.f;
    if (mine) step_bias = l.mid_b[o.sub * l.head_dim + tid];
  }
  if (!plain && op == OP_OUT_PROJECT) {
    // Eight lanes per row, one per stream: the stream's column of the mix, its output weight and its weight in the next sublayer's input.
    const int q = min(tid & 7, S - 1);
    const float* hc = l.hc + (down ? S * (S + 2) : 0) + S;
#pragma unroll
    for (int f = 0; f < kMaxStreams; ++f) mixes[f] = hc[S + min(f, S - 1) * S + q];
    out_weight = hc[q];
    next_weight = (down ? l.next2 : l.next1)[q];
    // All streams of the rows this workgroup owns: every output projection of a schedule deals the rows to the queues alike.  Their last writer is this thread's
    // wave, which has waited for its own later requests since, or does here.
    const int r = o.start + min(tid >> 3, m.rows - 1);
    if (s.ctl[3] == OP_OUT_PROJECT) release_stores();
    if (first) {
      const float e = bf2f(p.embed[static_cast<size_t>(token_of(p)) * D + r]);
#pragma unroll
      for (int f = 0; f < kMaxStreams; ++f) streams[f] = e;
    } else {
#pragma unroll
      for (int f = 0; f < kMaxStreams; ++f) streams[f] = ld_shared_f32(p.x + static_cast<size_t>(min(f, S - 1)) * D + r);
    }
  }
  HeadGates gates;
  const bool norms_heads = plain && op == OP_OUT_PROJECT && !down && type != QMK_MIXER_ATTENTION;
  if (norms_heads) gates.ask(p, l, uniform(tid / kWaveSize));
  stamp(p, s, 0);
  if constexpr (!plain) plan_next<PLAIN>(p, s, o);
  if (!plain && op == OP_LATENT_VALUE && !wait_stage(p, s, o)) return false;

  // The activation vector.
  float lru_gate, value_gate, wkv_gate, beta, unit_dot;
  if (reads_x) {
    residual_to_xs(p, s, o, lead, lead_at, residual, normed, op == OP_IN_PROJECT && o.extra, norm, norm_weight, [&] { g.rest(); });
  } else if (normed) {
    norm_to_xs(p, s, o, look, from_tag, norm, norm_weight, first, l.hc, [&] { g.rest(); });
    if (wkv_in) {
      auto mix = [&](int i, float was, float weight) {
        const float h = xs_value(s, i);
        if (o.extra) shift_new[i] = h;
        xs_value(s, i) = h + (was - h) * weight;
      };
#pragma unroll
      for (int j = 0; j < kHeld; ++j)
        if (tid + j * kThreads < D) mix(tid + j * kThreads, before[j], mix_weight[j]);
#pragma unroll 1
      for (int i = kHeldSpan + tid; i < D; i += kThreads) mix(i, shift_old[i], mu[i]);
    }
  } else if (!plain && op == OP_LATENT_VALUE) {   // merge the parts of this head
    const int heads16 = (l.heads + 15) & ~15, parts = o.extra;
    const float* sums = p.part + static_cast<size_t>(o.sub) * l.rank;
    const int pitch = heads16 * l.rank;
    if (tid < parts) {
      const uint64_t ml = ld_shared64(p.ml + (static_cast<size_t>(tid) * heads16 + o.sub) * 2);
      s.aux[tid] = __uint_as_float(static_cast<uint32_t>(ml));
      s.aux[kMaxParts + tid] = __uint_as_float(static_cast<uint32_t>(ml >> 32));
    }
    constexpr int kBatch = 16;
    static_assert(kMaxRank <= kThreads && kMaxParts <= kWaveSize, "one thread per latent element, one lane per part");
    const bool in = tid < l.rank;
    float v[kBatch];
    const float* column = sums + min(tid, l.rank - 1);
    auto request = [&](int base) {   // no branches: sixteen requests leave back to back
#pragma unroll
      for (int j = 0; j < kBatch; ++j) v[j] = ld_shared_f32(column + min(base + j, parts - 1) * pitch);
    };
    request(0);
    value_gate = unit_of(p, s, o, p.proj + l.heads * l.q_stride + o.sub * l.v_dim + o.start + min(tid, m.rows - 1), tag);
    __syncthreads();
    if (tid < kWaveSize) {   // weights of the parts
      const float mx = tid < parts ? s.aux[tid] : -INFINITY, top = wave_max(mx);
      const float w = exp2_fast(mx - top), sum = wave_sum(tid < parts ? w * s.aux[kMaxParts + tid] : 0.f);
      s.aux[tid] = tid < parts ? w / sum : 0.f;
    }
    __syncthreads();
    float acc = 0.f;
#pragma unroll 1
    for (int base = 0; base < parts; base += kBatch) {
      if (base != 0) request(base);
#pragma unroll
      for (int j = 0; j < kBatch; ++j) acc = fmaf(s.aux[base + j], v[j], acc);
    }
    if (in) s.xs[xs_at(tid)] = acc;
    g.rest();
  } else {
    load_vector(p, s, o, look, from, length, from_tag, [&] { g.rest(); });
    if (plain && op == OP_STATE_STEP) {
      // query, key (unit vectors for the delta rule) and values of the head
      const bool delta = type == QMK_MIXER_DELTA;
      const int dim = l.head_dim, keys = l.kv_heads * dim, kv = o.sub / (l.heads / l.kv_heads), c = min(tid, dim - 1);
      const uint64_t *proj = p.proj + l.proj_at, *steps = delta ? from + l.rank + l.gate_rank : proj;      // (all step sizes: whoever makes those of padding is waited for too)
      Gather<5> more{{proj + kv * dim + c, proj + keys + kv * dim + c, proj + 2 * keys + o.sub * l.v_dim + o.start + min(tid, o.count - 1), steps + (delta ? o.sub : 0),
                      steps + (delta ? min(tid, (l.heads + 15) / 16 * 16 - 1) : 0)}};
      more.ask();
      more.wait(p, s, o, tag);
      float q = more[0], k = more[1];
      const float v = more[2];
      beta = more[3];
      if (tid >= dim) q = k = 0.f;
      if (tid < o.count) s.aux[3 * kStateVector + tid] = v;
      if (!delta) q *= l.q_scale;                       // (the projection is left unscaled)
      float dots[3] = {q * q, k * k, q * k};
      block_sum3(dots, s.scratch);
      if (delta) {
        const float iq = l.q_scale / sqrtf(dots[0] + 1e-6f), ik = 1.f / sqrtf(dots[1] + 1e-6f);
        q *= iq;
        k *= ik;
        dots[2] *= iq * ik;
      }
      unit_dot = dots[2];
      if (tid < dim) {
        s.aux[tid] = q;
        s.aux[kStateVector + tid] = k;
      }
    } else if (!plain && op == OP_LRU_STEP) {
      lru_gate = unit_of(p, s, o, p.proj + o.sub * l.block_dim + o.start + (min(tid, m.rows - 1) >> 1), tag);
    } else if (!plain && op == OP_WKV_STEP) {
      const int n = l.head_dim, N = l.heads * n;
      const uint64_t* at = p.proj + o.sub * n + min(tid, n - 1);
      Gather<4> more{{at, at + N, at + 2 * N, at + 3 * N}};
      more.ask();
      more.wait(p, s, o, tag);
      wkv_gate = more[3];
      if (mine) {
        s.aux[tid] = more[0];
        s.aux[kMaxHeadDim + tid] = more[1];
        s.aux[2 * kMaxHeadDim + tid] = more[2];
        s.aux[4 * kMaxHeadDim + tid] = wkv_bonus;
      }
    }
    if (norms_heads) norm_heads(p, s, o, l, gates);
  }
  if (p.timeline != nullptr && tid == 0) s.t_wait = wall_clock64();
  __syncthreads();
  if (s.ctl[0] == 0) return false;
  stamp(p, s, 1);
  g.run(s);
  __syncthreads();
  stamp(p, s, 2);

  // What happens to the rows' sums; a pair of rows is a pair of lanes.
  float t = mine && (plain || op != OP_OUT_PROJECT) ? row_total(s, tid) : 0.f;
  static_assert(kMaxRows <= kThreads && kMaxStreams == 8, "one row per thread, eight values ahead");
  if (plain && op == OP_JOIN) {
    if (mine) put_unit(copy_of(p, l.x_to) + row, t, tag);
  } else if (op == OP_OUT_PROJECT && plain) {
    // (The feed-forward's rows with the residual that the run has read: its next reader looks at one vector less.)
    if (down) t += unit_of(p, s, o, copy_of(p, lead.x_to) + o.start + min(tid, m.rows - 1), tag_of(lead_at, 0));
    if (mine) put_unit(copy_of(p, lead.x_to) + static_cast<size_t>(1 + (down ? QMK_HYBRID_MAX_BRANCHES : l.branch)) * D + row, t, from_tag);
  } else if (op == OP_OUT_PROJECT) {
    const int r = tid >> 3, q = tid & 7;
    if (r < m.rows) {      // whole groups of eight lanes
      float now = out_weight * row_total(s, r);
#pragma unroll
      for (int f = 0; f < kMaxStreams; ++f)
        if (f < S) now = fmaf(mixes[f], streams[f], now);
      const float u = group8_sum(q < S ? next_weight * now : 0.f);
      if (q == 0) put_unit(p.u + o.start + r, u, from_tag);
      if (q < S) st_shared_f32(p.x + static_cast<size_t>(q) * D + o.start + r, now);
    }
  } else if (op == OP_UP_GATE) {
    const float up = dpp_f32<kDppQuadXor1>(0.f, t);
    if (mine && !(tid & 1)) put_unit(p.mix + l.ff_at + o.start + (tid >> 1), (l.act == QMK_ACT_SILU ? t * sigmoid(t) : gelu_tanh(t)) * up, tag_of(o.layer, 1));
  } else if (op == OP_IN_PROJECT) {
    const float pair = dpp_f32<kDppQuadXor1>(0.f, t);
    if (mine) {
      const int W = l.mix_width;
      int gate = 0;          // 1: sigmoid, 2: times sigmoid (silu), 3: gelu
      // Everything of the convolution but the current input; the kept inputs move up by one.
      auto convolved = [&](float bias) {
        float acc = bias;
        if (l.taps <= kFewTaps) {
#pragma unroll
          for (int j = 0; j < kFewTaps - 1; ++j) {
            if (j < l.taps - 1) {
              acc = fmaf(conv_weight[j], conv_in[j], acc);
              if (j > 0) shift_new[static_cast<size_t>(j - 1) * channels + channel] = conv_in[j];
            }
          }
        } else {
#pragma unroll 1
          for (int j = 0; j < l.taps - 1; ++j) {
            const float x = shift_old[static_cast<size_t>(j) * channels + channel];
            acc = fmaf(l.vec2[static_cast<size_t>(j) * channels + channel], x, acc);
            if (j > 0) shift_new[static_cast<size_t>(j - 1) * channels + channel] = x;
          }
        }
        if (l.taps > 1) shift_new[static_cast<size_t>(l.taps - 2) * channels + channel] = t;
        return fmaf(conv_now, t, acc);
      };
      if (!plain && type == QMK_MIXER_RGLRU) {
        t += in_bias;
        if (row < W) gate = 3;
        else t = convolved(conv_bias);
      } else if (!plain && type == QMK_MIXER_LATENT) {
        const int q_rows = l.heads * l.q_stride, g_rows = l.heads * l.v_dim;
        int d = -1;
        if (row < q_rows) d = row % l.q_stride - l.head_dim;
        else if (row < q_rows + g_rows) gate = 1;
        else d = row - q_rows - g_rows - l.rank;
        if (d >= 0 && d < l.rot_true) {
          const size_t at = static_cast<size_t>(p.position) * (l.rot_true / 2) + (d >> 1);
          const float c = l.rope_cos[at], sn = l.rope_sin[at];
          t = t * c + ((tid & 1) ? pair * sn : -(pair * sn));
        }
      } else if (plain && type == QMK_MIXER_ATTENTION) {
        const int q_rows = l.heads * l.q_stride, k_rows = l.kv_heads * l.head_dim, v_rows = l.kv_heads * l.v_dim;
        const int d = row < q_rows ? row % l.q_stride : row < q_rows + k_rows ? (row - q_rows) % l.head_dim : l.rot_true;
        if (d < l.rot_true) {
          const size_t at = static_cast<size_t>(p.position) * (l.rot_true / 2) + (d >> 1);
          const float c = l.rope_cos[at], sn = l.rope_sin[at];
          t = t * c + ((tid & 1) ? pair * sn : -(pair * sn));
        }
        if (row >= q_rows + k_rows + v_rows) gate = 1;
      } else if (plain && type == QMK_MIXER_DELTA) {
        if (row < channels) {
          t = convolved(0.f);
          gate = 2;
        } else if (row >= channels + l.rank + l.gate_rank) {
          gate = 1;
        }
      } else if (plain && type == QMK_MIXER_GLA) {
        const int from = 2 * l.heads * l.head_dim + l.heads * l.v_dim;
        if (row >= from && row < from + l.heads * l.v_dim) gate = 2;
      } else if (!plain && row >= 4 * W) {
        t = tanhf(t);
      } else if (!plain && row >= 3 * W) {
        gate = 2;
      }
      if (gate) {
        const float z = gate == 3 ? 1.5957691216057308f * (t + 0.044715f * t * t * t) : t;
        const float sg = sigmoid(z);
        t = gate == 1 ? sg : t * sg;
      }
      put_unit(p.proj + l.proj_at + row, t, tag);
    }
  } else if (!plain && op == OP_LRU_STEP) {
    const float gate = sigmoid(t + lru_bias), in_gate = dpp_f32<kDppQuadXor1>(0.f, gate);
    if (mine && !(tid & 1)) {
      const int c = o.start + (tid >> 1);
      const float log_a = gate * lru_rate;
      const float b = sqrtf(-expm1f(2.f * log_a)) * in_gate * s.xs[xs_at(c)];
      const float now = fmaf(expf(log_a), lru_state, b);
      *state = now;
      put_unit(p.mix + o.sub * l.block_dim + c, now * lru_gate, tag);
    }
  } else if (!plain && op == OP_LATENT_VALUE) {
    if (mine) put_unit(p.mix + o.sub * l.v_dim + row, t * value_gate, tag);
  } else if (!plain && op == OP_LATENT_ABSORB) {
    // What the attention's matrix tiles hold of it: in bf16 mode two rounded values a unit.
    if constexpr (sizeof(T) == 2) {
      const float odd = dpp_f32<kDppQuadXor1>(0.f, t);
      if (mine && !(tid & 1)) put_bits(p.absorbed + (o.sub * l.rank + row) / 2, f2bf2(t, odd), tag);
    } else {
      if (mine) put_unit(p.absorbed + o.sub * l.rank + row, t, tag);
    }
  } else if (!plain && op == OP_WKV_STEP) {
    const int n = l.head_dim, groups = kThreads / n, e = tid % n, group = tid / n;
    const float *r = s.aux, *k = r + kMaxHeadDim, *v = k + kMaxHeadDim, *w = v + kMaxHeadDim, *u = w + kMaxHeadDim;
    if (mine) s.aux[3 * kMaxHeadDim + tid] = expf(-expf(t + wkv_decay));
    __syncthreads();
    if (group < groups) {
      float acc = 0.f;
      auto key_row = [&](int i, float old) {
        const float kv = k[i] * v[e];
        acc = fmaf(r[i], fmaf(u[i], kv, old), acc);
        state[i * n] = fmaf(w[i], old, kv);
      };
#pragma unroll
      for (int j = 0; j < kMaxStreams; ++j)
        if (group + j * groups < n) key_row(group + j * groups, wkv_state[j]);
#pragma unroll 1
      for (int i = group + kMaxStreams * groups; i < n; i += groups) key_row(i, state[i * n]);
      s.xs[group * n + e] = acc;
    }
    __syncthreads();
    float val = 0.f;
    if (mine) {
#pragma unroll 4
      for (int i = 0; i < groups; ++i) val += s.xs[i * n + tid];
    }
    const float sq = block_sum(val * val, s.scratch);   // storage columns behind the true head size hold zeros
    const float inv = 1.f / sqrtf(sq / l.head_dim_true + p.eps);
    if (mine) put_unit(p.mix + o.sub * n + tid, val * inv * wkv_norm * wkv_gate, tag);
  } else if (plain && op == OP_STATE_STEP) {
    // S <- decay S, u = beta (v - S^T k), S <- S + k u^T, o = S^T q, with S^T k and S^T q taken together:
    // o = (decay S)^T q + (q . k) u.  Without the delta rule u = v.
    const bool delta = type == QMK_MIXER_DELTA;
    const int n = o.count, dim = l.head_dim, groups = kThreads / n, e = tid % n, group = tid / n;
    float *q = s.aux, *k = q + kStateVector, *w = k + kStateVector, *v = w + kStateVector;
    if (mine) w[tid] = delta ? delta_decay(l, o.sub, t + step_bias) : gla_decay(l, t + step_bias);
    __syncthreads();
    float ak = 0.f, aq = 0.f;
#pragma unroll
    for (int j0 = 0; j0 < kStateRows; j0 += kStateBatch) {
      if (j0 * groups < dim) {
#pragma unroll
        for (int j = j0; j < j0 + kStateBatch; ++j) {
          const int i = group + j * groups;
          held[j] *= w[i];
          ak = fmaf(k[i], held[j], ak);
          aq = fmaf(q[i], held[j], aq);
        }
      }
    }
    if (group < groups) {
      s.xs[group * n + e] = ak;
      s.xs[(groups + group) * n + e] = aq;
    }
    __syncthreads();
    ak = aq = 0.f;
#pragma unroll 4
    for (int i = 0; i < groups; ++i) {
      ak += s.xs[i * n + e];
      aq += s.xs[(groups + i) * n + e];
    }
    const float u = delta ? beta * (v[e] - ak) : v[e];
    if (tid < n) put_unit(p.mix + l.mix_at + o.sub * l.v_dim + o.start + tid, fmaf(unit_dot, u, aq), tag);
    stamp(p, s, 3);
    arrive_stage(p, o);      // (counted with the attention's parts of its stage, whose readers read nothing of it)
    if (group < groups) {
#pragma unroll
      for (int j0 = 0; j0 < kStateRows; j0 += kStateBatch) {
        if (j0 * groups < dim) {
#pragma unroll
          for (int j = j0; j < j0 + kStateBatch; ++j) {
            const int i = group + j * groups;
            const float now = fmaf(k[i], u, held[j]);
            if (i < dim) state[static_cast<size_t>(i) * l.v_dim] = now;
          }
        }
      }
    }
    return true;
  } else if (plain && op == OP_GATE) {
    if (mine) put_unit(p.proj + l.proj_at + l.in_rows + row, sigmoid(t), tag);
    arrive_stage(p, o);
  } else {   // OP_LM_HEAD
    if (plain) t = soft_cap(t * p.logit_scale, p.logit_softcap);
    if (mine) p.logits[row] = t;
    clear_share(p, s, plain ? l.x_from : -1);
    const bool real = mine && row < p.vocab;
    const float top = block_max(real ? t : -INFINITY, s.scratch);
    int where = wave_min_i32(real && t == top ? row : 0x7fffffff);   // smallest row among equals
    int* slots = reinterpret_cast<int*>(s.aux);
    if ((tid & (kWaveSize - 1)) == 0) slots[tid / kWaveSize] = where;
    __syncthreads();
    if (tid == 0) {
#pragma unroll 1
      for (int w = 1; w < kWaves; ++w) where = min(where, slots[w]);
      if (where != 0x7fffffff && (top > s.best_val || s.best_idx == 0x7fffffff)) {
        s.best_val = top;
        s.best_idx = where;
      }
    }
  }
  stamp(p, s, 3);
  return true;
}

// ---- matrix-core fragments: eight consecutive k per lane, for both element types.  An fp32 product of 32 k is eight
// 16x16x4 instructions, the j-th taking every lane's j-th element: the order of k is the same permutation on both sides.
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <class T>
struct Frag;
template <>
struct Frag<u16> {
  bf16x8_t v;
  __device__ __forceinline__ void set(int j, u16 e) { v[j] = __builtin_bit_cast(__bf16, e); }
};
template <>
struct Frag<float> {
  float v[8];
  __device__ __forceinline__ void set(int j, float e) { v[j] = e; }
};
__device__ __forceinline__ Frag<u16> load_frag(const u16* q) { return {*reinterpret_cast<const bf16x8_t*>(q)}; }
__device__ __forceinline__ Frag<float> load_frag(const float* q) {
  Frag<float> f;
  const float4 a = reinterpret_cast<const float4*>(q)[0], b = reinterpret_cast<const float4*>(q)[1];
  f.v[0] = a.x; f.v[1] = a.y; f.v[2] = a.z; f.v[3] = a.w;
  f.v[4] = b.x; f.v[5] = b.y; f.v[6] = b.z; f.v[7] = b.w;
  return f;
}
__device__ __forceinline__ Frag<float> widen(const Frag<u16>& a) {
  Frag<float> f;
#pragma unroll
  for (int j = 0; j < 8; ++j) f.v[j] = static_cast<float>(a.v[j]);
  return f;
}
__device__ __forceinline__ Frag<float> widen(const Frag<float>& a) { return a; }
__device__ __forceinline__ f32x4 mma(const Frag<u16>& a, const Frag<u16>& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma(const Frag<float>& a, const Frag<float>& b, f32x4 c) {
#pragma unroll
  for (int j = 0; j < 8; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[j], b.v[j], c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ f32x4 mma(const Frag<u16>& a, const Frag<float>& b, f32x4 c) { return mma(widen(a), b, c); }
__device__ __forceinline__ f32x4 mma(const Frag<float>& a, const Frag<u16>& b, f32x4 c) { return mma(a, widen(b), c); }

constexpr float kLog2e = 1.4426950408889634f;

// Keys of one tile of OP_ATTEND, and the LDS floats it needs for this cache row width (host and device).
__host__ __device__ constexpr int attend_keys(int element_bytes) { return element_bytes == 2 ? 64 : 32; }
__host__ __device__ constexpr int attend_floats(int row_elements, int element_bytes) {
  const int stride = (row_elements + 31) / 32 * 32 + 8, keys = attend_keys(element_bytes), slices = kWaves / (keys / 16);
  return (16 + keys) * stride * element_bytes / 4 + slices * keys * 16 + keys * 16 + 16 * (keys + 8) + 16;
}

// Part `start` of `count` of the visible keys, sixteen heads.  Scores: matrix tiles of 16 keys x 16 heads, the row's columns
// split over the waves of a tile; then the weights and the running sums of weight x value, of which an instruction keeps
// columns [128 extra, 128 extra + 128), sixteen a wave.
// Latent: heads [16 sub, 16 sub + 16), a row is [latent | rotated key], the latent is the value.  Attention: the heads of key
// head g = sub / b, sixteen of them from 16 (sub % b) on, b = ceil(heads per key head / 16); a row is g's [key | value], and
// the step's own row comes from the projections (one instruction per key head puts it into the cache).
template <class T, bool PLAIN>
__device__ __forceinline__ bool op_attend(const DecodeParams& p, Smem& s, const Op& o) {
  constexpr int kKeys = attend_keys(sizeof(T)), kTiles = kKeys / 16, kSlices = kWaves / kTiles, kPer = kKeys * 16 / kThreads, kSp = kKeys + 8;
  constexpr int kUnit = 16 / sizeof(T);
  LayerRef& l = layer_of(p, o.layer);
  const int heads16 = (l.heads + 15) & ~15;
  const uint32_t tag = tag_of(o.layer, 0);
  constexpr bool latent = !PLAIN;
  if (l.type != (latent ? QMK_MIXER_LATENT : QMK_MIXER_ATTENTION) || o.sub < 0 || o.start < 0 || o.count <= 0 || o.count > p.max_splits || o.start >= o.count || o.extra < 0)
    return bad_operand(p, o, o.start);
  const int group = latent ? l.heads : l.heads / l.kv_heads, blocks = (group + 15) / 16, kv = o.sub / blocks, block = o.sub % blocks;
  const int values = latent ? l.rank : l.v_dim, value_at = latent ? 0 : l.head_dim;      // columns of a row that are its value
  const int head0 = kv * group + block * 16, heads = min(16, group - block * 16);
  if (kv >= (latent ? 1 : l.kv_heads) || o.extra * 16 * kWaves >= values) return bad_operand(p, o, o.sub);
  const int tid = threadIdx.x, lane = tid & (kWaveSize - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWaveSize);
  const int width = latent ? l.rank + l.rot_dim : l.head_dim + l.v_dim, width32 = (width + 31) & ~31, stride = width32 + 8;
  const int pitch = latent ? width : l.kv_heads * width;      // elements between cache rows
  T* sq = reinterpret_cast<T*>(s.attend);
  T* sc = sq + 16 * stride;
  float* sred = reinterpret_cast<float*>(sc + kKeys * stride);   // [slice][key][16]
  float* ss = sred + kSlices * kKeys * 16;                        // [key][16]
  T* sp = reinterpret_cast<T*>(ss + kKeys * 16);                  // [16][kSp]
  float* sa = ss + kKeys * 16 + 16 * kSp;                         // [16]

  const int first = p.position + 1 > l.window ? p.position + 1 - l.window : 0, visible = p.position + 1 - first;
  const int per = ((visible + o.count - 1) / o.count + 31) & ~31;
  const int lo = first + o.start * per, hi = min(lo + per, p.position + 1);
  const int units = width32 / kUnit;
  const int rows = l.ring, offset = p.slot * rows;
  T* cache = static_cast<T*>(l.cache) + kv * width;
  // Rows base .. base + kKeys - 1 -> sc, but for the row another workgroup of this launch appends.  (A part is never
  // longer than the ring, so a position wraps at most once.)
  const uint32_t per_unit = 0xffffffffu / units + 1u;      // exact: units of a tile times units of a row stay far below 2^32
  auto load_tile = [&](int base) {
    constexpr int kBatch = 9;      // 64 rows of 576 bf16: all requests at once
    const int at0 = base % rows, count = kKeys * units;
#pragma unroll 1
    for (int first = tid; first < count; first += kBatch * kThreads) {
      v4u v[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const int id = first + j * kThreads, r = __umulhi(id, per_unit), c = id - r * units, at = at0 + r >= rows ? at0 + r - rows : at0 + r;
        v[j] = v4u{0u, 0u, 0u, 0u};
        if (id < count && base + r < hi && base + r != p.position && c * kUnit < width)
          v[j] = *reinterpret_cast<const v4u*>(cache + static_cast<size_t>(offset + at) * pitch + c * kUnit);
      }
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const int id = first + j * kThreads, r = __umulhi(id, per_unit), c = id - r * units;
        if (id < count) *reinterpret_cast<v4u*>(sc + r * stride + c * kUnit) = v[j];
      }
    }
  };
  // The appended row, where this part holds it (it is then the part's last).
  auto load_appended = [&](int base) {
    if (p.position >= hi || p.position < base || p.position >= base + kKeys) return;
    if (!latent) {   // neighbouring elements, both of the key or both of the value
      const uint64_t* from = p.proj + l.proj_at + l.heads * l.q_stride;
      const bool put = block == 0 && o.extra == 0;
      T* row = cache + static_cast<size_t>(offset + p.position % rows) * pitch;
#pragma unroll 1
      for (int c = tid * 2; c < width; c += kThreads * 2) {
        const uint64_t* pair = from + (c < l.head_dim ? kv * l.head_dim + c : l.kv_heads * l.head_dim + kv * l.v_dim + c - l.head_dim);
        Units<2> v;
        v.ask(pair, 0, 1, 2);
        v.wait(p, s, o, pair, 0, 1, 2, tag);
        T* at = sc + (p.position - base) * stride + c;
        at[0] = from_f32<T>(v[0]);
        at[1] = from_f32<T>(v[1]);
        if (put) {
          row[c] = at[0];
          row[c + 1] = at[1];
        }
      }
      return;
    }
    // Normed latent, rotated key part: every workgroup that needs the row makes it, which takes no longer than to fetch it.
    const uint64_t* from = p.proj + l.heads * (l.q_stride + l.v_dim);
    T *to = sc + (p.position - base) * stride, *row = cache + static_cast<size_t>(offset + p.position % rows) * pitch;
    const bool put = o.sub == 0 && o.extra == 0;
    static_assert(kMaxRank <= kThreads, "one latent element per thread");
    const float v = unit_of(p, s, o, from + min(tid, l.rank - 1), tag);
    const float inv = 1.f / sqrtf(block_sum(tid < l.rank ? v * v : 0.f, s.scratch) / l.rank_true + p.eps);
    auto leave = [&](int i, float e) {
      to[i] = from_f32<T>(e);
      if (put) row[i] = to[i];
    };
    if (tid < l.rank) leave(tid, v * inv * l.vec0[tid]);
#pragma unroll 1
    for (int i = tid; i < l.rot_dim; i += kThreads) leave(l.rank + i, unit_of(p, s, o, from + l.rank + i, tag));
  };
  // Queries of the sixteen heads: units of the absorbed ones (in bf16 mode pairs) and of the projections, as they lie side by side, dealt to the threads; the first
  // look ahead of the keys.
  constexpr int kPair = latent && sizeof(T) == 2 ? 2 : 1, kQueries = 8;
  const int per_a = latent ? l.rank / kPair : 0, per_b = latent ? l.rot_dim : l.q_stride, count_a = heads * per_a, count_b = heads * per_b;
  const uint32_t inverse_a = 0xffffffffu / max(per_a, 1) + 1u, inverse_b = 0xffffffffu / per_b + 1u;
  Gather<latent ? kQueries : 1> queries;
  Gather<latent ? 2 : kQueries> rest;
  int asked = 0;
  auto ask_queries = [&](int base) {
    asked = base;
#pragma unroll
    for (int j = 0; j < (latent ? kQueries : 1); ++j) queries.at[j] = latent ? p.absorbed + head0 * per_a + min(base + tid + j * kThreads, count_a - 1) : p.proj + l.proj_at + head0 * per_b;
#pragma unroll
    for (int j = 0; j < (latent ? 2 : kQueries); ++j) {
      const int id = min((latent ? base / (kQueries / 2) : base) + tid + j * kThreads, count_b - 1), h = __umulhi(id, inverse_b), c = id - h * per_b;
      rest.at[j] = latent ? p.proj + (head0 + h) * l.q_stride + l.head_dim + c : p.proj + l.proj_at + head0 * l.q_stride + id;
    }
    queries.ask();
    rest.ask();
  };
  auto put_queries = [&] {
    if constexpr (latent) {
#pragma unroll
      for (int j = 0; j < kQueries; ++j) {
        const int id = asked + tid + j * kThreads, h = __umulhi(id, inverse_a), c = id - h * per_a;
        if (id >= count_a) continue;
        if constexpr (kPair == 2) reinterpret_cast<uint32_t*>(sq + h * stride)[c] = static_cast<uint32_t>(queries.r[j]);
        else sq[h * stride + c] = from_f32<T>(queries[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < (latent ? 2 : kQueries); ++j) {
      const int id = (latent ? asked / (kQueries / 2) : asked) + tid + j * kThreads, h = __umulhi(id, inverse_b), c = id - h * per_b;
      if (id < count_b) sq[h * stride + (latent ? l.rank : 0) + c] = from_f32<T>(rest[j]);
    }
  };
  if (lo < hi) {
    ask_queries(0);
    // Heads and columns that are not there.
    const int end = latent ? width : l.q_stride;
#pragma unroll 1
    for (int h = wave; h < 16; h += kWaves)
      for (int c = (h < heads ? end : 0) + lane; c < (latent ? width32 : end); c += kWaveSize) sq[h * stride + c] = from_f32<T>(0.f);
    load_tile(lo);
    __syncthreads();     // the tile's row that load_appended fills has been zeroed
    load_appended(lo);
  }
  stamp(p, s, 0);
  if constexpr (latent) plan_next<PLAIN>(p, s, o);
  if (lo < hi) {
    queries.wait(p, s, o, tag);
    rest.wait(p, s, o, tag);
    put_queries();
#pragma unroll 1
    for (int base = kQueries * kThreads; base < max(count_a, count_b * (latent ? kQueries / 2 : 1)); base += kQueries * kThreads) {
      ask_queries(base);
      queries.wait(p, s, o, tag);
      rest.wait(p, s, o, tag);
      put_queries();
    }
  } else {      // No keys.  What it leaves all the same takes the place of parts that the attention before may still be merging: every query comes behind that.
    unit_of(p, s, o, latent ? p.absorbed + head0 * per_a : p.proj + l.proj_at + head0 * per_b, tag);
  }
  if (p.timeline != nullptr && tid == 0) s.t_wait = wall_clock64();

  stamp(p, s, 1);
  const int head = tid & 15, key0 = tid >> 4;      // this thread's scores: keys key0, key0 + 32, ...
  float m = -INFINITY, lsum = 0.f;
  f32x4 acc = {};
  const int column0 = (o.extra * kWaves + wave) * 16;      // this wave's sixteen columns of the latent
  const bool columns = column0 < values;
#pragma unroll 1
  for (int base = lo; base < hi; base += kKeys) {
    if (base != lo) {
      load_tile(base);
      __syncthreads();
      load_appended(base);
    }
    __syncthreads();
    {
      const int tile = wave % kTiles, slice = wave / kTiles, steps = (latent ? width32 : l.q_stride) / 32;
      f32x4 d = {};
      for (int k = slice; k < steps; k += kSlices)
        d = mma(load_frag(sc + (tile * 16 + (lane & 15)) * stride + k * 32 + (lane >> 4) * 8),
                load_frag(sq + (lane & 15) * stride + k * 32 + (lane >> 4) * 8), d);
#pragma unroll
      for (int i = 0; i < 4; ++i) sred[(slice * kKeys + tile * 16 + (lane >> 4) * 4 + i) * 16 + (lane & 15)] = d[i];
    }
    __syncthreads();
    float score[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int key = key0 + 32 * j;
      score[j] = -INFINITY;
      if (base + key < hi) {
        float t = 0.f;
#pragma unroll
        for (int q = 0; q < kSlices; ++q) t += sred[(q * kKeys + key) * 16 + head];
        score[j] = t * (l.scale * kLog2e);
      }
    }
    float top = score[0];
#pragma unroll
    for (int j = 1; j < kPer; ++j) top = fmaxf(top, score[j]);
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    if (lane < 16) ss[wave * 16 + head] = top;
    __syncthreads();
    top = m;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) top = fmaxf(top, ss[k * 16 + head]);
    const float shrink = exp2_fast(m - top);
    lsum *= shrink;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const float w = exp2_fast(score[j] - top);
      lsum += w;
      sp[head * kSp + key0 + 32 * j] = from_f32<T>(w);
    }
    m = top;
    if (key0 == 0) sa[head] = shrink;
    __syncthreads();
    if (columns) {
      acc *= sa[lane & 15];
#pragma unroll
      for (int kk = 0; kk < kKeys / 32; ++kk) {
        Frag<T> cf;
#pragma unroll
        for (int j = 0; j < 8; ++j) cf.set(j, sc[(kk * 32 + (lane >> 4) * 8 + j) * stride + value_at + column0 + (lane & 15)]);
        acc = mma(cf, load_frag(sp + (lane & 15) * kSp + kk * 32 + (lane >> 4) * 8), acc);
      }
    }
    __syncthreads();
  }
  stamp(p, s, 2);
  // Every thread of a head has the same maximum; the sums of its key columns are added up here.
  lsum += __shfl_xor(lsum, 16);
  lsum += __shfl_xor(lsum, 32);
  if (lane < 16) ss[wave * 16 + head] = lsum;
  __syncthreads();
  float* ml = p.ml + (static_cast<size_t>(o.start) * heads16 + head0) * 2;
  if (key0 == 0 && o.extra == 0 && (latent || head < heads)) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) t += ss[k * 16 + head];
    st_shared_f32(ml + head * 2, m);
    st_shared_f32(ml + head * 2 + 1, t);
  }
  if (columns && (latent || (lane & 15) < heads)) {
    uint64_t* at = reinterpret_cast<uint64_t*>(p.part + (static_cast<size_t>(o.start) * heads16 + head0 + (lane & 15)) * values + column0 + (lane >> 4) * 4);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __hip_atomic_store(at + i, (static_cast<uint64_t>(__float_as_uint(acc[2 * i + 1])) << 32) | __float_as_uint(acc[2 * i]), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  stamp(p, s, 3);
  release_stores();
  __syncthreads();
  if (s.ctl[0] == 0) return false;
  arrive_stage(p, o);
  return true;
}

// The parts of one head put together, times its output gate.
__device__ __forceinline__ bool op_attend_merge(const DecodeParams& p, Smem& s, const Op& o) {
  LayerRef& l = layer_of(p, o.layer);
  if (l.type != QMK_MIXER_ATTENTION || o.sub < 0 || o.sub >= l.heads || o.count <= 0 || o.count > p.max_splits || o.count > kMaxParts)
    return bad_operand(p, o, o.sub);
  const int tid = threadIdx.x, heads16 = (l.heads + 15) & ~15, parts = o.count, n = l.v_dim, groups = kThreads / n, e = tid % n, group = tid / n;
  if (!wait_stage(p, s, o)) return false;
  if (tid < parts) {
    const uint64_t ml = ld_shared64(p.ml + (static_cast<size_t>(tid) * heads16 + o.sub) * 2);
    s.aux[tid] = __uint_as_float(static_cast<uint32_t>(ml));
    s.aux[kMaxParts + tid] = __uint_as_float(static_cast<uint32_t>(ml >> 32));
  }
  constexpr int kBatch = 8;
  float v[kBatch];
  const float* column = p.part + static_cast<size_t>(o.sub) * n + e;
  auto request = [&](int base) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j) v[j] = ld_shared_f32(column + static_cast<size_t>(min(base + j * groups, parts - 1)) * heads16 * n);
  };
  request(group);
  const float gate = unit_of(p, s, o, p.proj + l.proj_at + l.heads * l.q_stride + l.kv_heads * (l.head_dim + n) + o.sub * n + min(tid, n - 1), tag_of(o.layer, 0));
  __syncthreads();
  if (tid < kWaveSize) {   // weights of the parts
    const float mx = tid < parts ? s.aux[tid] : -INFINITY, top = wave_max(mx);
    const float w = exp2_fast(mx - top), sum = wave_sum(tid < parts ? w * s.aux[kMaxParts + tid] : 0.f);
    s.aux[tid] = tid < parts ? w / sum : 0.f;
  }
  __syncthreads();
  float acc = 0.f;
  if (group < groups) {
#pragma unroll 1
    for (int base = group; base < parts; base += kBatch * groups) {
      if (base != group) request(base);
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        if (base + j * groups < parts) acc = fmaf(s.aux[base + j * groups], v[j], acc);
    }
    s.xs[group * n + e] = acc;
  }
  __syncthreads();
  if (tid < n) {
    acc = 0.f;
#pragma unroll 4
    for (int i = 0; i < groups; ++i) acc += s.xs[i * n + tid];
    put_unit(p.mix + l.mix_at + o.sub * n + tid, acc * gate, tag_of(o.layer, 0));
  }
  return s.ctl[0] != 0;
}

}  // namespace hybrid
}  // namespace qmk
