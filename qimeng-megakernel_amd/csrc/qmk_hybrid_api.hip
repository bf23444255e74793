// The hybrid route's kernels for gfx950 and their C ABI (include/qmk_hybrid.h).
//
// Decode: the persistent interpreter of the other routes (one workgroup per instruction queue, tagged units and, for attention parts, counters with
// bounded waits, the last workgroup to retire clears them) over the ops of qmk_hybrid_ops.h.  Prefill: the launches of
// qmk_hybrid_prefill.h, qmk_hybrid_plain.h and qmk_hybrid_chunks.h, layer by layer, on the caller's stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "qmk_hybrid_ops.h"
#include "qmk_hybrid_prefill.h"
#include "qmk_hybrid_plain.h"
#include "qmk_hybrid_chunks.h"

namespace qmk {
namespace hybrid {

constexpr int kStatusWords = 8;
constexpr int kMaxDevices = 16;
constexpr int kMaxQueues = 1024;
__device__ int32_t g_status[kStatusWords];

// The launch's parameters as one instruction sees them: read from the kernel-argument segment through a pointer the
// compiler cannot look behind, so that an op loads what it needs of them and keeps nothing across the instruction loop
// (held in scalar registers for the whole kernel they are parked in vector lanes, one move per use).
static_assert(std::is_trivially_copyable<DecodeParams>::value && std::is_standard_layout<DecodeParams>::value, "copied byte for byte into the segment");
__device__ __forceinline__ const DecodeParams& params_of_this_instruction() {
  auto args = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return *(const DecodeParams*)args;   // the only kernel argument: offset 0 of the segment
}

template <class T, bool PLAIN>
__global__ __launch_bounds__(kThreads, 1) void decode_megakernel_hybrid(const DecodeParams p_launch) {
  const DecodeParams& p_loop = p_launch;
  __shared__ __align__(16) Smem s;
  if (threadIdx.x == 0) {
    s.best_val = -INFINITY;
    s.best_idx = 0x7fffffff;
    s.ctl[0] = 1;
    s.ctl[2] = 0;
    s.ctl[3] = OP_NOOP;
  }
  const int num_insts = p_loop.num_insts;
  const int32_t* queue = p_loop.instructions + static_cast<size_t>(blockIdx.x) * num_insts * kInstWords;
  bool ok = true;
  // The words of instruction i + 2 are asked for while instruction i runs.
  int32_t word = (threadIdx.x < kInstWords && num_insts > 0) ? queue[threadIdx.x] : 0;
  int32_t word1 = (threadIdx.x < kInstWords && num_insts > 1) ? queue[kInstWords + threadIdx.x] : 0;
  if (threadIdx.x < kInstWords) s.inst[0][threadIdx.x] = word;
  __syncthreads();
  if (uniform(threadIdx.x) < kWaveSize) plan_of<PLAIN>(p_loop, s, 0);
  for (int i = 0; i < num_insts && ok; ++i) {
    if (threadIdx.x < kInstWords) {
      s.inst[(i + 1) & 1][threadIdx.x] = word1;
      word1 = (i + 2 < num_insts) ? queue[(i + 2) * kInstWords + threadIdx.x] : 0;
    }
    __syncthreads();
    const DecodeParams& p = params_of_this_instruction();
    auto operand = [&](int w) { return static_cast<int>(uniform(s.inst[i & 1][w])); };
    const Op o{i, operand(0), operand(1), operand(2), operand(3), operand(4), operand(5), operand(6), operand(7), operand(8)};
    unsigned long long t_start = 0;
    if (p.timeline != nullptr && threadIdx.x == 0) t_start = s.t_wait = wall_clock64();
    if (o.opcode != OP_NOOP && (o.layer < 0 || o.layer >= p.num_layers || o.wait_stage >= 4 * p.groups || o.arrive_stage >= 4 * p.groups)) {
      ok = bad_operand(p, o, o.layer);
    } else {
      switch (o.opcode) {
        case OP_NOOP:
          if constexpr (!PLAIN) plan_next<PLAIN>(p, s, o);
          break;
        case OP_IN_PROJECT:
        case OP_LRU_STEP:
        case OP_LATENT_ABSORB:
        case OP_LATENT_VALUE:
        case OP_WKV_STEP:
        case OP_OUT_PROJECT:
        case OP_UP_GATE:
        case OP_LM_HEAD:
        case OP_STATE_STEP:
        case OP_JOIN:
        case OP_GATE: ok = op_rows<T, PLAIN>(p, s, o); break;
        case OP_ATTEND: ok = op_attend<T, PLAIN>(p, s, o); break;
        case OP_ATTEND_MERGE:
          if constexpr (PLAIN) ok = op_attend_merge(p, s, o);
          else ok = bad_operand(p, o, o.opcode);
          break;
        default:
          if (threadIdx.x == 0) report_error(counters_of(p), QMK_DEV_BAD_OPCODE, i, o.opcode, 0);
          ok = false;
          break;
      }
    }
    if constexpr (PLAIN) plan_next<PLAIN>(p, s, o);
    if (p.timeline != nullptr && threadIdx.x == 0) {
      uint64_t* rec = p.timeline + (static_cast<size_t>(blockIdx.x) * p.num_insts + i) * 8;
      rec[0] = t_start;
      rec[1] = s.t_wait;
      rec[2] = wall_clock64();
      rec[3] = static_cast<uint64_t>(o.opcode) | (static_cast<uint64_t>(static_cast<uint32_t>(o.layer)) << 8);
      for (int k = 0; k < 4; ++k) rec[4 + k] = s.stamps[k];
    }
    __syncthreads();
    if (threadIdx.x == 0 && o.opcode != OP_NOOP) s.ctl[3] = o.opcode;      // (read behind the next instruction's barriers)
  }
  const DecodeParams& p = params_of_this_instruction();

  // Retire, also behind an error: the last workgroup to arrive owns the counters and units alone, clears them (its and the others' shares have been, behind
  // the last norm's input) and picks the token among the workgroups' candidates (largest logit, smallest row among equals).
  const bool sampling = p.token_out != nullptr;
  if (sampling && threadIdx.x == 0) {
    const uint32_t bits = __float_as_uint(s.best_val);
    const uint32_t key = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
    __hip_atomic_store(p.candidates + blockIdx.x, (static_cast<uint64_t>(key) << 32) | (0xffffffffu - static_cast<uint32_t>(s.best_idx)),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  release_stores();
  __syncthreads();
  int32_t* done = counter_ptr(counters_of(p), 0, kStageGroupRows - 1, kStageGroupSlots - 1);
  if (threadIdx.x == 0) {      // upper half: workgroups that have cleared nothing
    const int mine = s.ctl[2] ? 1 : 0x10001, all = __hip_atomic_fetch_add(done, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine;
    s.ctl[1] = (all & 0xffff) == static_cast<int>(gridDim.x);
    s.ctl[2] = all >> 16 == 0;
  }
  __syncthreads();
  if (!s.ctl[1]) return;
  const int copy = PLAIN ? layer_of(p, p.num_layers - 1).x_from : -1;
  if (!s.ctl[2]) clear_units(p.units, p.all_units, threadIdx.x, kThreads);
  else if (copy >= 0) clear_units(copy_of(p, copy), (2 + QMK_HYBRID_MAX_BRANCHES) * p.width, threadIdx.x, kThreads);
  else clear_units(p.units + p.early_units, p.all_units - p.early_units, threadIdx.x, kThreads);
  const int total = p.groups * kStageGroupRows * kStageGroupSlots;
  for (int i = threadIdx.x; i < total; i += kThreads) __hip_atomic_store(p.barriers + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!sampling || threadIdx.x >= kWaveSize) return;
  uint64_t best = 0;
  for (int q = threadIdx.x; q < static_cast<int>(gridDim.x); q += kWaveSize) {
    const uint64_t c = ld_shared64(p.candidates + q);
    best = c > best ? c : best;
  }
  for (int off = 1; off < kWaveSize; off <<= 1) {
    const uint32_t lo = __shfl_xor(static_cast<uint32_t>(best), off), hi = __shfl_xor(static_cast<uint32_t>(best >> 32), off);
    const uint64_t other = (static_cast<uint64_t>(hi) << 32) | lo;
    best = other > best ? other : best;
  }
  const uint32_t token = 0xffffffffu - static_cast<uint32_t>(best);
  if (threadIdx.x == 0 && token < static_cast<uint32_t>(p.vocab)) *p.token_out = token;
}

struct DeviceInfo {
  bool ready = false;
  int max_queues = 0;
  int32_t* status = nullptr;
};
DeviceInfo g_devices[kMaxDevices];
std::mutex g_mutex;

int device_info(DeviceInfo** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return QMK_ERR_NO_DEVICE;
  std::lock_guard<std::mutex> lock(g_mutex);
  DeviceInfo& d = g_devices[dev];
  if (!d.ready) {
    hipDeviceProp_t prop;
    int blocks = kMaxQueues;
    auto fits = [&](auto kernel) {
      int n = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kThreads, 0) != hipSuccess) return false;
      blocks = std::min(blocks, n);
      return true;
    };
    void* sym = nullptr;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess || !fits(decode_megakernel_hybrid<u16, false>) || !fits(decode_megakernel_hybrid<float, false>) ||
        !fits(decode_megakernel_hybrid<u16, true>) || !fits(decode_megakernel_hybrid<float, true>) || hipGetSymbolAddress(&sym, HIP_SYMBOL(g_status)) != hipSuccess || hipMemset(sym, 0, sizeof(int32_t) * kStatusWords) != hipSuccess)
      return QMK_ERR_NO_DEVICE;
    d.max_queues = std::min(blocks * prop.multiProcessorCount, kMaxQueues);
    d.status = static_cast<int32_t*>(sym);
    d.ready = true;
  }
  *out = &d;
  return QMK_OK;
}

inline size_t align_up(size_t n) { return (n + 255) & ~size_t(255); }
inline bool m16(int v) { return v > 0 && v % 16 == 0; }
inline int element(const QmkHybridArgs* a) { return a->dtype == QMK_HYBRID_F32 ? 4 : 2; }

// Entries of a plain residual: where they read x, and how a run's branches stand in the table.
bool plain_ok(const QmkHybridArgs* a, int i) {
  const QmkHybridLayer& l = a->layers[i];
  const bool run = l.type >= QMK_MIXER_GLA && l.type <= QMK_MIXER_DELTA;
  if (!run && l.type != QMK_ENTRY_JOIN && l.type != QMK_ENTRY_FINAL) return false;
  if ((i + 1 == a->num_layers) != (l.type == QMK_ENTRY_FINAL)) return false;
  if (l.branch < 0 || l.branches < 1 || l.branches > QMK_HYBRID_MAX_BRANCHES || l.branch >= l.branches || (!run && l.branches != 1)) return false;
  if (i - l.branch < 0 || i - l.branch + l.branches > a->num_layers) return false;
  for (int b = 0; b < l.branches; ++b) {
    const QmkHybridLayer& other = a->layers[i - l.branch + b];
    if (other.branch != b || other.branches != l.branches || (b > 0 && other.has_mlp)) return false;
  }
  if (l.x_from < -1 || l.x_from > 1 || l.x_to < 0 || l.x_to > 1 || l.x_from == l.x_to) return false;
  if (l.prev < -1 || l.prev >= i || (l.prev >= 0 && (a->layers[l.prev].branch != 0 || a->layers[l.prev].type > QMK_MIXER_DELTA || l.x_from < 0))) return false;
  return l.norm >= QMK_NORM_RMS && l.norm <= QMK_NORM_LAYER && l.proj_at >= 0 && l.proj_at % 16 == 0 && l.mix_at >= 0 && l.mix_at % 16 == 0 && l.ff_at >= 0 &&
         l.ff_at % 16 == 0;
}

bool layer_ok(const QmkHybridArgs* a, int i) {
  const QmkHybridLayer& l = a->layers[i];
  if (a->streams == 0 ? !plain_ok(a, i) : l.type > QMK_MIXER_WKV) return false;
  if (l.type == QMK_ENTRY_JOIN) return 2 * a->width <= kMaxK;
  if (l.type == QMK_ENTRY_FINAL) return true;
  if (!m16(l.in_rows) || !m16(l.mix_width) || l.mix_width > kMaxK) return false;
  if (l.has_mlp && (!m16(l.ff) || l.ff > kMaxK)) return false;
  switch (l.type) {
    case QMK_MIXER_RGLRU:
      return l.taps >= 1 && l.taps <= kMaxTaps && l.blocks > 0 && m16(l.block_dim) && l.blocks * l.block_dim == l.mix_width && l.in_rows == 2 * l.mix_width;
    case QMK_MIXER_LATENT:
      return l.heads > 0 && m16(l.head_dim) && m16(l.rot_dim) && l.rot_true > 0 && l.rot_true % 2 == 0 && l.rot_true <= l.rot_dim && m16(l.v_dim) &&
             l.v_dim <= 256 && m16(l.rank) && l.rank <= kMaxRank && l.rank_true > 0 && l.rank_true <= l.rank && l.q_stride % 32 == 0 &&
             l.q_stride >= l.head_dim + l.rot_dim && l.q_stride <= 256 && l.window > 0 && l.ring > 0 && l.mix_width == l.heads * l.v_dim &&
             l.in_rows == l.heads * (l.q_stride + l.v_dim) + l.rank + l.rot_dim &&
             attend_floats(l.rank + l.rot_dim, element(a)) <= kAttendFloats;
    case QMK_MIXER_WKV:
      return l.heads > 0 && m16(l.head_dim) && l.head_dim <= kMaxHeadDim && l.head_dim_true > 0 && l.head_dim_true <= l.head_dim && m16(l.rank) &&
             l.rank <= kMaxK && l.mix_width == l.heads * l.head_dim && l.in_rows == 4 * l.mix_width + l.rank;
    case QMK_MIXER_ATTENTION:
      return l.heads > 0 && l.kv_heads > 0 && l.heads % l.kv_heads == 0 && m16(l.head_dim) && m16(l.v_dim) && l.v_dim <= 256 && l.rot_dim == 0 &&
             l.rot_true >= 0 && l.rot_true % 2 == 0 && l.rot_true <= l.head_dim && l.q_stride == (l.head_dim + 31) / 32 * 32 && l.q_stride <= 256 &&
             l.window > 0 && l.ring > 0 && l.mix_width == l.heads * l.v_dim &&
             l.in_rows == l.heads * (l.q_stride + l.v_dim) + l.kv_heads * (l.head_dim + l.v_dim) &&
             attend_floats(l.head_dim + l.v_dim, element(a)) <= kAttendFloats;
    case QMK_MIXER_GLA:
    case QMK_MIXER_DELTA: {
      const bool delta = l.type == QMK_MIXER_DELTA;
      if (l.heads < 1 || l.kv_heads < 1 || l.heads % l.kv_heads != 0 || !m16(l.head_dim) || l.head_dim > kMaxHeadDim || !m16(l.v_dim) || l.v_dim > kMaxHeadDim ||
          l.v_true < 1 || l.v_true > l.v_dim || !m16(l.rank) || l.mix_width != l.heads * l.v_dim)
        return false;
      if (!delta) return l.kv_heads == l.heads && l.gate_rank == 0 && l.rank <= kMaxK && l.in_rows == 2 * l.heads * (l.head_dim + l.v_dim) + l.rank;
      return m16(l.gate_rank) && l.rank + l.gate_rank <= kMaxK && l.taps >= 1 && l.taps <= kMaxTaps &&
             l.in_rows == conv_channels(l) + l.rank + l.gate_rank + (l.heads + 15) / 16 * 16;
    }
    default: return false;
  }
}

int check_shape(const QmkHybridArgs* a) {
  if (a == nullptr || a->layers == nullptr) return QMK_ERR_NULL_ARG;
  if (a->struct_size != sizeof(QmkHybridArgs)) return QMK_ERR_ABI;
  if (a->dtype > QMK_HYBRID_F32) return QMK_ERR_MODEL;
  if (a->num_layers < 1 || !m16(a->width) || a->width > kMaxK || a->width_true < 1 || a->width_true > a->width || a->streams < 0 ||
      a->streams > kMaxStreams || a->vocab < 1 || !m16(a->vocab_rows) || a->vocab > a->vocab_rows || !(a->eps >= 0.f) ||
      !(a->logit_softcap >= 0.f))
    return QMK_ERR_SHAPE;
  for (int i = 0; i < a->num_layers; ++i)
    if (!layer_ok(a, i)) return QMK_ERR_SHAPE;
  return QMK_OK;
}

bool layer_pointers(const QmkHybridLayer& l) {
  if (l.type == QMK_ENTRY_JOIN) return l.in_w != nullptr;
  if (l.type == QMK_ENTRY_FINAL) return l.norm1 != nullptr;
  if (l.type >= QMK_MIXER_GLA) {
    bool ok = l.in_w && l.o_w && (l.branch > 0 || l.norm1) && (!l.has_mlp || (l.mlp_w && l.down_w)) && (l.branches > 1) == (l.out_norm != nullptr);
    if (l.type == QMK_MIXER_ATTENTION) return ok && l.cache && ((l.rope_cos && l.rope_sin) || l.rot_true == 0);
    ok = ok && l.mid_w && l.mid_b && l.vec0 && l.state;
    return ok && (l.type == QMK_MIXER_GLA || (l.gate_w && l.vec1 && l.vec2 && (l.shift || l.taps == 1)));
  }
  bool ok = l.norm1 && l.in_w && l.mid_w && l.vec0;
  if (l.type == QMK_MIXER_LATENT) ok = ok && l.uk_w && l.uv_w && l.rope_cos && l.rope_sin && l.cache;
  else ok = ok && l.mid_b && l.vec1 && l.vec2 && l.state && (l.shift || (l.type == QMK_MIXER_RGLRU && l.taps == 1));
  if (l.type == QMK_MIXER_RGLRU) ok = ok && l.in_b;
  if (l.has_mlp) ok = ok && l.norm2 && l.mlp_w && l.down_w && l.next2;
  return ok && l.o_w && l.hc && l.next1;
}

int check_launch(const QmkHybridArgs* a, int tokens) {
  if (int rc = check_shape(a); rc != QMK_OK) return rc;
  if (!a->layers_device || !a->embed || !a->final_norm || !a->head || !a->token_in || !a->workspace) return QMK_ERR_NULL_ARG;
  for (int i = 0; i < a->num_layers; ++i)
    if (!layer_pointers(a->layers[i])) return QMK_ERR_NULL_ARG;
  if (a->slots < 1 || a->slot < 0 || a->slot >= a->slots || (a->flip != 0 && a->flip != 1)) return QMK_ERR_SHAPE;
  if (tokens < 1 || a->position < 0 || a->position > a->max_positions - tokens) return QMK_ERR_POSITION;
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    // every key a query of the launch sees must still have its row when the launch's rows have been written
    if ((l.type == QMK_MIXER_LATENT || l.type == QMK_MIXER_ATTENTION) && l.ring < std::min(a->position + tokens, l.window - 1 + tokens)) return QMK_ERR_SHAPE;
  }
  if (reinterpret_cast<uintptr_t>(a->workspace) % 256 != 0) return QMK_ERR_SHAPE;
  return QMK_OK;
}

struct Carver {
  char* base;
  size_t used = 0;
  template <class T>
  T* take(size_t n) {
    T* t = base == nullptr ? nullptr : reinterpret_cast<T*>(base + used);
    used += align_up(n * sizeof(T));
    return t;
  }
};

struct DecodeBuffers {
  uint64_t *candidates, *units, *proj, *mix, *absorbed, *u, *sums;
  float *x, *part, *ml;
  int early_units, all_units;
};
size_t decode_buffers(const QmkHybridArgs* a, void* base, DecodeBuffers* b) {
  size_t proj = 0, mix = 0, absorbed = 0, part = 0, ml = 0;
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    if (l.type > QMK_MIXER_DELTA) continue;
    proj = std::max<size_t>(proj, static_cast<size_t>(l.proj_at) + l.in_rows + (l.type == QMK_MIXER_DELTA ? l.mix_width : 0));
    mix = std::max<size_t>(mix, std::max(static_cast<size_t>(l.mix_at) + l.mix_width, l.has_mlp ? static_cast<size_t>(l.ff_at) + l.ff : 0));
    if (l.type == QMK_MIXER_ATTENTION) {
      const size_t heads16 = (l.heads + 15) & ~15;
      part = std::max(part, a->max_splits * heads16 * l.v_dim);
      ml = std::max(ml, a->max_splits * heads16 * 2);
    }
    if (l.type == QMK_MIXER_LATENT) {
      const size_t heads16 = (l.heads + 15) & ~15;
      absorbed = std::max<size_t>(absorbed, static_cast<size_t>(l.heads) * l.rank);
      part = std::max(part, a->max_splits * heads16 * l.rank);
      ml = std::max(ml, a->max_splits * heads16 * 2);
    }
  }
  Carver c{static_cast<char*>(base)};
  b->candidates = c.take<uint64_t>(kMaxQueues);
  const size_t units = c.used;
  b->proj = c.take<uint64_t>(proj);
  b->mix = c.take<uint64_t>(mix);
  b->absorbed = c.take<uint64_t>(absorbed);
  b->early_units = static_cast<int>((c.used - units) / sizeof(uint64_t));
  b->u = c.take<uint64_t>(a->streams > 0 ? a->width : 0);
  b->sums = c.take<uint64_t>(a->streams > 0 ? 0 : static_cast<size_t>(2 * (2 + QMK_HYBRID_MAX_BRANCHES)) * a->width);
  b->all_units = static_cast<int>((c.used - units) / sizeof(uint64_t));
  b->units = b->proj;
  b->x = c.take<float>(static_cast<size_t>(a->streams) * a->width);
  b->part = c.take<float>(part);
  b->ml = c.take<float>(ml);
  return c.used;
}

inline size_t values_cap(const QmkHybridArgs* a) { return (static_cast<size_t>(a->max_positions) + 31) & ~size_t(31); }

// Parts of products that are cut along K (fp32 mode).  The tickets are zero at a portion's start (begin_portion) and after every product.
struct SplitBuffers {
  int32_t* tickets;
  f32x4* partial;
};
inline SplitBuffers split_buffers(Carver& c) {
  SplitBuffers b;
  b.tickets = c.take<int32_t>(kMaxTickets);
  b.partial = c.take<f32x4>(kPartialUnits);
  return b;
}

// Rows that products read: `count` elements, in fp32 mode whole or as three bf16 parts.  They are in parts where the kernels that
// stage tiles straight to LDS take their product: a multiple of 64 columns, and more than 64 (shorter products keep the fp32
// instruction).  us, split by the workgroups that read them -> by the kernel that makes them: 200 x 2048 x 2048 and x 6144 with the
// residual's streams 45 -> 36 on the average, 200 x 5696 x 2048 41 -> 33, five of 200 x 2048 x 2048 60 -> 36, 200 x 12288 x 2048 63 -> 63,
// 1 x 151936 x 2048 429 -> 147; the kernels that make them take as long as before.
template <class T>
struct OperandRows {
  T* at = nullptr;
  size_t count = 0;
  OperandRows() = default;
  OperandRows(Carver& c, size_t n) : at(c.take<T>(sizeof(T) == 4 ? n / 2 * 3 : n)), count(n) {}
  Operand<T> of(int columns) const { return Operand<T>{at, sizeof(T) == 4 && columns > 64 && columns % 64 == 0 ? count : 0}; }
};

// What the recurrences of portions keep between their launches: as large as the largest of its layers needs.
struct ChunkBuffers {
  float *chunks = nullptr, *starts = nullptr, *fades = nullptr;
  size_t chunk_count = 0, start_count = 0, fade_count = 0;
  void fit(size_t tokens, size_t heads, size_t dim, size_t n, bool segments) {
    chunk_count = std::max(chunk_count, chunks_of(static_cast<int>(tokens)) * heads * chunk_floats(static_cast<int>(dim)));
    if (!segments) return;
    const size_t most = segments_of(static_cast<int>(tokens), kSegmentChunks);
    start_count = std::max(start_count, most * heads * dim * n);
    fade_count = std::max(fade_count, most * heads * dim);
  }
  void take(Carver& c) {
    chunks = c.take<float>(chunk_count);
    starts = c.take<float>(start_count);
    fades = c.take<float>(fade_count);
  }
};

template <class T>
struct PlainBuffers {
  SplitBuffers split;
  float *x, *branch, *qkv, *values, *decay, *beta, *o;
  ChunkBuffers state;
  T *q, *low, *gate, *vt;
  OperandRows<T> h, mix;
};
template <class T>
size_t plain_buffers(const QmkHybridArgs* a, void* base, PlainBuffers<T>* b) {
  const size_t P = a->portion_rows, D = a->width;
  ChunkBuffers state;
  size_t h = P * D, branch = 0, qkv = 0, values = 0, decay = 0, beta = 0, o = 0, q = 0, low = 0, gate = 0, mix = 0, vt = 0;
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    if (l.type == QMK_ENTRY_JOIN) h = std::max(h, 2 * P * D);
    if (l.type > QMK_MIXER_DELTA) continue;
    mix = std::max(mix, P * std::max<size_t>(l.mix_width, l.has_mlp ? l.ff : 0));
    gate = std::max(gate, P * l.mix_width);
    if (l.branches > 1) branch = std::max(branch, l.branches * P * D);
    if (l.type == QMK_MIXER_ATTENTION) {
      q = std::max(q, P * l.heads * l.q_stride);
      vt = std::max(vt, values_cap(a) * l.kv_heads * l.v_dim);
      continue;
    }
    decay = std::max(decay, P * l.heads * l.head_dim);
    o = std::max(o, P * l.mix_width);
    low = std::max(low, P * (l.rank + l.gate_rank));
    state.fit(P, l.heads, l.head_dim, l.v_dim, l.type == QMK_MIXER_GLA);
    if (l.type == QMK_MIXER_DELTA) {
      qkv = std::max(qkv, P * conv_channels(l));
      values = std::max(values, static_cast<size_t>(chunks_of(static_cast<int>(P))) * kChunkTokens * l.mix_width);
      beta = std::max(beta, P * ((l.heads + 15) / 16 * 16));
    } else {
      qkv = std::max(qkv, P * (2 * l.heads * l.head_dim + l.mix_width));
    }
  }
  Carver c{static_cast<char*>(base)};
  PlainBuffers<T> local;
  if (b == nullptr) b = &local;
  b->split = split_buffers(c);
  b->x = c.take<float>(P * D);
  b->branch = c.take<float>(branch);
  b->qkv = c.take<float>(qkv);
  b->values = c.take<float>(values);
  b->decay = c.take<float>(decay);
  b->beta = c.take<float>(beta);
  b->o = c.take<float>(o);
  state.take(c);
  b->state = state;
  b->h = OperandRows<T>(c, h);
  b->q = c.take<T>(q);
  b->low = c.take<T>(low);
  b->gate = c.take<T>(gate);
  b->mix = OperandRows<T>(c, mix);
  b->vt = c.take<T>(vt);
  return c.used;
}

inline int keys_cap(const QmkHybridArgs* a, const QmkHybridLayer& l) { return (std::min(l.window - 1 + a->portion_rows, a->max_positions) + 31) & ~31; }

template <class T>
struct PrefillBuffers {
  SplitBuffers split;
  float *x, *u, *fa, *fb, *raw;
  ChunkBuffers state;
  T *p0, *p1, *p2, *rows, *kn, *vt;
  OperandRows<T> h, mix;
};
template <class T>
size_t prefill_buffers(const QmkHybridArgs* a, void* base, PrefillBuffers<T>* b) {
  if (a->streams == 0) return plain_buffers<T>(a, base, nullptr);
  const size_t P = a->portion_rows, D = a->width;
  ChunkBuffers state;
  size_t h = P * D, fa = 0, fb = 0, raw = 0, p0 = 0, p1 = 0, p2 = 0, mix = 0, rows = 0, kn = 0, vt = 0;
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    const size_t W = l.mix_width;
    mix = std::max(mix, P * std::max<size_t>(W, l.has_mlp ? l.ff : 0));
    if (l.type == QMK_MIXER_RGLRU) {
      p0 = std::max(p0, P * W);
      p1 = std::max(p1, P * W);
      p2 = std::max(p2, P * W);
      fa = std::max(fa, P * W);
      fb = std::max(fb, P * W);
    } else if (l.type == QMK_MIXER_LATENT) {
      const size_t keys = keys_cap(a, l);
      p0 = std::max(p0, P * l.heads * l.q_stride);
      p1 = std::max(p1, P * W);
      raw = std::max(raw, P * (l.rank + l.rot_dim));
      rows = std::max(rows, keys * (l.rank + l.rot_dim));
      kn = std::max(kn, keys * l.heads * l.head_dim);
      vt = std::max(vt, keys * W);
    } else {
      h = std::max(h, 5 * P * D);
      p0 = std::max(p0, P * W);
      p1 = std::max(p1, P * l.rank);
      fa = std::max(fa, 3 * P * W);
      fb = std::max(fb, P * W);
      raw = std::max(raw, P * W);
      state.fit(P, l.heads, l.head_dim, l.head_dim, true);
    }
  }
  Carver c{static_cast<char*>(base)};
  b->split = split_buffers(c);
  b->x = c.take<float>(P * a->streams * D);
  b->u = c.take<float>(P * D);
  b->fa = c.take<float>(fa);
  b->fb = c.take<float>(fb);
  b->raw = c.take<float>(raw);
  state.take(c);
  b->state = state;
  b->h = OperandRows<T>(c, h);
  b->p0 = c.take<T>(p0);
  b->p1 = c.take<T>(p1);
  b->p2 = c.take<T>(p2);
  b->mix = OperandRows<T>(c, mix);
  b->rows = c.take<T>(rows);
  b->kn = c.take<T>(kn);
  b->vt = c.take<T>(vt);
  return c.used;
}

template <class S, int KIND>
constexpr bool priced_as = kTileCosts[KIND].bm == S::BM && kTileCosts[KIND].bn == S::BN && kTileCosts[KIND].bk == S::BK;
static_assert(priced_as<Tiles64, 0> && priced_as<Wide256, 1> && priced_as<Wide64, 2> && priced_as<Turns96, 3> && priced_as<Turns128, 4> && priced_as<Tall192, 5>, "tiles and their prices");
static_assert(priced_as<Tall256, 6> && priced_as<Turns192, 7> && priced_as<Turns256, 8> && priced_as<Tiles32, 9> && priced_as<Few64, 10> && priced_as<Few32, 11>, "tiles and their prices");
template <class S, int KIND>
constexpr bool priced_as_parts = kPartCosts[KIND].bm == S::BM && kPartCosts[KIND].bn == S::BN && S::kSplits;
static_assert(priced_as_parts<Parts32, 0> && priced_as_parts<Parts64, 1> && priced_as_parts<PartsWide, 2>, "tiles of operands in parts and their prices");

template <class TA, class TW, class T>
void launch_gemm(GemmArgs g, const SplitBuffers& split, hipStream_t st) {
  const int n = std::max(g.N, g.last_n);
  g.tickets = split.tickets;
  g.partial = reinterpret_cast<float*>(split.partial);
  auto launch = [&](auto kernel, int bm, int bn, int threads) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((n + bn - 1) / bn * ((g.M + bm - 1) / bm) * g.splits), 1, g.groups), dim3(threads), 0, st, g);
  };
  g.splits = 1;
  if constexpr (sizeof(TA) == 2 && sizeof(TW) == 2) {
    if (g.K % 64 == 0) {
      auto direct = [&](auto s) { using S = decltype(s); launch(gemm_direct<T, S>, S::BM, S::BN, S::kThreadCount); };
      auto pipe = [&](auto s) { using S = decltype(s); launch(gemm_pipe<T, S>, S::BM, S::BN, S::kThreadCount); };
      auto few = [&](auto s) { using S = decltype(s); launch(gemm_few<T, S>, S::BM, S::BN, S::kThreadCount); };
      auto turns = [&](auto s) { using S = decltype(s); launch(gemm_turns<T, S>, S::BM, S::BN, S::kThreadCount); };
      switch (choose_tiles(g.M, n, g.K, g.groups, g.epi == EPI_RESIDUAL)) {
        case 0: pipe(Tiles64{}); break;
        case 1: pipe(Wide256{}); break;
        case 2: direct(Wide64{}); break;
        case 3: pipe(Turns96{}); break;
        case 4: pipe(Turns128{}); break;
        case 5: pipe(Tall192{}); break;
        case 6: pipe(Tall256{}); break;
        case 7: turns(Turns192{}); break;
        case 8: turns(Turns256{}); break;
        case 9: pipe(Tiles32{}); break;
        case 10: direct(Few64{}); break;
        default: few(Few32{}); break;
      }
      return;
    }
  }
  if constexpr (sizeof(TA) == 4 && sizeof(TW) == 2) {
    if (g.a_part != 0) {
      const PartTiles tiles = choose_part_tiles(g.M, n, g.K, g.groups);
      g.splits = tiles.splits;
      auto parts = [&](auto s) { using S = decltype(s); launch(gemm_pipe<T, S, 3>, S::BM, S::BN, S::kThreadCount); };
      switch (tiles.kind) {
        case 0: parts(Parts32{}); break;
        case 1: parts(Parts64{}); break;
        default: parts(PartsWide{}); break;
      }
      return;
    }
  }
  if constexpr (sizeof(TA) == 4 || sizeof(TW) == 4) {
    if (g.K <= 64) {
      launch(gemm_short<TA, TW, T>, 64, 64, kPfThreads);
      return;
    }
  }
  const RegisterTiles c = choose_register_tiles(g.M, n, g.K, g.groups, sizeof(TA) == 4 || sizeof(TW) == 4);
  g.splits = c.splits;
  if (c.large) launch(gemm<TA, TW, T, 128, 128, 2>, 128, 128, kPfThreads);
  else launch(gemm<TA, TW, T, 64, 64, 1>, 64, 64, kPfThreads);
}

// Two bf16 products that need nothing of each other: in one launch where both take tiles of 64 x 64, whose time is mostly a launch's beginning and end (us, 443 x 2048 x 512 and
// 2048 x 443 x 512, two launches -> one: 12.0 -> 8.4; larger tiles fill the chip by themselves; the kinds for fewer tokens, as of a short portion with nothing before it, stay two launches:
// not tried).
template <class T>
void launch_gemm_pair(GemmPair pair, const SplitBuffers& split, hipStream_t st) {
  auto small = [](const GemmArgs& g) { return g.groups == 1 && g.K % 64 == 0 && choose_tiles(g.M, g.N, g.K, 1, g.epi == EPI_RESIDUAL) == 0; };
  if (!small(pair.g[0]) || !small(pair.g[1])) {
    for (const GemmArgs& g : pair.g) launch_gemm<u16, u16, T>(g, split, st);
    return;
  }
  using S = Tiles64;
  unsigned tiles = 0;
  for (GemmArgs& g : pair.g) {
    g.splits = 1;
    tiles = std::max(tiles, static_cast<unsigned>((g.N + S::BN - 1) / S::BN * ((g.M + S::BM - 1) / S::BM)));
  }
  hipLaunchKernelGGL((gemm_pipe_pair<T, S>), dim3(tiles, 2), dim3(S::kThreadCount), 0, st, pair);
}

// Ahead of a portion's other launches.
template <class T>
void begin_portion(const SplitBuffers& split, hipStream_t st) {
  if constexpr (sizeof(T) == 4) hipLaunchKernelGGL(clear_tickets, dim3(1), dim3(kPfThreads), 0, st, split.tickets, kMaxTickets);
}

// A recurrence over the portion, from its projections to what its norm reads; of the delta rule all but its scan.
template <class T, int KIND>
void run_chunks(ChunkArgs g, hipStream_t st) {
  g.segment = segment_chunks<T>(g.M);
  const int chunks = chunks_of(g.M), segments = segments_of(g.M, g.segment);
  auto run = [&](auto wave_tiles) {
    constexpr int kTiles = decltype(wave_tiles)::value;
    const dim3 block(kPfThreads);
    hipLaunchKernelGGL((chunk_prepare<KIND, kTiles>), dim3(chunks, g.heads), block, 0, st, g);
    if constexpr (KIND != CHUNK_DELTA) {
      const unsigned groups = g.heads * ((g.n + 63) / 64);
      if (segments > 1) {
        hipLaunchKernelGGL((segment_scan<kTiles * 4, false>), dim3(groups * (segments - 1)), block, 0, st, g);
        if (segments > kOwnStarts) hipLaunchKernelGGL(segment_starts, dim3((g.heads * g.dim * (g.n / 4) + kPfThreads - 1) / kPfThreads), block, 0, st, g);
      }
      hipLaunchKernelGGL((segment_scan<kTiles * 4, true>), dim3(groups * segments), block, 0, st, g);
    }
  };
  switch (chunk_tiles(g.dim)) {
    case 4: return run(std::integral_constant<int, 1>{});
    case 8: return run(std::integral_constant<int, 2>{});
    default: return run(std::integral_constant<int, 4>{});
  }
}

// The delta rule's chunks one after the other.
inline void launch_scan(const ChunkArgs& g, hipStream_t st) {
  auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(g.heads, g.n / 16), dim3(kPfThreads), 0, st, g); };
  switch (chunk_tiles(g.dim)) {
    case 4: return run(chunk_scan<1, kChunkWaves>);
    case 8: return run(chunk_scan<2, kChunkWaves>);
    default: return run(chunk_scan<4, kChunkWaves>);
  }
}

// Whether a delta rule's chunks are walked in the launch of the attention beside it: where a CU holds a workgroup of either.  Elsewhere (fp32, larger heads) the branches follow one
// another, each with its output gate ahead of its chunks: the order that one launch needs only costs there (us a call of the 1b shape in fp32, 64 tokens behind 500 1907 and so 1894, 200 behind 500
// 2870 and 2846; two layers with heads of 256, 530 tokens 607 and 602).
template <class T>
bool one_launch(const QmkHybridLayer& attention, const QmkHybridLayer& delta) {
  return sizeof(T) == 2 && attention.q_stride <= 128 && attention.v_dim <= 128 && chunk_tiles(delta.head_dim) <= 8;
}

// rows: where the rotated part of a latent attention's keys is, behind the latent.  In fp32 two groups of waves share a workgroup's queries, except for
// the largest heads, where they take 140 KB of LDS and more registers than there are (us a portion of one layer, 16 heads of 256 | 256, one group -> two:
// 4000 tokens 2963 -> 3416, 1025 tokens 453 -> 508).  In bf16 the largest heads leave no registers for a second wave a SIMD, and take stages of 32 keys.
// In bf16 heads of 128 and of 192 share a stage's work among the waves of 16 queries while such workgroups are all on the chip at once, two a CU of 128 and one of 192 (us, 16 heads behind
// 400 keys, a wave's queries by themselves -> shared: 192 | 128, 43 tokens 16.2 -> 13.4, 200 tokens 19.3 -> 16.3, 500 tokens 25.6 -> 32.4; 128 | 128, 20 tokens 16.6 -> 11.8,
// 200 tokens 19.0 -> 14.8, 500 tokens 25.4 -> 21.2, 1000 tokens 35.1 -> 46.9; behind 1000 keys 192 | 128, 43 tokens 28.2 -> 24.3, 250 tokens 32.0 -> 27.9; 128 | 128, 43 tokens 27.6 -> 22.2,
// 250 tokens 31.2 -> 26.0, 500 tokens 35.9 -> 33.3; behind 4000 and 16000 keys 128 | 128, 260 tokens 81 -> 74 and 284 -> 262, 500 tokens 88 -> 84 and 291 -> 287; 192 | 128, 250 tokens 86 -> 80 and
// 297 -> 281: keys are read four times as often, but out of the caches).
// In fp32 the same heads take few_attention with one a CU (us, 16 heads, window_attention -> few_attention: 192 | 128, 43 tokens 16.1 -> 12.2, 200 tokens 30.0 -> 20.7, 400 tokens 50.2 -> 55.8;
// behind 1000 keys 250 tokens 133 -> 83, behind 16000 1641 -> 1027; 128 | 128 behind 200 keys, 43 tokens 29.2 -> 19.0, 400 tokens 58.6 -> 63.2, behind 1000 keys 250 tokens 113 -> 72, behind
// 16000 1294 -> 796).
// `beside`: a delta rule that shares the launch, its chunks prepared.
template <class T>
void launch_attention(const QmkHybridArgs* a, const QmkHybridLayer& l, const T* q, Keys<T> keys, const T* rows, const T* vt, const T* gate, int first, int cap, Operand<T> out,
                      const ChunkArgs* beside, hipStream_t st) {
  if constexpr (sizeof(T) == 2) {
    const AttentionArgs args{q, keys, rows, vt, gate, l, first, a->position, a->tokens, cap, out.at};
    auto workgroups = [&](int queries) { return static_cast<unsigned>((a->tokens + queries - 1) / queries * l.heads); };
    if (beside != nullptr) {
      auto both = [&](auto one_tile, auto two_tiles, int queries) {
        const dim3 grid(beside->heads * (beside->n / 16) + workgroups(queries));
        if (chunk_tiles(beside->dim) == 4) hipLaunchKernelGGL(one_tile, grid, dim3(kPfThreads), 0, st, *beside, args);
        else hipLaunchKernelGGL(two_tiles, grid, dim3(kPfThreads), 0, st, *beside, args);
      };
      if (l.v_dim <= 64) both(scan_and_attend<1, 4, 4, 64, 2, false>, scan_and_attend<2, 4, 4, 64, 2, false>, 64);
      else if (workgroups(16) <= 512) both(scan_and_attend<1, 4, 8, 64, 2, true>, scan_and_attend<2, 4, 8, 64, 2, true>, 16);
      else both(scan_and_attend<1, 4, 8, 64, 2, false>, scan_and_attend<2, 4, 8, 64, 2, false>, 64);
      return;
    }
    auto launch = [&](auto kernel, int queries) { hipLaunchKernelGGL(kernel, dim3(workgroups(queries)), dim3(kPfThreads), 0, st, args); };
    auto rows_of = [&](auto shared, auto all, int a_cu) { workgroups(16) <= 256u * a_cu ? launch(shared, 16) : launch(all, 64); };
    if (l.q_stride <= 128 && l.v_dim <= 64) launch(attention_rows<4, 4, 64, 2, 2>, 64);
    else if (l.q_stride <= 128 && l.v_dim <= 128) rows_of(attention_rows<4, 8, 64, 2, 2, true>, attention_rows<4, 8, 64, 2, 2>, 2);
    else if (l.q_stride <= 192 && l.v_dim <= 128) rows_of(attention_rows<6, 8, 64, 2, 1, true>, attention_rows<6, 8, 64, 2, 2>, 1);
    else launch(attention_rows<8, 16, 32, 3, 1>, 64);
  } else {
    const int few_runs = (a->tokens + 15) / 16;
    auto launch_few = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(few_runs, l.heads), dim3(kPfThreads), 0, st, q, keys, rows, vt, gate, l, first, a->position, a->tokens, cap, out);
    };
    auto launch = [&](auto kernel, int groups) {
      hipLaunchKernelGGL(kernel, dim3((a->tokens + 63) / 64, l.heads), dim3(kPfThreads * groups), 0, st, q, keys, rows, vt, gate, l, first, a->position, a->tokens, cap, out);
    };
    const bool few = few_runs * l.heads <= 256;
    if (l.q_stride <= 128 && l.v_dim <= 64) launch(window_attention<4, 4, 2>, 2);
    else if (l.q_stride <= 128 && l.v_dim <= 128) few ? launch_few(few_attention<4, 8>) : launch(window_attention<4, 8, 2>, 2);
    else if (l.q_stride <= 192 && l.v_dim <= 128) few ? launch_few(few_attention<6, 8>) : launch(window_attention<6, 8, 2>, 2);
    else launch(window_attention<8, 16, 1>, 1);
  }
}

template <class T>
int prefill_plain(const QmkHybridArgs* a);

template <class T>
int prefill(const QmkHybridArgs* a) {
  if (a->streams == 0) return prefill_plain<T>(a);
  PrefillBuffers<T> b;
  if (prefill_buffers<T>(a, a->workspace, &b) > a->workspace_bytes) return QMK_ERR_SCRATCH;
  const hipStream_t st = static_cast<hipStream_t>(a->stream);
  begin_portion<T>(b.split, st);
  const int M = a->tokens, D = a->width, S = a->streams, P = a->portion_rows;
  const dim3 block(kPfThreads);
  hipLaunchKernelGGL(embed_tokens, dim3(M), block, 0, st, a->embed, a->token_in, a->vocab, a->layers[0].hc, S, D, b.x, b.u);
  auto gemm_args = [&](Operand<T> in, int lda, const u16* w, int N, int K, const QmkHybridLayer& l, int epi) {
    GemmArgs g{};
    g.a = in.at; g.a_part = in.part; g.lda = lda; g.w = w; g.ldw = K; g.M = M; g.N = g.last_n = N; g.K = K; g.groups = 1;
    g.layer = l; g.epi = epi; g.position = a->position; g.streams = S; g.width = D; g.rows_cap = P;
    return g;
  };
  auto whole = [](T* rows) { return Operand<T>{rows, 0}; };
  auto residual = [&](const u16* w, int K, const QmkHybridLayer& l, bool down) {
    GemmArgs g = gemm_args(b.mix.of(K), K, w, D, K, l, EPI_RESIDUAL);
    g.f0 = b.x; g.f1 = b.u; g.down = down; g.next = down ? l.next2 : l.next1;
    launch_gemm<T, u16, T>(g, b.split, st);
  };
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    const int W = l.mix_width;
    if (l.type != QMK_MIXER_WKV)
      hipLaunchKernelGGL(norm_rows<T>, dim3(M), block, 0, st, b.u, l.norm1, nullptr, M, D, a->width_true, a->eps, b.h.of(D));
    if (l.type == QMK_MIXER_RGLRU) {
      GemmArgs g = gemm_args(b.h.of(D), D, l.in_w, l.in_rows, D, l, EPI_RGLRU_IN);
      g.out = b.p0; g.out2 = b.p1;
      launch_gemm<T, u16, T>(g, b.split, st);
      const long long quads = static_cast<long long>(M) * (W / 4);
      hipLaunchKernelGGL(causal_conv<T>, dim3(static_cast<unsigned>((quads + kPfThreads - 1) / kPfThreads)), block, 0, st, b.p1, l, a->slot, a->flip, M, b.p2);
      GemmArgs e = gemm_args(whole(b.p2), W, l.mid_w, 2 * l.block_dim, l.block_dim, l, EPI_LRU_GATES);
      e.groups = l.blocks; e.a_step = l.block_dim; e.w_step = 2LL * l.block_dim * l.block_dim;
      e.src = b.p2; e.f0 = b.fa; e.f1 = b.fb;
      launch_gemm<T, u16, T>(e, b.split, st);
      hipLaunchKernelGGL(lru_scan<T>, dim3(W / kScanChannels), dim3(kScanChannels * kScanRuns), 0, st, b.fa, b.fb, b.p0, l, a->slot, M, b.mix.of(W));
    } else if (l.type == QMK_MIXER_LATENT) {
      GemmArgs g = gemm_args(b.h.of(D), D, l.in_w, l.in_rows, D, l, EPI_LATENT_IN);
      g.out = b.p0; g.out2 = b.p1; g.f0 = b.raw;
      launch_gemm<T, u16, T>(g, b.split, st);
      const int first = std::max(0, a->position + 1 - l.window), keys = a->position + M - first, cap = keys_cap(a, l), width = l.rank + l.rot_dim;
      hipLaunchKernelGGL(latent_rows<T>, dim3(keys), block, 0, st, b.raw, l, a->slot, first, a->position, a->eps, b.rows);
      GemmArgs k = gemm_args(whole(b.rows), width, l.uk_w, l.heads * l.head_dim, l.rank, l, EPI_STORE);
      k.M = keys; k.out = b.kn; k.ldo = l.heads * l.head_dim;
      GemmArgs v = gemm_args(whole(nullptr), l.rank, nullptr, keys, l.rank, l, sizeof(T) == 2 ? EPI_STORE_VALUES : EPI_STORE);   // transposed: W_uv rows x keys
      v.a = l.uv_w; v.w = b.rows; v.ldw = width; v.M = l.heads * l.v_dim; v.out = b.vt; v.ldo = cap;
      if constexpr (sizeof(T) == 2) {
        launch_gemm_pair<T>({{k, v}}, b.split, st);
      } else {
        launch_gemm<T, u16, T>(k, b.split, st);
        launch_gemm<u16, T, T>(v, b.split, st);
      }
      const Keys<T> expanded{b.kn, l.heads * l.head_dim, l.head_dim, 1};
      launch_attention<T>(a, l, b.p0, expanded, b.rows, b.vt, b.p1, first, cap, b.mix.of(W), nullptr, st);
    } else {
      const int N = W;
      hipLaunchKernelGGL(shift_mix<T>, dim3(M), block, 0, st, b.u, l, a->slot, a->flip, M, P, D, a->width_true, a->eps, b.h.of(D));
      GemmArgs g = gemm_args(b.h.of(D), D, l.in_w, N, D, l, EPI_WKV_IN);
      g.groups = 5; g.last_n = l.rank; g.a_step = static_cast<long long>(P) * D; g.w_step = static_cast<long long>(N) * D;
      g.f0 = b.fa; g.out = b.p0; g.out2 = b.p1;
      launch_gemm<T, u16, T>(g, b.split, st);
      GemmArgs d = gemm_args(whole(b.p1), l.rank, l.mid_w, N, l.rank, l, EPI_WKV_DECAY);
      d.f0 = b.fb; d.ldo = N;
      launch_gemm<T, u16, T>(d, b.split, st);
      const size_t step = static_cast<size_t>(P) * N;
      ChunkArgs c{};
      c.layer = l; c.q = b.fa; c.k = b.fa + step; c.values = b.fa + 2 * step; c.decay = b.fb; c.out = b.raw;
      c.chunks = b.state.chunks; c.starts = b.state.starts; c.fades = b.state.fades;
      c.M = M; c.heads = l.heads; c.dim = c.n = l.head_dim; c.ld = c.value_ld = N; c.slot = a->slot; c.flip = a->flip;
      run_chunks<T, CHUNK_WKV>(c, st);
      hipLaunchKernelGGL(wkv_out<T>, dim3((M * l.heads + 3) / 4), block, 0, st, b.raw, b.p0, l, M, a->eps, b.mix.of(W));
    }
    residual(l.o_w, W, l, false);
    if (l.has_mlp) {
      hipLaunchKernelGGL(norm_rows<T>, dim3(M), block, 0, st, b.u, l.norm2, nullptr, M, D, a->width_true, a->eps, b.h.of(D));
      GemmArgs g = gemm_args(b.h.of(D), D, l.mlp_w, 2 * l.ff, D, l, EPI_GEGLU);
      g.out = b.mix.at; g.out_part = b.mix.of(l.ff).part;
      launch_gemm<T, u16, T>(g, b.split, st);
      residual(l.down_w, l.ff, l, true);
    }
    if (a->layer_out != nullptr)
      hipLaunchKernelGGL(sum_streams, dim3(M), block, 0, st, b.x, S, D, a->layer_out + static_cast<size_t>(i) * M * D);
  }
  if (a->num_want > 0) {
    hipLaunchKernelGGL(norm_rows<T>, dim3(a->num_want), block, 0, st, b.u, a->final_norm, a->want, M, D, a->width_true, a->eps, b.h.of(D));
    GemmArgs g = gemm_args(b.h.of(D), D, a->head, a->vocab_rows, D, a->layers[0], EPI_LOGITS);
    g.M = a->num_want; g.f0 = a->logits; g.ldo = a->vocab_rows;
    launch_gemm<T, u16, T>(g, b.split, st);
  }
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_LAUNCH;
}

template <class T>
int prefill_plain(const QmkHybridArgs* a) {
  PlainBuffers<T> b;
  if (plain_buffers<T>(a, a->workspace, &b) > a->workspace_bytes) return QMK_ERR_SCRATCH;
  const hipStream_t st = static_cast<hipStream_t>(a->stream);
  begin_portion<T>(b.split, st);
  const int M = a->tokens, D = a->width;
  const size_t rows = static_cast<size_t>(a->portion_rows) * D;
  const dim3 block(kPfThreads);
  auto gemm_args = [&](Operand<T> in, const u16* w, int N, int K, const QmkHybridLayer& l, int epi) {
    GemmArgs g{};
    g.a = in.at; g.a_part = in.part; g.lda = K; g.w = w; g.ldw = K; g.M = M; g.N = g.last_n = N; g.K = K; g.groups = 1;
    g.layer = l; g.epi = epi; g.position = a->position; g.slot = a->slot; g.width = D; g.ldo = D;
    g.logit_scale = a->logit_scale; g.logit_softcap = a->logit_softcap;
    return g;
  };
  auto whole = [](T* rows) { return Operand<T>{rows, 0}; };
  auto project_attention = [&](const QmkHybridLayer& l) {
    GemmArgs g = gemm_args(b.h.of(D), l.in_w, l.in_rows, D, l, EPI_ATTENTION_IN);
    g.out = b.q; g.out2 = b.gate;
    launch_gemm<T, u16, T>(g, b.split, st);
  };
  auto attend = [&](const QmkHybridLayer& l, const ChunkArgs* beside) {
    const int row = l.head_dim + l.v_dim, pitch = l.kv_heads * row, keys = a->position + M, cap = static_cast<int>(values_cap(a));
    const T* cache = static_cast<const T*>(l.cache) + static_cast<size_t>(a->slot) * l.ring * pitch;
    hipLaunchKernelGGL(transpose_values<T>, dim3((keys + 63) / 64, (l.v_dim + 63) / 64, l.kv_heads), block, 0, st, cache, pitch, row, l.head_dim, l.v_dim, keys, cap, b.vt);
    launch_attention<T>(a, l, b.q, Keys<T>{cache, pitch, row, l.heads / l.kv_heads}, nullptr, b.vt, b.gate, 0, cap, b.mix.of(l.mix_width), beside, st);
  };
  auto chunk_args = [&](const QmkHybridLayer& l) {
    ChunkArgs c{};
    c.layer = l; c.decay = b.decay; c.chunks = b.state.chunks; c.starts = b.state.starts; c.fades = b.state.fades; c.out = b.o;
    c.M = M; c.heads = l.heads; c.dim = l.head_dim; c.n = l.v_dim; c.slot = a->slot; c.flip = a->flip;
    return c;
  };
  auto decays = [&](const QmkHybridLayer& l, int ld, int epi) {
    const int keys = l.heads * l.head_dim;
    GemmArgs e = gemm_args(whole(b.low), l.mid_w, keys, l.rank, l, epi);
    e.lda = ld; e.f0 = b.decay; e.ldo = keys;
    launch_gemm<T, u16, T>(e, b.split, st);
  };
  auto delta_gate = [&](const QmkHybridLayer& l) {
    GemmArgs f = gemm_args(whole(b.low + l.rank), l.gate_w, l.mix_width, l.gate_rank, l, EPI_SIGMOID);
    f.lda = l.rank + l.gate_rank; f.out = b.gate; f.ldo = l.mix_width;
    launch_gemm<T, u16, T>(f, b.split, st);
  };
  // A delta rule up to its scan.  `gate`: with its output gate, which lies where that of an attention does; in one launch with that it comes behind.
  auto prepare_delta = [&](const QmkHybridLayer& l, bool gate) {
    const int beta_ld = (l.heads + 15) / 16 * 16;
    GemmArgs g = gemm_args(b.h.of(D), l.in_w, l.in_rows, D, l, EPI_DELTA_IN);
    g.f1 = b.qkv; g.out2 = b.low; g.f0 = b.beta; g.ldo = beta_ld;
    launch_gemm<T, u16, T>(g, b.split, st);
    decays(l, l.rank + l.gate_rank, EPI_DELTA_DECAY);
    if (gate) delta_gate(l);
    ChunkArgs c = chunk_args(l);
    c.q = b.qkv; c.beta = b.beta; c.beta_ld = beta_ld; c.values = b.values;
    run_chunks<T, CHUNK_DELTA>(c, st);
    return c;
  };
  auto state_rows = [&](const QmkHybridLayer& l) {
    hipLaunchKernelGGL(state_out<T>, dim3((M * l.heads + 3) / 4), block, 0, st, b.o, b.gate, l, M, a->eps, b.mix.of(l.mix_width));
  };
  auto finish_delta = [&](const QmkHybridLayer& l) {
    const int channels = conv_channels(l);
    if (l.taps > 1)
      hipLaunchKernelGGL(keep_inputs, dim3((channels + kPfThreads - 1) / kPfThreads), block, 0, st, b.qkv, l, channels, a->slot, a->flip, M);
    state_rows(l);
  };
  auto run_gla = [&](const QmkHybridLayer& l) {
    const int W = l.mix_width, keys = l.heads * l.head_dim;
    GemmArgs g = gemm_args(b.h.of(D), l.in_w, l.in_rows, D, l, EPI_GLA_IN);
    g.f0 = b.qkv; g.out = b.gate; g.out2 = b.low;
    launch_gemm<T, u16, T>(g, b.split, st);
    decays(l, l.rank, EPI_GLA_DECAY);
    ChunkArgs c = chunk_args(l);
    c.q = b.qkv; c.k = b.qkv + keys; c.values = b.qkv; c.ld = c.value_ld = 2 * keys + W; c.value_at = 2 * keys;
    run_chunks<T, CHUNK_GLA>(c, st);
    state_rows(l);
  };
  auto project_out = [&](const QmkHybridLayer& l) {
    GemmArgs o = gemm_args(b.mix.of(l.mix_width), l.o_w, D, l.mix_width, l, l.branches > 1 ? EPI_LOGITS : EPI_ADD);
    o.f0 = l.branches > 1 ? b.branch + l.branch * rows : b.x;
    launch_gemm<T, u16, T>(o, b.split, st);
  };
  int runs_done = 0;
  // x as entry l reads it: its norm (or [x; embedding]) -> h; `want`: of those rows alone, x stays.
  auto residual = [&](const QmkHybridLayer& l, const int32_t* want, int count, bool added, float* dump) {
    ResidualArgs g{};
    g.x = b.x; g.table = a->embed; g.tokens = a->token_in; g.vocab = a->vocab; g.want = want; g.dump = dump;
    g.weight = l.type == QMK_ENTRY_JOIN ? nullptr : l.norm1;
    g.embed = l.x_from < 0; g.M = M; g.D = D; g.width = a->width_true; g.norm = l.norm; g.eps = a->eps;
    if (added && l.prev >= 0 && a->layers[l.prev].branches == 2) {
      const QmkHybridLayer* before = a->layers + l.prev;
      g.a = b.branch; g.b = b.branch + rows; g.wa = before[0].out_norm; g.wb = before[1].out_norm; g.scale = before[0].out_scale;
    }
    hipLaunchKernelGGL(residual_rows<T>, dim3(count), block, 0, st, g, b.h.of(l.type == QMK_ENTRY_JOIN ? 2 * D : D));
  };
  auto dump_of = [&](const QmkHybridLayer& l) {   // where the run before this entry is asked for
    return a->layer_out != nullptr && l.prev >= 0 ? a->layer_out + static_cast<size_t>(runs_done++) * M * D : nullptr;
  };
  bool walked = false;      // the next entry's chunks, beside the attention of this one
  for (int i = 0; i < a->num_layers; ++i) {
    const QmkHybridLayer& l = a->layers[i];
    if (l.type == QMK_ENTRY_FINAL) {
      float* dump = dump_of(l);
      if (dump != nullptr) residual(l, nullptr, M, true, dump);     // (and x is complete)
      if (a->num_want > 0) {
        residual(l, a->want, a->num_want, dump == nullptr, nullptr);
        GemmArgs g = gemm_args(b.h.of(D), a->head, a->vocab_rows, D, l, EPI_CAPPED_LOGITS);
        g.M = a->num_want; g.f0 = a->logits; g.ldo = a->vocab_rows;
        launch_gemm<T, u16, T>(g, b.split, st);
      }
      break;
    }
    if (l.branch == 0) residual(l, nullptr, M, true, dump_of(l));
    if (l.type == QMK_ENTRY_JOIN) {
      GemmArgs g = gemm_args(b.h.of(2 * D), l.in_w, D, 2 * D, l, EPI_LOGITS);
      g.f0 = b.x;
      launch_gemm<T, u16, T>(g, b.split, st);
      continue;
    }
    if (l.type == QMK_MIXER_ATTENTION) {
      project_attention(l);
      walked = l.branch + 1 < l.branches && a->layers[i + 1].type == QMK_MIXER_DELTA && one_launch<T>(l, a->layers[i + 1]);
      const ChunkArgs c = walked ? prepare_delta(a->layers[i + 1], false) : ChunkArgs{};
      attend(l, walked ? &c : nullptr);
    } else if (l.type == QMK_MIXER_DELTA) {
      if (walked) delta_gate(l);
      else launch_scan(prepare_delta(l, true), st);
      walked = false;
      finish_delta(l);
    } else {
      run_gla(l);
    }
    project_out(l);
    if (l.branch + 1 == l.branches) {
      const QmkHybridLayer& head = a->layers[i - l.branch];
      if (head.has_mlp) {
        GemmArgs g = gemm_args(b.h.of(D), head.mlp_w, 2 * head.ff, D, head, EPI_GEGLU);
        g.out = b.mix.at; g.out_part = b.mix.of(head.ff).part;
        launch_gemm<T, u16, T>(g, b.split, st);
        GemmArgs d = gemm_args(b.mix.of(head.ff), head.down_w, D, head.ff, head, EPI_ADD);
        d.f0 = b.x;
        launch_gemm<T, u16, T>(d, b.split, st);
      }
    }
  }
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_LAUNCH;
}

}  // namespace hybrid
}  // namespace qmk

using namespace qmk;
using namespace qmk::hybrid;

extern "C" uint64_t qmk_hybrid_decode_bytes(const QmkHybridArgs* a) {
  if (check_shape(a) != QMK_OK || a->max_splits < 1 || a->max_splits > kMaxParts) return 0;
  DecodeBuffers b;
  return decode_buffers(a, nullptr, &b);
}

extern "C" uint64_t qmk_hybrid_prefill_bytes(const QmkHybridArgs* a) {
  if (check_shape(a) != QMK_OK || a->portion_rows < 1 || a->max_positions < 1) return 0;
  if (a->dtype == QMK_HYBRID_F32) {
    PrefillBuffers<float> b;
    return prefill_buffers<float>(a, nullptr, &b);
  }
  PrefillBuffers<u16> b;
  return prefill_buffers<u16>(a, nullptr, &b);
}

extern "C" int qmk_hybrid_prefill(const QmkHybridArgs* a) {
  if (a == nullptr) return QMK_ERR_NULL_ARG;
  if (int rc = check_launch(a, a->tokens); rc != QMK_OK) return rc;
  if (a->tokens > a->portion_rows || a->num_want < 0 || a->num_want > a->tokens) return QMK_ERR_SHAPE;
  if (a->num_want > 0 && (a->want == nullptr || a->logits == nullptr)) return QMK_ERR_NULL_ARG;
  return a->dtype == QMK_HYBRID_F32 ? prefill<float>(a) : prefill<u16>(a);
}

extern "C" int qmk_hybrid_decode_step(const QmkHybridArgs* a) {
  if (int rc = check_launch(a, 1); rc != QMK_OK) return rc;
  if (a->instructions == nullptr || a->barriers == nullptr || a->logits == nullptr) return QMK_ERR_NULL_ARG;
  if (a->num_queues < 1 || a->num_insts < 1 || a->barrier_groups < 1 || a->max_splits < 1 || a->max_splits > kMaxParts) return QMK_ERR_SHAPE;
  if (reinterpret_cast<uintptr_t>(a->barriers) % 128 != 0) return QMK_ERR_SHAPE;
  DecodeBuffers b;
  if (decode_buffers(a, a->workspace, &b) > a->workspace_bytes) return QMK_ERR_SCRATCH;
  DeviceInfo* dev = nullptr;
  if (int rc = device_info(&dev); rc != QMK_OK) return rc;
  if (a->num_queues > dev->max_queues) return QMK_ERR_TOO_MANY_QUEUES;
  DecodeParams p{};
  p.instructions = a->instructions; p.layers = a->layers_device; p.barriers = a->barriers; p.status = dev->status; p.timeline = a->timeline;
  p.candidates = b.candidates; p.embed = a->embed; p.head = a->head; p.final_norm = a->final_norm; p.token_in = a->token_in; p.token_out = a->token_out;
  p.logits = a->logits; p.units = b.units; p.early_units = b.early_units; p.all_units = b.all_units; p.u = b.u; p.x = b.x; p.sums = b.sums; p.proj = b.proj; p.mix = b.mix; p.absorbed = b.absorbed; p.part = b.part; p.ml = b.ml;
  p.num_insts = a->num_insts; p.num_layers = a->num_layers; p.groups = a->barrier_groups; p.width = a->width; p.width_true = a->width_true;
  p.streams = a->streams; p.vocab = a->vocab; p.vocab_rows = a->vocab_rows; p.slot = a->slot; p.position = a->position; p.flip = a->flip;
  p.max_splits = a->max_splits; p.eps = a->eps; p.logit_scale = a->logit_scale; p.logit_softcap = a->logit_softcap; p.spin_limit = a->spin_limit != 0 ? a->spin_limit : kDefaultSpinLimit;
  const hipStream_t st = static_cast<hipStream_t>(a->stream);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(a->num_queues), dim3(kThreads), 0, st, p); };
  const bool plain = a->streams == 0;
  if (a->dtype == QMK_HYBRID_F32) plain ? launch(decode_megakernel_hybrid<float, true>) : launch(decode_megakernel_hybrid<float, false>);
  else plain ? launch(decode_megakernel_hybrid<u16, true>) : launch(decode_megakernel_hybrid<u16, false>);
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_LAUNCH;
}

extern "C" int qmk_hybrid_status_fetch(void* stream, int32_t detail[4]) {
  DeviceInfo* dev = nullptr;
  if (int rc = device_info(&dev); rc != QMK_OK) return rc;
  if (hipStreamSynchronize(static_cast<hipStream_t>(stream)) != hipSuccess) return QMK_ERR_NO_DEVICE;
  int32_t host[kStatusWords] = {0};
  if (hipMemcpy(host, dev->status, sizeof(host), hipMemcpyDeviceToHost) != hipSuccess) return QMK_ERR_NO_DEVICE;
  if (detail != nullptr)
    for (int i = 0; i < 4; ++i) detail[i] = host[1 + i];
  if (host[0] != 0 && hipMemset(dev->status, 0, sizeof(host)) != hipSuccess) return QMK_ERR_NO_DEVICE;
  return host[0];
}

extern "C" int qmk_hybrid_max_queues(void) {
  DeviceInfo* dev = nullptr;
  return device_info(&dev) == QMK_OK ? dev->max_queues : -QMK_ERR_NO_DEVICE;
}

extern "C" int qmk_hybrid_abi_version(void) { return QMK_HYBRID_ABI_VERSION; }
