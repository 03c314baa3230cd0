// C ABI of the MI355X attention library (see include/mi355_attn.h): handle
// lifetime, host-side validation of every shape before a kernel is launched,
// status/error-message conventions, staging for host-pointer callers.
#include "../../include/mi355_attn.h"

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <new>
#include <string>
#include <vector>

#include "attn_params.h"
#include "kernels.h"

using namespace mi355;

// Workspace of mi355_attn_decode_noalloc: the split-KV partials of one call, (head_dim + 2) floats per
// (layer, sequence, query head, partition), in device memory that exists from the moment the library
// is loaded. Each GPU holds its own copy; host code reaches it only through the address that
// hipGetSymbolAddress returns with that GPU current (resolved in mi355_attn_create), never through
// the array's name.
constexpr size_t kNoAllocSlots = 8192;  // partial slots: 8192 x 258 floats = 8.06 MiB per GPU
constexpr int kNoAllocHeadDim = 256;
static __device__ __align__(256) float scratch[kNoAllocSlots * (kNoAllocHeadDim + 2)];

namespace {

constexpr int kMaxDevices = 64;
float* g_scratch_ptr[kMaxDevices] = {};  // [device]: address of `scratch` on that GPU, set once by create
// Calls on different streams of one GPU share that GPU's `scratch`: each call waits (on its stream, not on the
// host) for the event that the previous call left behind when that call ran on another stream, so eager calls
// never overlap in the workspace. The events are made once per GPU by create. (Captured calls skip this: an
// event recorded inside a capture belongs to the graph.)
hipEvent_t g_scratch_done[kMaxDevices] = {};
hipStream_t g_scratch_stream[kMaxDevices] = {};
bool g_scratch_used[kMaxDevices] = {};

constexpr int kRingSlots = 64;
constexpr int kMaxSplits = kMaxDecodeSplits;

int fail(char** error_msg, int code, const char* fmt, ...) {
  if (error_msg) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    const size_t len = strlen(buf) + 1;
    char* msg = static_cast<char*>(malloc(len));
    if (msg) memcpy(msg, buf, len);
    *error_msg = msg;
  }
  return code;
}

#define HIP_OR_RETURN(expr)                                                                       \
  do {                                                                                            \
    hipError_t e_ = (expr);                                                                       \
    if (e_ != hipSuccess)                                                                         \
      return fail(error_msg, e_ == hipErrorOutOfMemory ? MI355_ATTN_RESOURCE_EXHAUSTED            \
                                                       : MI355_ATTN_INTERNAL,                     \
                  "%s failed: %s", #expr, hipGetErrorString(e_));                                 \
  } while (0)

__global__ void iota_items_kernel(int32_t* lens, int32_t* seq_ids, int n, int q_pos0, int seq) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    lens[i] = q_pos0 + i + 1;
    seq_ids[i] = seq;
  }
}

}  // namespace

constexpr int kSchedInts = 64;  // prefill queue counters and the stream probe's sink word, on a cache line of their own
static_assert(kPrefillSchedInts + 1 <= kSchedInts, "the counters and the sink word");
constexpr int kI8MinRows = 16;  // int8 cache: prefill calls of fewer rows take the row-wise path unless an option moves that

struct mi355_attn {
  mi355_attn_config cfg{};
  CacheGeom geom{};
  int device = 0;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  uint8_t* cache = nullptr;
  uint64_t cache_bytes = 0;
  float* scales = nullptr;
  int32_t* d_window = nullptr;
  int32_t* d_sched = nullptr;  // prefill work-queue counters
  uint32_t* d_tickets = nullptr;  // tickets of launches that merge their own partials, all zero between launches (behind the counters)
  PrefillPlans pf_plans;       // prefill work plans by launch shape
  float* d_pf_acc = nullptr;   // prefill key split: parts of split tiles, allocated on first use
  float* d_pf_ml = nullptr;
  size_t pf_rows = 0;          // rows (of head_dim / of 2 floats) the two hold
  void* d_q_stage = nullptr;   // prefill whose queries are staged (float32 activations; bfloat16 ones over an int8 cache)
  size_t q_stage_bytes = 0;
  void* d_kv_stage = nullptr;  // prefill over an int8 cache: the half planes of the layers of a pass
  size_t kv_stage_bytes = 0;
  int prefill_i8_min_rows = kI8MinRows;  // int8 cache: calls of fewer rows take the row-wise path
  int prefill_i8_stage_mib = 2048;  // int8 cache: limit of the staging area (a pass covers as many layers as fit, at least one)
  int prefill_short = -1;      // the kernel for short calls: 1 always, 0 never, < 0 by rule
  int prefill_key_split = -1;  // < 0 by rule, 0 off, > 0 key blocks per work item
  int prefill_rows16 = -1;     // which prefill kernel: 1 the one on 16x16x32 MFMAs, 0 the one on 32x32x16, < 0 by rule
  // the step before attention: per-layer constants in HBM and what is switched on
  struct LayerTransform {
    bool set = false, rope = false, norm_q = false, norm_k = false, norm_v = false, q_scaled = false, k_scaled = false;
    float eps = 1e-6f, weight_offset = 1.f;
  };
  float* d_transform = nullptr;  // [num_layers][transform_floats(head_dim)]
  std::vector<LayerTransform> transform;
  std::vector<int32_t> window;
  std::vector<int32_t> filled;  // [layer][seq] rows written since the last reset
  // Partials of kFixedRows rows, behind the cache in its allocation and there from creation on: the parts of short prefill
  // calls and the partitions of decode calls of so many partial results, one after the other on the handle's stream.
  float* d_parts = nullptr;
  // partials of larger decode calls, allocated on first use
  float* ws = nullptr;
  size_t ws_rows = 0;
  bool ws_recorded = false;      // a recorded call writes to `ws`
  std::vector<float*> ws_kept;   // earlier ones that recorded calls write to

  // ring of (kv_lens, seq_ids) uploads
  int32_t* h_ring = nullptr;
  int32_t* d_ring = nullptr;
  hipEvent_t ring_ev[kRingSlots] = {};
  bool ring_used[kRingSlots] = {};
  int ring_next = 0;
  int ring_slot_ints = 0;
  // per-row items of the row-wise prefill path
  int32_t* d_items = nullptr;
  size_t d_items_cap = 0;
  // staging for host_io
  void* stage[4] = {nullptr, nullptr, nullptr, nullptr};
  size_t stage_cap[4] = {0, 0, 0, 0};
  // timing
  bool timing = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  bool timed = false;
  DecodeTuning tuning;
  bool rowwise_prefill = false;  // force the row-wise prefill path (cross-checks)
  int prefill_workgroups = 0;    // 0 = one per CU
};

namespace {

int io_size(const mi355_attn* h) { return dtype_size(h->cfg.io_dtype); }
int kv_size(const mi355_attn* h) { return dtype_size(h->cfg.kv_dtype); }

int ensure_stage(mi355_attn* h, int which, size_t bytes, char** error_msg) {
  if (h->stage_cap[which] >= bytes) return 0;
  HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  if (h->stage[which]) HIP_OR_RETURN(hipFree(h->stage[which]));
  h->stage[which] = nullptr;
  h->stage_cap[which] = 0;
  const size_t cap = std::max(bytes, (size_t)1 << 20);
  HIP_OR_RETURN(hipMalloc(&h->stage[which], cap));
  h->stage_cap[which] = cap;
  return 0;
}

// Device view of a caller buffer that the kernels read.
int stage_in(mi355_attn* h, int which, const void* p, size_t bytes, const void** dev, char** error_msg) {
  if (!h->cfg.host_io) {
    *dev = p;
    return 0;
  }
  if (int rc = ensure_stage(h, which, bytes, error_msg)) return rc;
  HIP_OR_RETURN(hipMemcpyAsync(h->stage[which], p, bytes, hipMemcpyHostToDevice, h->stream));
  *dev = h->stage[which];
  return 0;
}

int stage_out_begin(mi355_attn* h, int which, void* p, size_t bytes, void** dev, char** error_msg) {
  if (!h->cfg.host_io) {
    *dev = p;
    return 0;
  }
  if (int rc = ensure_stage(h, which, bytes, error_msg)) return rc;
  *dev = h->stage[which];
  return 0;
}

int stage_out_end(mi355_attn* h, int which, void* p, size_t bytes, char** error_msg) {
  if (!h->cfg.host_io) return 0;
  HIP_OR_RETURN(hipMemcpyAsync(p, h->stage[which], bytes, hipMemcpyDeviceToHost, h->stream));
  HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  return 0;
}

// A room for `rows` partial results: accumulator rows, then (max, sum) pairs.
constexpr size_t kFixedRows = (size_t)kShortPartSlots * kShortPartRows;
float* partials_ml(const mi355_attn* h, float* acc, size_t rows) { return acc + rows * h->cfg.head_dim; }
size_t partials_bytes(const mi355_attn* h, size_t rows) { return rows * (h->cfg.head_dim + 2) * sizeof(float); }

// What the rule of plan_decode asks for, at most: below 2,048 workgroups of a KV head's query heads.
size_t rule_rows(const mi355_attn* h) { return (size_t)2048 * (h->cfg.num_q_heads / h->cfg.num_kv_heads); }

// Room for calls of more than kFixedRows partial results. It is made for whatever the rule may ask for, so that no later
// length or batch allocates again; only counts of partitions that a caller gives can outgrow it. A recorded call goes on
// writing to the room that it was recorded with, so that one is kept until the handle goes.
int ensure_workspace(mi355_attn* h, size_t rows, char** error_msg) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  // (the default stream cannot be captured, and asking about it while another stream is captured is an error)
  if (h->stream) HIP_OR_RETURN(hipStreamIsCapturing(h->stream, &capturing));
  const bool recording = capturing != hipStreamCaptureStatusNone;
  if (h->ws_rows >= rows) {
    h->ws_recorded |= recording;
    return 0;
  }
  if (recording)
    return fail(error_msg, MI355_ATTN_FAILED_PRECONDITION,
                "decode with %zu partial results while the stream is being captured: more than %zu need a workspace that the "
                "handle allocates on first use (make such a call before the capture)",
                rows, std::max(h->ws_rows, kFixedRows));
  HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  if (h->ws_recorded) {
    try {
      h->ws_kept.push_back(h->ws);
    } catch (const std::bad_alloc&) {
      return fail(error_msg, MI355_ATTN_RESOURCE_EXHAUSTED, "out of host memory");
    }
  } else if (h->ws) {
    HIP_OR_RETURN(hipFree(h->ws));
  }
  h->ws = nullptr;
  h->ws_rows = 0;
  h->ws_recorded = false;
  size_t room = std::max(rows, rule_rows(h));
  hipError_t e = hipMalloc(&h->ws, partials_bytes(h, room));
  if (e == hipErrorOutOfMemory && room > rows) {
    (void)hipGetLastError();
    room = rows;
    e = hipMalloc(&h->ws, partials_bytes(h, room));
  }
  HIP_OR_RETURN(e);
  h->ws_rows = room;
  return 0;
}

// Uploads lengths, cache slots and rows in dispatch order (longest sequence
// first) through a ring of pinned slots so that calls can be queued back to
// back without waiting for earlier uploads.
int upload_items(mi355_attn* h, const int32_t* seq_ids, const int32_t* kv_lens, int batch,
                 const int32_t** d_lens, const int32_t** d_seq, const int32_t** d_rows, char** error_msg) {
  const int slot = h->ring_next;
  h->ring_next = (slot + 1) % kRingSlots;
  if (h->ring_used[slot]) HIP_OR_RETURN(hipEventSynchronize(h->ring_ev[slot]));
  int32_t* hs = h->h_ring + (size_t)slot * h->ring_slot_ints;
  int32_t* ds = h->d_ring + (size_t)slot * h->ring_slot_ints;
  int32_t* order = hs + 2 * (size_t)batch;
  for (int b = 0; b < batch; ++b) order[b] = b;
  std::stable_sort(order, order + batch, [&](int x, int y) { return kv_lens[x] > kv_lens[y]; });
  for (int j = 0; j < batch; ++j) {
    hs[j] = kv_lens[order[j]];
    hs[batch + j] = seq_ids ? seq_ids[order[j]] : order[j];
  }
  const size_t bytes = sizeof(int32_t) * batch * 3;
  HIP_OR_RETURN(hipMemcpyAsync(ds, hs, bytes, hipMemcpyHostToDevice, h->stream));
  HIP_OR_RETURN(hipEventRecord(h->ring_ev[slot], h->stream));
  h->ring_used[slot] = true;
  *d_lens = ds;
  *d_seq = ds + batch;
  *d_rows = ds + 2 * (size_t)batch;
  return 0;
}

// Rows count as appended only while they extend the unbroken prefix [0, filled) of their
// (layer, sequence): rows written behind a gap are stored, but attention never takes the unwritten
// (or, after a reset, stale) rows of the gap for appended ones.
void note_rows_written(mi355_attn* h, int layer, int seq, int pos, int n) {
  int32_t& f = h->filled[(size_t)layer * h->cfg.max_seqs + seq];
  if (pos <= f) f = std::max(f, pos + n);
}

int check_layers(const mi355_attn* h, int layer_begin, int n_layers, char** error_msg) {
  if (layer_begin < 0 || n_layers < 1 || layer_begin + n_layers > h->cfg.num_layers)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "layers [%d, %d) outside [0, %d)", layer_begin,
                layer_begin + n_layers, h->cfg.num_layers);
  return 0;
}

void fill_decode_common(const mi355_attn* h, DecodeLaunch* l) {
  DecodeArgs& a = l->args;
  a.cache = h->cache;
  a.scales = h->scales;
  a.plane_bytes = h->geom.plane_bytes;
  a.hkv = h->geom.hkv;
  a.max_seqs = h->geom.max_seqs;
  a.hq = h->cfg.num_q_heads;
  a.group = h->cfg.num_q_heads / h->cfg.num_kv_heads;
  a.hkv_inverse = h->geom.hkv > 1 ? (uint32_t)(((1ull << 32) + h->geom.hkv - 1) / h->geom.hkv) : 0;
  a.scale = h->cfg.scale;
  a.softcap = h->cfg.softcap;
  l->esize = h->geom.esize;
  l->tables.layer_window = h->d_window;
}

// The windows of layers layer_begin .. layer_begin + n_layers - 1 and their partition sizes into the launch (reads
// max_kv_len, num_splits and align), unless there are too many layers or different windows: then the kernels read the table in
// memory.
void fill_inline_windows(const mi355_attn* h, DecodeLaunch* l) {
  if (l->n_layers > kInlineLayers) return;
  auto& t = l->work.layers;
  int windows = 0;
  for (int i = 0; i < l->n_layers; ++i) {
    const int window = h->window[l->args.layer_begin + i];
    int w = 0;
    while (w < windows && t.window[w] != window) ++w;
    if (w == windows) {
      if (windows == kDecodeWindows) return;
      t.window[w] = window;
      t.per[w] = decode_partition_tokens(l->max_kv_len, window, l->args.num_splits, l->args.align);
      ++windows;
    }
    t.code[i >> 4] |= (uint32_t)w << (2 * (i & 15));
  }
  l->inline_layers = true;
}

// Raw projections of the one new token of every sequence (mi355_attn_decode_step): the decode kernel runs the
// step before attention itself.
struct NewRows {
  const void* k;
  const void* v;
};

// The partitions of a decode launch by rule. `heads`: layers x sequences x KV heads; `block`: tokens a wave loads at a time.
//
// While every block of every sequence can have a wave of its own and every partition a compute unit, latency is all there
// is: one partition of up to eight blocks (two for each of four waves; nothing to merge), else partitions of up to four
// blocks (a wave each), so many that the merge still has its rows in one trip (32), or two blocks and up to 256 partitions
// where the context needs more. One layer's step, 4 heads on 1, fp16, us, before this rule (64-token partitions, one up to
// 512 tokens) / now: 300 tokens 11.3 / 8.1, 520 9.0 / 8.4, 1,152 10.6 / 8.8 (window 512: 9.2 / 7.8), 4,096 12.3 / 10.0,
// 8,000 14.5 / 10.8; 8 sequences, one partition / a block each: 220 tokens 8.5 / 10.7, 380 11.3 / 10.9. Five blocks a
// partition of a 16-bit cache are still better than more workgroups where there are three to eight partitions (16 sequences
// of 1,200, 8 on 2: 11.6 against 12.4, 40 of 900, 4 on 1, 11.2 against 11.9; with 16 partitions 12.7 against 12.3).
//
// Larger launches: about 1,024 workgroups, in at most 64 partitions a sequence (one or two KV heads have fewer workgroups
// then), partitions of whole 64 tokens (4 layers x 15 float32 sequences of 3,170: 53 us in partitions of 176 tokens, 39 of
// 192), and one for contexts of up to 512 tokens (64 sequences of 256 / 512 tokens, Hq8/Hkv2: 9.7 / 15.4 us against 11.0 /
// 16.1 split and merged, 256 sequences 26.9 / 46.3 against 32.4 / 51.8). Half as many workgroups would make decode steps of
// equal lengths 4 to 7 % faster (64 sequences of 2,000, 8 on 2, fp16 48.3 against 51.9 us; decode itself 43.5 / 45.6, over an
// int8 cache 1 % slower, in the mean of 34 shapes as fast), but would lose precision: probabilities enter P.V as halves
// relative to the maximum of a wave's keys, so the heaviest key of each wave is exact, and with half the waves the error
// against 64 bits grows (30 layers x 4,096 2.67e-4 to 2.73e-4, 32 int8 sequences 3.40e-4 to 3.44e-4, over 12 seeds each,
// whose spread is 1e-6).
//
// Over a float32 cache a block's 128 matrix instructions of 32 cycles bound a wave: up to one workgroup a compute unit, of
// four waves, where that still cuts every sequence in two (in 1024 single waves / so, decode and decode step: 20 of 3,000,
// 4 on 1, 26.0 / 24.9 and 35.6 / 27.4, 40 of up to 1,120, 8 on 2, 28.1 / 26.6 and 41.2 / 30.5, 9 of up to 5,000, 4 on 1, 16.9 /
// 13.9 and 21.8 / 16.4). Several layers of unequal lengths in one call are better in 1024 (4 layers x 15 of up to 3,170: 39
// against 43.6).
struct DecodeSplits { int count, align; };
DecodeSplits choose_decode_splits(int max_len, int min_len, int widest, int narrowest, int n_layers, int heads, int block) {
  const int blocks = (decode_span(max_len, widest, block) + block - 1) / block;
  if (heads <= kLatencyWorkgroups) {
    if (blocks <= 8) return {1, block};
    const int few = std::min({32, blocks, kLatencyWorkgroups / heads});
    if (blocks <= (block == 32 && few >= 3 && few <= 8 ? 5 : 4) * few) return {few, block};
    const int many = std::min((blocks + 1) / 2, kLatencyWorkgroups / heads);
    if (many > 32 && blocks <= 4 * many) return {many, block};
  }
  if (max_len <= 512) return {1, kTokenAlign};
  const int most = decode_span(max_len, widest, 1), least = decode_span(min_len, narrowest, 1);
  const bool unequal = least * 4 < most * 3;
  if (block == 16 && heads <= kLatencyWorkgroups / 2 && !(unequal && n_layers > 1)) return {kLatencyWorkgroups / heads, kTokenAlign};
  return {std::max(1, std::min({(1024 + heads - 1) / heads, (max_len + 63) / 64, 64})), kTokenAlign};
}

// What a decode launch looks like: its partitions, those of them that hold anything, and the partial results they leave.
struct DecodeShape {
  const int32_t* window;  // of its layers
  int n_layers, batch;
  int rule_batch;         // as in DecodeLaunch
  int hq, hkv, esize;
  int max_len, min_len;
};
struct DecodePlan {
  int num_splits, align;
  int asked;              // partitions before those that hold nothing are left out
  int widest;             // window of its layers, 0: a layer without one
  size_t rows;            // partial results (0: one partition)
  bool merges_itself;
};
// num_splits: 0 by rule, then so many that `most_rows` hold their results (at least one).
DecodePlan plan_decode(const DecodeShape& s, int num_splits, size_t most_rows) {
  DecodePlan p{num_splits, kTokenAlign, num_splits, s.window[0], 0, false};
  int narrowest = p.widest;
  for (int l = 1; l < s.n_layers; ++l) {
    const int w = s.window[l];
    if (w == 0 || (p.widest > 0 && w > p.widest)) p.widest = w;
    if (w > 0 && (narrowest == 0 || w < narrowest)) narrowest = w;
  }
  const size_t heads = (size_t)s.n_layers * s.batch * s.hq;
  if (num_splits == 0) {
    const DecodeSplits splits = choose_decode_splits(s.max_len, s.min_len, p.widest, narrowest, s.n_layers,
                                                     s.n_layers * s.rule_batch * s.hkv, decode_block_tokens(s.esize));
    p.align = splits.align;
    p.asked = std::max(1, (int)std::min((size_t)splits.count, most_rows / heads));
  }
  // Partitions are rounded up, so fewer may cover the context than were asked for (4,096 tokens in 18: sixteen of 256): the
  // launch has no workgroups for the others. (Their size stays what it is: any count in between gives the same.)
  int used = 1;
  for (int l = 0; l < s.n_layers; ++l) {
    if (l > 0 && s.window[l] == s.window[l - 1]) continue;
    const int per = decode_partition_tokens(s.max_len, s.window[l], p.asked, p.align);
    used = std::max(used, (decode_span(s.max_len, s.window[l], p.align) + per - 1) / per);
  }
  p.num_splits = used;
  p.rows = used > 1 ? heads * used : 0;
  p.merges_itself = decode_merges_itself(s.n_layers, s.rule_batch, s.hkv, used);
  return p;
}

// no_alloc: the call may not allocate (mi355_attn_decode_noalloc): device pointers only, and partials
// that do not fit the handle's fixed room go to this GPU's `scratch` instead of the handle's workspace.
// new_rows: q holds raw query projections and the new token's key / value rows come with the call
// (its row, kv_lens[b] - 1, need not have been appended).
// The batch a launch is a part of (mi355_attn_decode_step cuts large batches into several launches): the launch rules
// then look at the whole batch, so that every part runs as the same sequences would in one launch of all of them,
// partitions and waves included, and the results are the same bits.
struct WholeBatch { int batch, max_len, min_len; };

int decode_impl(mi355_attn* h, int layer_begin, int n_layers, const int32_t* seq_ids, const int32_t* kv_lens,
                int batch, const void* q, void* out, int num_splits, char** error_msg, bool no_alloc = false,
                const NewRows* new_rows = nullptr, const WholeBatch* whole = nullptr) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (new_rows) {
    if (!new_rows->k || !new_rows->v) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null k or v");
    if (batch > kInlineItems)  // (mi355_attn_decode_step cuts larger batches into launches of this size)
      return fail(error_msg, MI355_ATTN_INTERNAL, "a fused decode step launch holds up to %d sequences (got %d)",
                  kInlineItems, batch);
  }
  if (no_alloc && h->cfg.host_io)
    return fail(error_msg, MI355_ATTN_FAILED_PRECONDITION,
                "mi355_attn_decode_noalloc needs device pointers (the handle was created with host_io = 1, "
                "whose staging buffers are allocated on demand)");
  if (int rc = check_layers(h, layer_begin, n_layers, error_msg)) return rc;
  if (!kv_lens || !q || !out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null kv_lens, q or out");
  if (batch < 1 || batch > h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "batch %d outside [1, max_seqs=%d]", batch,
                h->cfg.max_seqs);
  if (num_splits < 0 || num_splits > kMaxSplits)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "num_splits %d outside [0, %d]", num_splits, kMaxSplits);
  if (batch > 65535) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "batch %d exceeds the launch grid (65535)", batch);
  if (!decode_supported(h->cfg.kv_dtype, h->cfg.io_dtype, h->cfg.head_dim))
    return fail(error_msg, MI355_ATTN_UNIMPLEMENTED, "decode: unsupported kv/io dtype pair %d/%d",
                h->cfg.kv_dtype, h->cfg.io_dtype);
  int max_len = 0, min_len = INT32_MAX;
  for (int b = 0; b < batch; ++b) {
    const int seq = seq_ids ? seq_ids[b] : b;
    if (seq < 0 || seq >= h->cfg.max_seqs)
      return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq_ids[%d]=%d outside [0, %d)", b, seq,
                  h->cfg.max_seqs);
    const int len = kv_lens[b];
    if (len < 1 || len > h->cfg.max_tokens)
      return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "kv_lens[%d]=%d outside [1, max_tokens=%d]", b, len,
                  h->cfg.max_tokens);
    for (int l = layer_begin; l < layer_begin + n_layers; ++l)
      if (len - (new_rows ? 1 : 0) > h->filled[(size_t)l * h->cfg.max_seqs + seq])
        return fail(error_msg, MI355_ATTN_OUT_OF_RANGE,
                    "kv_lens[%d]=%d but only %d rows of layer %d, sequence %d were appended", b, len,
                    h->filled[(size_t)l * h->cfg.max_seqs + seq], l, seq);
    if (new_rows)  // every sequence gets one new row: the same sequence twice would write two
      for (int c = 0; c < b; ++c)
        if ((seq_ids ? seq_ids[c] : c) == seq)
          return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq_ids[%d] and seq_ids[%d] name the same sequence %d", c,
                      b, seq);
    max_len = std::max(max_len, len);
    min_len = std::min(min_len, len);
  }
  HIP_OR_RETURN(hipSetDevice(h->device));
  const int items = n_layers * batch;
  if (whole) {
    max_len = whole->max_len;
    min_len = whole->min_len;
  }
  // no_alloc: the library's own choice of partitions is trimmed to the workspace; an explicit count is an error
  const size_t asked = (size_t)items * h->cfg.num_q_heads * num_splits;
  if (no_alloc && num_splits > 1 && asked > kNoAllocSlots)
    return fail(error_msg, MI355_ATTN_RESOURCE_EXHAUSTED,
                "mi355_attn_decode_noalloc: %d layers x %d sequences x %d query heads x %d partitions = %zu partial "
                "results, the fixed workspace holds %zu (pass fewer partitions, or 0 to let the library choose)",
                n_layers, batch, h->cfg.num_q_heads, num_splits, asked, kNoAllocSlots);
  const DecodeShape shape{h->window.data() + layer_begin, n_layers, batch, whole ? whole->batch : batch, h->cfg.num_q_heads,
                          h->cfg.num_kv_heads, h->geom.esize, max_len, min_len};
  const DecodePlan plan = plan_decode(shape, num_splits, no_alloc ? kNoAllocSlots : SIZE_MAX);
  num_splits = plan.num_splits;
  // The partials: in the handle's fixed room where they fit it, so that a call of up to a workgroup a compute unit neither
  // allocates nor depends on an earlier call, recorded or not; larger ones in the workspace of the handle, or (no_alloc) in
  // this GPU's `scratch`.
  const bool in_scratch = no_alloc && plan.rows > kFixedRows;
  if (!no_alloc && plan.rows > kFixedRows)
    if (int rc = ensure_workspace(h, plan.rows, error_msg)) return rc;
  DecodeLaunch launch;
  DecodeArgs& a = launch.args;
  fill_decode_common(h, &launch);
  if (plan.rows <= kFixedRows) {
    a.ws_acc = h->d_parts;
    a.ws_ml = partials_ml(h, a.ws_acc, kFixedRows);
  } else if (in_scratch) {
    a.ws_acc = g_scratch_ptr[h->device];
    a.ws_ml = a.ws_acc + kNoAllocSlots * kNoAllocHeadDim;
  } else {
    a.ws_acc = h->ws;
    a.ws_ml = partials_ml(h, h->ws, h->ws_rows);
  }
  const size_t io_bytes = (size_t)items * h->cfg.num_q_heads * h->cfg.head_dim * io_size(h);
  const void* dq = nullptr;
  void* dout = nullptr;
  if (int rc = stage_in(h, 0, q, io_bytes, &dq, error_msg)) return rc;
  if (new_rows) {
    const size_t kv_bytes = (size_t)batch * h->cfg.num_kv_heads * h->cfg.head_dim * io_size(h);
    if (int rc = stage_in(h, 2, new_rows->k, kv_bytes, &launch.pre.k, error_msg)) return rc;
    if (int rc = stage_in(h, 3, new_rows->v, kv_bytes, &launch.pre.v, error_msg)) return rc;
    launch.fused = true;
    launch.pre.q = dq;
    const mi355_attn::LayerTransform& lt = h->transform[layer_begin];  // never set: a plain append
    launch.pre.constants = h->d_transform + (size_t)layer_begin * transform_floats(h->cfg.head_dim);
    launch.pre.rope = lt.rope;
    launch.pre.norm_q = lt.norm_q;
    launch.pre.norm_k = lt.norm_k;
    launch.pre.norm_v = lt.norm_v;
    launch.pre.q_scaled = lt.q_scaled;
    launch.pre.k_scaled = lt.k_scaled;
    launch.pre.eps = lt.eps;
    launch.pre.weight_offset = lt.weight_offset;
  }
  if (int rc = stage_out_begin(h, 1, out, io_bytes, &dout, error_msg)) return rc;
  if (batch <= kInlineItems) {
    launch.inline_items = true;
    // dispatch order: longest sequence first (rows keep their places in q and out)
    int order[kInlineItems];
    for (int b = 0; b < batch; ++b) order[b] = b;
    std::stable_sort(order, order + batch, [&](int x, int y) { return kv_lens[x] > kv_lens[y]; });
    for (int j = 0; j < batch; ++j) {
      const int b = order[j];
      launch.work.item[j] = DecodeItem{(uint32_t)kv_lens[b] | (uint32_t)b << kDecodeLenBits, seq_ids ? seq_ids[b] : b};
    }
  } else {
    // lengths and slots of a larger batch go up through the pinned ring: a copy and, when the ring wraps, a wait
    // on the host - neither can be part of a stream capture
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    HIP_OR_RETURN(hipStreamIsCapturing(h->stream, &capturing));
    if (capturing != hipStreamCaptureStatusNone)
      return fail(error_msg, MI355_ATTN_FAILED_PRECONDITION,
                  "decode of %d sequences while the stream is being captured: more than %d sequences per call need "
                  "an upload that a capture cannot hold (capture calls of up to %d sequences)",
                  batch, kInlineItems, kInlineItems);
    if (int rc = upload_items(h, seq_ids, kv_lens, batch, &launch.tables.kv_lens, &launch.tables.seq_ids, &launch.tables.rows, error_msg)) return rc;
  }
  a.q = dq;
  a.out = dout;
  a.layer_begin = layer_begin;
  a.batch = batch;
  launch.n_layers = n_layers;
  launch.max_kv_len = max_len;
  launch.min_kv_len = min_len;
  launch.widest_window = plan.widest;
  launch.rule_batch = shape.rule_batch;
  launch.rule_splits = plan.asked;
  a.num_splits = num_splits;
  a.align = plan.align;
  if (plan.merges_itself) a.tickets = h->d_tickets;
  fill_inline_windows(h, &launch);
  bool scratch_fence = false;
  if (in_scratch) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    HIP_OR_RETURN(hipStreamIsCapturing(h->stream, &capturing));
    scratch_fence = capturing == hipStreamCaptureStatusNone;
    if (scratch_fence && g_scratch_used[h->device] && g_scratch_stream[h->device] != h->stream)
      HIP_OR_RETURN(hipStreamWaitEvent(h->stream, g_scratch_done[h->device], 0));
  }
  HIP_OR_RETURN(launch_decode(launch, h->cfg.kv_dtype, h->cfg.io_dtype, h->tuning, h->stream,
                              h->timing ? h->ev0 : nullptr, h->timing ? h->ev1 : nullptr));
  if (scratch_fence) {
    HIP_OR_RETURN(hipEventRecord(g_scratch_done[h->device], h->stream));
    g_scratch_stream[h->device] = h->stream;
    g_scratch_used[h->device] = true;
  }
  h->timed = h->timing;
  if (new_rows)
    for (int b = 0; b < batch; ++b) note_rows_written(h, layer_begin, seq_ids ? seq_ids[b] : b, kv_lens[b] - 1, 1);
  return stage_out_end(h, 1, out, io_bytes, error_msg);
}

// The key split of a tiled launch, its workspace bounded where the rule decides.
constexpr size_t kSplitRowsMax = (size_t)256 << 10;  // 256 Ki rows = 258 MiB at head_dim 256
PrefillSplit split_of(const PrefillArgs& a, int option, int cus = 0) {
  const PrefillSplit split = plan_prefill_split(a, option, cus);
  return option < 0 && split.rows > kSplitRowsMax ? PrefillSplit{} : split;
}

// Whether a prefill call runs on the kernel for short calls (prefill_short.hip): option prefill_short, or by rule where
// no option asks for a particular one of the other kernels (a float32 cache has no other but the row-wise path, so the
// options that choose among the tiled kernels say nothing there).
bool short_prefill_takes(int n_layers, int n) { return n_layers <= kInlineLayers && n <= 65535; }
bool takes_short_prefill(const mi355_attn* h, int layer_begin, int n_layers, int q_pos0, int n) {
  if (h->rowwise_prefill || !short_prefill_takes(n_layers, n) || h->prefill_short == 0) return false;
  if (h->prefill_short == 1) return true;
  if (h->cfg.kv_dtype == MI355_ATTN_I8 && n < h->prefill_i8_min_rows) return false;
  if (h->cfg.kv_dtype != MI355_ATTN_F32 && (h->prefill_rows16 >= 0 || h->prefill_key_split >= 0 || h->prefill_workgroups > 0))
    return false;
  return prefill_short_wanted(h->cfg.kv_dtype, h->cfg.num_q_heads, h->cfg.num_kv_heads, h->window.data() + layer_begin,
                              n_layers, q_pos0, n);
}

int prefill_impl(mi355_attn* h, int layer_begin, int n_layers, int seq, int q_pos0, int n, const void* q,
                 void* out, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (int rc = check_layers(h, layer_begin, n_layers, error_msg)) return rc;
  if (!q || !out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null q or out");
  if (seq < 0 || seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  if (n < 1 || q_pos0 < 0 || (int64_t)q_pos0 + n > h->cfg.max_tokens)
    return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "rows [%d, %lld) outside [0, max_tokens=%d]", q_pos0,
                (long long)q_pos0 + n, h->cfg.max_tokens);
  for (int l = layer_begin; l < layer_begin + n_layers; ++l)
    if (q_pos0 + n > h->filled[(size_t)l * h->cfg.max_seqs + seq])
      return fail(error_msg, MI355_ATTN_OUT_OF_RANGE,
                  "prefill over rows [0, %d) but only %d rows of layer %d, sequence %d were appended",
                  q_pos0 + n, h->filled[(size_t)l * h->cfg.max_seqs + seq], l, seq);
  HIP_OR_RETURN(hipSetDevice(h->device));
  const size_t io_bytes = (size_t)n_layers * n * h->cfg.num_q_heads * h->cfg.head_dim * io_size(h);
  const void* dq = nullptr;
  void* dout = nullptr;
  if (int rc = stage_in(h, 0, q, io_bytes, &dq, error_msg)) return rc;
  if (int rc = stage_out_begin(h, 1, out, io_bytes, &dout, error_msg)) return rc;
  hipEvent_t e0 = h->timing ? h->ev0 : nullptr, e1 = h->timing ? h->ev1 : nullptr;
  // The short kernel first: it reads the planes as they are, and the room for its parts and its tickets are there from the
  // handle's creation, so nothing is allocated, neither now nor while a graph is recorded.
  if (takes_short_prefill(h, layer_begin, n_layers, q_pos0, n)) {
    PrefillShortArgs a{};
    a.q = dq;
    a.out = dout;
    a.cache = h->cache;
    a.scales = h->scales;
    a.ws_acc = h->d_parts;
    a.ws_ml = partials_ml(h, a.ws_acc, kFixedRows);
    a.tickets = h->d_tickets;
    a.plane_bytes = h->geom.plane_bytes;
    a.hkv = h->geom.hkv;
    a.max_seqs = h->geom.max_seqs;
    a.hq = h->cfg.num_q_heads;
    a.group = h->cfg.num_q_heads / h->cfg.num_kv_heads;
    a.layer_begin = layer_begin;
    a.seq = seq;
    a.q_pos0 = q_pos0;
    a.n = n;
    a.scale = h->cfg.scale;
    a.softcap = h->cfg.softcap;
    HIP_OR_RETURN(launch_prefill_short(a, h->window.data() + layer_begin, n_layers, h->cfg.kv_dtype, h->cfg.io_dtype, h->stream, e0, e1));
    h->timed = h->timing;
    return stage_out_end(h, 1, out, io_bytes, error_msg);
  }
  bool rowwise = !prefill_supported(h->cfg.kv_dtype, h->cfg.io_dtype, h->cfg.head_dim) || h->rowwise_prefill;
  // An int8 cache goes to the matrix cores through half planes staged per call (prefill_attn.hip): from a tile's
  // worth of rows on, in passes of as many layers as the staging area's limit holds.
  const bool i8 = h->cfg.kv_dtype == MI355_ATTN_I8;
  int layers_per_pass = n_layers;
  if (!rowwise && i8) {
    if (n < h->prefill_i8_min_rows) {
      rowwise = true;
    } else {
      const int64_t kStageMax = (int64_t)h->prefill_i8_stage_mib << 20;
      const int64_t per_layer = prefill_i8_stage_bytes(h->geom, 1, q_pos0 + n);
      layers_per_pass = (int)std::min<int64_t>(n_layers, std::max<int64_t>(1, kStageMax / per_layer));
      const size_t need = (size_t)per_layer * layers_per_pass;
      if (h->kv_stage_bytes < need) {
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        HIP_OR_RETURN(hipStreamIsCapturing(h->stream, &capturing));
        if (capturing != hipStreamCaptureStatusNone) {
          rowwise = true;  // (nothing can be allocated while a graph is recorded: the path that needs no room)
        } else {
          HIP_OR_RETURN(hipStreamSynchronize(h->stream));
          if (h->d_kv_stage) HIP_OR_RETURN(hipFree(h->d_kv_stage));
          h->d_kv_stage = nullptr;
          h->kv_stage_bytes = 0;
          HIP_OR_RETURN(hipMalloc(&h->d_kv_stage, need));
          h->kv_stage_bytes = need;
        }
      }
    }
  }
  const size_t layer_io_bytes = (size_t)n * h->cfg.num_q_heads * h->cfg.head_dim * io_size(h);
  for (int l0 = 0; !rowwise && l0 < n_layers; l0 += layers_per_pass) {
    const int nl = std::min(layers_per_pass, n_layers - l0);
    hipEvent_t pe0 = l0 == 0 ? e0 : nullptr, pe1 = l0 + nl == n_layers ? e1 : nullptr;
    PrefillArgs a{};
    a.q = static_cast<const uint8_t*>(dq) + l0 * layer_io_bytes;
    a.out = static_cast<uint8_t*>(dout) + l0 * layer_io_bytes;
    a.cache = h->cache;
    a.scales = h->scales;
    a.layer_window = h->d_window;
    a.sched = h->d_sched;
    a.geom = h->geom;
    a.hq = h->cfg.num_q_heads;
    a.group = h->cfg.num_q_heads / h->cfg.num_kv_heads;
    a.layer_begin = layer_begin + l0;
    a.n_layers = nl;
    a.seq = seq;
    a.q_pos0 = q_pos0;
    a.n = n;
    a.scale = h->cfg.scale;
    a.softcap = h->cfg.softcap;
    a.max_workgroups = h->prefill_workgroups;
    a.rows16 = h->prefill_rows16;
    a.host_window = h->window.data();
    if (h->cfg.io_dtype != h->cfg.kv_dtype && !(i8 && h->cfg.io_dtype == MI355_ATTN_F16)) {
      const size_t need = (size_t)nl * n * h->cfg.num_q_heads * h->cfg.head_dim * 2;
      if (h->q_stage_bytes < need) {
        HIP_OR_RETURN(hipStreamSynchronize(h->stream));
        if (h->d_q_stage) HIP_OR_RETURN(hipFree(h->d_q_stage));
        h->d_q_stage = nullptr;
        h->q_stage_bytes = 0;
        HIP_OR_RETURN(hipMalloc(&h->d_q_stage, need));
        h->q_stage_bytes = need;
      }
      a.q_stage = h->d_q_stage;
    }
    a.kv_stage = h->d_kv_stage;
    a.kv_stage_bytes = (int64_t)h->kv_stage_bytes;
    const PrefillSplit split = split_of(a, h->prefill_key_split);
    if (split.kchunk > 0) {
      if (split.rows > kSplitRowsMax)
        return fail(error_msg, MI355_ATTN_RESOURCE_EXHAUSTED, "prefill_key_split=%d needs %zu workspace rows (limit %zu)",
                    h->prefill_key_split, split.rows, kSplitRowsMax);
      if (h->pf_rows < split.rows) {
        HIP_OR_RETURN(hipStreamSynchronize(h->stream));
        if (h->d_pf_acc) HIP_OR_RETURN(hipFree(h->d_pf_acc));
        if (h->d_pf_ml) HIP_OR_RETURN(hipFree(h->d_pf_ml));
        h->d_pf_acc = h->d_pf_ml = nullptr;
        h->pf_rows = 0;
        HIP_OR_RETURN(hipMalloc(&h->d_pf_acc, split.rows * h->cfg.head_dim * sizeof(float)));
        HIP_OR_RETURN(hipMalloc(&h->d_pf_ml, split.rows * 2 * sizeof(float)));
        h->pf_rows = split.rows;
      }
      a.kchunk = split.kchunk;
      a.smax = split.smax;
      a.direct = split.direct;
      a.ws_acc = h->d_pf_acc;
      a.ws_ml = h->d_pf_ml;
    }
    HIP_OR_RETURN(launch_prefill(a, h->cfg.kv_dtype, h->cfg.io_dtype, &h->pf_plans, h->stream, pe0, pe1));
  }
  if (rowwise) {
    // Row-wise path (fp32 and int8 caches): every query row is one decode item
    // whose key range ends at its own position.
    if (!decode_supported(h->cfg.kv_dtype, h->cfg.io_dtype, h->cfg.head_dim))
      return fail(error_msg, MI355_ATTN_UNIMPLEMENTED, "prefill: unsupported kv/io dtype pair %d/%d",
                  h->cfg.kv_dtype, h->cfg.io_dtype);
    if (n > 65535)
      return fail(error_msg, MI355_ATTN_UNIMPLEMENTED,
                  "row-wise prefill (fp32 / int8 cache): %d rows exceed the launch grid (65535); call in chunks", n);
    if (h->d_items_cap < (size_t)n) {  // (never for an int8 or float32 cache: theirs is there from the start)
      hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
      HIP_OR_RETURN(hipStreamIsCapturing(h->stream, &capturing));
      if (capturing != hipStreamCaptureStatusNone)
        return fail(error_msg, MI355_ATTN_FAILED_PRECONDITION,
                    "row-wise prefill needs its item list allocated, which cannot happen while the stream is being "
                    "captured: run one row-wise prefill before the capture");
      HIP_OR_RETURN(hipStreamSynchronize(h->stream));
      if (h->d_items) HIP_OR_RETURN(hipFree(h->d_items));
      h->d_items = nullptr;
      h->d_items_cap = 0;
      HIP_OR_RETURN(hipMalloc(&h->d_items, sizeof(int32_t) * 2 * (size_t)h->cfg.max_tokens));
      h->d_items_cap = h->cfg.max_tokens;
    }
    int32_t* lens = h->d_items;
    int32_t* seqs = h->d_items + h->d_items_cap;
    hipLaunchKernelGGL(iota_items_kernel, dim3((n + 255) / 256), dim3(256), 0, h->stream, lens, seqs, n, q_pos0,
                       seq);
    HIP_OR_RETURN(hipGetLastError());
    DecodeLaunch launch;
    DecodeArgs& a = launch.args;
    fill_decode_common(h, &launch);
    a.q = dq;
    a.out = dout;
    launch.tables.kv_lens = lens;
    launch.tables.seq_ids = seqs;
    a.layer_begin = layer_begin;
    a.batch = n;
    a.num_splits = 1;
    a.align = kTokenAlign;
    launch.n_layers = n_layers;
    launch.max_kv_len = q_pos0 + n;
    launch.rule_batch = n;
    fill_inline_windows(h, &launch);
    HIP_OR_RETURN(launch_decode(launch, h->cfg.kv_dtype, h->cfg.io_dtype, h->tuning, h->stream, e0, e1));
  }
  h->timed = h->timing;
  return stage_out_end(h, 1, out, io_bytes, error_msg);
}

}  // namespace

extern "C" {

const char* mi355_attn_version(void) { return "mi355_attn 0.1 (gfx950)"; }

int mi355_attn_create(const mi355_attn_config* c, mi355_attn** out, char** error_msg) {
  if (out) *out = nullptr;
  if (!c || !out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null config or out");
  if (c->struct_size != sizeof(mi355_attn_config))
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "config.struct_size %u != %zu", c->struct_size,
                sizeof(mi355_attn_config));
  if (c->num_layers < 1 || c->num_q_heads < 1 || c->num_kv_heads < 1 || c->max_tokens < 1 || c->max_seqs < 1)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "layers, heads, max_tokens and max_seqs must be >= 1");
  if (c->num_q_heads % c->num_kv_heads)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "num_q_heads %d is not a multiple of num_kv_heads %d",
                c->num_q_heads, c->num_kv_heads);
  if (c->num_q_heads / c->num_kv_heads > kMaxGroup)
    return fail(error_msg, MI355_ATTN_UNIMPLEMENTED, "more than %d query heads per KV head", kMaxGroup);
  if (c->head_dim != 256)
    return fail(error_msg, MI355_ATTN_UNIMPLEMENTED, "head_dim %d (only 256 is built)", c->head_dim);
  if (c->kv_dtype < MI355_ATTN_F32 || c->kv_dtype > MI355_ATTN_I8 || c->io_dtype < MI355_ATTN_F32 ||
      c->io_dtype > MI355_ATTN_BF16)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "bad kv_dtype %d or io_dtype %d", c->kv_dtype,
                c->io_dtype);
  if (!decode_supported(c->kv_dtype, c->io_dtype, c->head_dim))
    return fail(error_msg, MI355_ATTN_UNIMPLEMENTED,
                "kv_dtype %d with io_dtype %d (supported: equal f32 / f16 / bf16; f16 or bf16 cache with f32 io; int8 "
                "cache with f16, bf16 or f32 io)",
                c->kv_dtype, c->io_dtype);
  if (c->softcap < 0.f || c->scale < 0.f)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "scale and softcap must be >= 0");
  if (c->layer_window)
    for (int l = 0; l < c->num_layers; ++l)
      if (c->layer_window[l] < 0)
        return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "layer_window[%d] < 0", l);

  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(error_msg, MI355_ATTN_UNAVAILABLE, "no HIP device");
  if (c->device < 0 || c->device >= ndev)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "device %d outside [0, %d)", c->device, ndev);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, c->device) != hipSuccess)
    return fail(error_msg, MI355_ATTN_UNAVAILABLE, "cannot query device %d", c->device);
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(error_msg, MI355_ATTN_UNAVAILABLE, "device %d is %s; this library is built for gfx950 only",
                c->device, prop.gcnArchName);

  mi355_attn* h = new (std::nothrow) mi355_attn();
  if (!h) return fail(error_msg, MI355_ATTN_RESOURCE_EXHAUSTED, "out of host memory");
  h->cfg = *c;
  h->cfg.layer_window = nullptr;
  if (h->cfg.scale == 0.f) h->cfg.scale = 1.0f / sqrtf((float)c->head_dim);
  h->device = c->device;
  h->window.assign(c->num_layers, 0);
  if (c->layer_window) h->window.assign(c->layer_window, c->layer_window + c->num_layers);
  h->filled.assign((size_t)c->num_layers * c->max_seqs, 0);
  h->geom.num_layers = c->num_layers;
  h->geom.max_seqs = c->max_seqs;
  h->geom.hkv = c->num_kv_heads;
  h->geom.head_dim = c->head_dim;
  h->geom.cap = (int32_t)round_up64(c->max_tokens, kTokenAlign);
  h->geom.esize = dtype_size(c->kv_dtype);
  h->geom.plane_bytes = (int64_t)h->geom.cap * c->head_dim * h->geom.esize;
  // the kernels address a plane through a 32-bit buffer descriptor and 32-bit block offsets
  if (h->geom.plane_bytes > (int64_t)INT32_MAX) {
    const long long pb = (long long)h->geom.plane_bytes;
    delete h;
    return fail(error_msg, MI355_ATTN_UNIMPLEMENTED, "max_tokens %d: one plane would hold %lld bytes (limit 2 GiB - 1)",
                c->max_tokens, pb);
  }
  h->cache_bytes = (uint64_t)h->geom.plane_bytes * 2 * c->num_kv_heads * c->max_seqs * c->num_layers;

  auto bail = [&](int code, const char* what, hipError_t e) {
    int rc = fail(error_msg, code, "%s: %s", what, hipGetErrorString(e));
    mi355_attn_destroy(h);
    return rc;
  };
  hipError_t e;
  if ((e = hipSetDevice(h->device)) != hipSuccess) return bail(MI355_ATTN_UNAVAILABLE, "hipSetDevice", e);
  if (h->device >= kMaxDevices) {
    int rc = fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "device %d: at most %d devices", h->device, kMaxDevices);
    mi355_attn_destroy(h);
    return rc;
  }
  if (!g_scratch_ptr[h->device]) {  // once per GPU, with that GPU current
    float* p = nullptr;
    if ((e = hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch))) != hipSuccess || !p)
      return bail(MI355_ATTN_INTERNAL, "hipGetSymbolAddress(scratch)", e);
    g_scratch_ptr[h->device] = p;
  }
  if (!g_scratch_done[h->device] &&
      (e = hipEventCreateWithFlags(&g_scratch_done[h->device], hipEventDisableTiming)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "hipEventCreate", e);
  if (c->own_stream) {
    if ((e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking)) != hipSuccess)
      return bail(MI355_ATTN_INTERNAL, "hipStreamCreate", e);
    h->own_stream = true;
  } else {
    h->stream = static_cast<hipStream_t>(c->stream);  // nullptr is the HIP default stream
  }
  // Behind the cache, in one allocation (another of its own took creating and freeing a handle 0.35 ms longer): the fixed room
  // for partials, 4 MiB. Here and not on first use: a call that is recorded into a graph then runs as it does eagerly.
  const uint64_t parts_at = (h->cache_bytes + 255) / 256 * 256;
  if ((e = hipMalloc(&h->cache, parts_at + partials_bytes(h, kFixedRows))) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "KV cache allocation", e);
  h->d_parts = reinterpret_cast<float*>(h->cache + parts_at);
  // Rows that were never written must read as finite numbers: a masked key
  // still enters P.V with probability 0, and 0 * NaN would poison the output.
  if ((e = hipMemsetAsync(h->cache, 0, h->cache_bytes, h->stream)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "KV cache clear", e);
  if (c->kv_dtype == MI355_ATTN_I8) {
    const size_t nsc = (size_t)c->num_layers * c->max_seqs * 2 * c->num_kv_heads * c->head_dim;
    if ((e = hipMalloc(&h->scales, nsc * sizeof(float))) != hipSuccess)
      return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "scale allocation", e);
    if ((e = hipMemsetAsync(h->scales, 0, nsc * sizeof(float), h->stream)) != hipSuccess)
      return bail(MI355_ATTN_INTERNAL, "scale clear", e);
  }
  if ((e = hipMalloc(&h->d_window, sizeof(int32_t) * c->num_layers)) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "window table", e);
  if ((e = hipMemcpyAsync(h->d_window, h->window.data(), sizeof(int32_t) * c->num_layers, hipMemcpyHostToDevice,
                          h->stream)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "window upload", e);
  if ((e = hipMalloc(&h->d_sched, sizeof(int32_t) * (kSchedInts + kDecodeTickets))) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "queue counters and tickets", e);
  h->d_tickets = reinterpret_cast<uint32_t*>(h->d_sched + kSchedInts);
  static_assert(kShortPartSlots <= kDecodeTickets, "short prefill calls and decode use the same tickets");
  h->transform.assign(c->num_layers, mi355_attn::LayerTransform{});
  const size_t transform_bytes = sizeof(float) * (size_t)c->num_layers * transform_floats(c->head_dim);
  if ((e = hipMalloc(&h->d_transform, transform_bytes)) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "layer transform constants", e);
  if ((e = hipMemsetAsync(h->d_transform, 0, transform_bytes, h->stream)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "layer transform clear", e);
  if ((e = hipMemsetAsync(h->d_sched, 0, sizeof(int32_t) * (kSchedInts + kDecodeTickets), h->stream)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "queue counters and tickets clear", e);
  if (c->kv_dtype == MI355_ATTN_I8 || c->kv_dtype == MI355_ATTN_F32) {
    // the row-wise prefill path's item list (these caches may take that path inside a captured graph, where nothing
    // can be allocated)
    if ((e = hipMalloc(&h->d_items, sizeof(int32_t) * 2 * (size_t)c->max_tokens)) != hipSuccess)
      return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "row-wise prefill items", e);
    h->d_items_cap = c->max_tokens;
  }
  h->ring_slot_ints = 3 * c->max_seqs;
  if ((e = hipHostMalloc(&h->h_ring, sizeof(int32_t) * h->ring_slot_ints * kRingSlots)) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "pinned ring", e);
  if ((e = hipMalloc(&h->d_ring, sizeof(int32_t) * h->ring_slot_ints * kRingSlots)) != hipSuccess)
    return bail(MI355_ATTN_RESOURCE_EXHAUSTED, "device ring", e);
  for (int i = 0; i < kRingSlots; ++i)
    if ((e = hipEventCreateWithFlags(&h->ring_ev[i], hipEventDisableTiming)) != hipSuccess)
      return bail(MI355_ATTN_INTERNAL, "hipEventCreate", e);
  if ((e = hipEventCreate(&h->ev0)) != hipSuccess || (e = hipEventCreate(&h->ev1)) != hipSuccess)
    return bail(MI355_ATTN_INTERNAL, "hipEventCreate", e);
  if ((e = hipStreamSynchronize(h->stream)) != hipSuccess) return bail(MI355_ATTN_INTERNAL, "create sync", e);
  *out = h;
  return MI355_ATTN_OK;
}

void mi355_attn_destroy(mi355_attn* h) {
  if (!h) return;
  (void)hipSetDevice(h->device);
  (void)hipStreamSynchronize(h->stream);
  if (h->cache) (void)hipFree(h->cache);
  if (h->scales) (void)hipFree(h->scales);
  if (h->d_window) (void)hipFree(h->d_window);
  if (h->d_sched) (void)hipFree(h->d_sched);
  free_prefill_plans(&h->pf_plans);
  if (h->d_pf_acc) (void)hipFree(h->d_pf_acc);
  if (h->d_pf_ml) (void)hipFree(h->d_pf_ml);
  if (h->d_q_stage) (void)hipFree(h->d_q_stage);
  if (h->d_kv_stage) (void)hipFree(h->d_kv_stage);
  if (h->d_transform) (void)hipFree(h->d_transform);
  if (h->ws) (void)hipFree(h->ws);
  for (float* ws : h->ws_kept) (void)hipFree(ws);
  if (h->d_ring) (void)hipFree(h->d_ring);
  if (h->h_ring) (void)hipHostFree(h->h_ring);
  if (h->d_items) (void)hipFree(h->d_items);
  for (auto& s : h->stage)
    if (s) (void)hipFree(s);
  for (auto& ev : h->ring_ev)
    if (ev) (void)hipEventDestroy(ev);
  if (h->ev0) (void)hipEventDestroy(h->ev0);
  if (h->ev1) (void)hipEventDestroy(h->ev1);
  if (h->device < kMaxDevices && g_scratch_stream[h->device] == h->stream && g_scratch_used[h->device]) {
    // (the stream was synchronised above: its last use of the shared workspace is over, and a later stream
    // that happens to get the same address must not be taken for it)
    g_scratch_used[h->device] = false;
    g_scratch_stream[h->device] = nullptr;
  }
  if (h->own_stream && h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

int mi355_attn_kv_append(mi355_attn* h, int32_t layer, int32_t seq, int32_t pos, int32_t n, const void* k,
                         const void* v, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (seq < 0 || seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  if (n < 0 || pos < 0 || (int64_t)pos + n > h->cfg.max_tokens)
    return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "rows [%d, %lld) outside [0, max_tokens=%d]", pos,
                (long long)pos + n, h->cfg.max_tokens);
  if (n == 0) return MI355_ATTN_OK;
  if (!k || !v) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null k or v");
  HIP_OR_RETURN(hipSetDevice(h->device));
  const size_t bytes = (size_t)n * h->cfg.num_kv_heads * h->cfg.head_dim * kv_size(h);
  const void *dk = nullptr, *dv = nullptr;
  if (int rc = stage_in(h, 2, k, bytes, &dk, error_msg)) return rc;
  if (int rc = stage_in(h, 3, v, bytes, &dv, error_msg)) return rc;
  KvCopyArgs a{};
  a.cache = h->cache;
  a.geom = h->geom;
  a.v_half = h->cfg.kv_dtype == MI355_ATTN_BF16;
  a.layer = layer;
  a.seq = seq;
  a.pos = pos;
  a.n = n;
  a.k = const_cast<void*>(dk);
  a.v = const_cast<void*>(dv);
  HIP_OR_RETURN(launch_kv_append(a, h->stream));
  if (h->cfg.host_io) HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  note_rows_written(h, layer, seq, pos, n);
  return MI355_ATTN_OK;
}

int mi355_attn_kv_set_scales(mi355_attn* h, int32_t layer, int32_t seq, const float* k_scale,
                             const float* v_scale, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (h->cfg.kv_dtype != MI355_ATTN_I8)
    return fail(error_msg, MI355_ATTN_FAILED_PRECONDITION, "scales apply to an int8 cache only");
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (seq < 0 || seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  if (!k_scale || !v_scale) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null scales");
  HIP_OR_RETURN(hipSetDevice(h->device));
  const size_t n = (size_t)h->cfg.num_kv_heads * h->cfg.head_dim;
  const hipMemcpyKind kind = h->cfg.host_io ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
  HIP_OR_RETURN(hipMemcpyAsync(h->scales + h->geom.scale_offset(layer, seq, 0, 0), k_scale, n * sizeof(float), kind,
                               h->stream));
  HIP_OR_RETURN(hipMemcpyAsync(h->scales + h->geom.scale_offset(layer, seq, 1, 0), v_scale, n * sizeof(float), kind,
                               h->stream));
  if (h->cfg.host_io) HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  return MI355_ATTN_OK;
}

int mi355_attn_set_layer_transform(mi355_attn* h, int32_t layer, const mi355_attn_layer_transform* t,
                                   char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (!t || t->struct_size != sizeof(mi355_attn_layer_transform))
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null transform or struct_size mismatch");
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (!(t->eps >= 0.f) || !std::isfinite(t->eps) || !std::isfinite(t->weight_offset))
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "eps %g must be finite and >= 0, weight_offset %g finite",
                (double)t->eps, (double)t->weight_offset);
  const int D = h->cfg.head_dim;
  if (t->rope_inv_freq)
    for (int d = 0; d < D / 2; ++d)
      if (!std::isfinite(t->rope_inv_freq[d]))
        return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "rope_inv_freq[%d] is not finite", d);
  HIP_OR_RETURN(hipSetDevice(h->device));
  // the constants are host arrays whatever host_io says; copied before this call returns
  std::vector<float> row((size_t)transform_floats(D), 0.f);
  if (t->rope_inv_freq) memcpy(row.data(), t->rope_inv_freq, sizeof(float) * (D / 2));
  if (t->q_weight) memcpy(row.data() + D / 2, t->q_weight, sizeof(float) * D);
  if (t->k_weight) memcpy(row.data() + D / 2 + D, t->k_weight, sizeof(float) * D);
  HIP_OR_RETURN(hipStreamSynchronize(h->stream));  // earlier launches may still read the old constants
  HIP_OR_RETURN(hipMemcpy(h->d_transform + (size_t)layer * transform_floats(D), row.data(), sizeof(float) * row.size(),
                          hipMemcpyHostToDevice));
  mi355_attn::LayerTransform& lt = h->transform[layer];
  lt.set = true;
  lt.rope = t->rope_inv_freq != nullptr;
  lt.norm_q = t->norm_q != 0;
  lt.norm_k = t->norm_k != 0;
  lt.norm_v = t->norm_v != 0;
  lt.q_scaled = lt.norm_q && t->q_weight != nullptr;
  lt.k_scaled = lt.norm_k && t->k_weight != nullptr;
  lt.eps = t->eps;
  lt.weight_offset = t->weight_offset;
  return MI355_ATTN_OK;
}

int mi355_attn_pre_attention(mi355_attn* h, int32_t layer, int32_t seq, int32_t pos, int32_t n, const void* q,
                             const void* k, const void* v, void* q_out, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (seq < 0 || seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  if (n < 0 || pos < 0 || (int64_t)pos + n > h->cfg.max_tokens)
    return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "rows [%d, %lld) outside [0, max_tokens=%d]", pos,
                (long long)pos + n, h->cfg.max_tokens);
  if (n == 0) return MI355_ATTN_OK;
  if (!q || !k || !v || !q_out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null q, k, v or q_out");
  HIP_OR_RETURN(hipSetDevice(h->device));
  const size_t q_bytes = (size_t)n * h->cfg.num_q_heads * h->cfg.head_dim * io_size(h);
  const size_t kv_bytes = (size_t)n * h->cfg.num_kv_heads * h->cfg.head_dim * io_size(h);
  const void *dq = nullptr, *dk = nullptr, *dv = nullptr;
  void* dout = nullptr;
  if (int rc = stage_in(h, 0, q, q_bytes, &dq, error_msg)) return rc;
  if (int rc = stage_in(h, 2, k, kv_bytes, &dk, error_msg)) return rc;
  if (int rc = stage_in(h, 3, v, kv_bytes, &dv, error_msg)) return rc;
  if (int rc = stage_out_begin(h, 1, q_out, q_bytes, &dout, error_msg)) return rc;
  const mi355_attn::LayerTransform& lt = h->transform[layer];  // never set: a plain append
  PreAttentionArgs a{};
  a.q = dq;
  a.k = dk;
  a.v = dv;
  a.q_out = dout;
  a.cache = h->cache;
  a.scales = h->scales;
  a.constants = h->d_transform + (size_t)layer * transform_floats(h->cfg.head_dim);
  a.geom = h->geom;
  a.layer = layer;
  a.seq = seq;
  a.pos = pos;
  a.n = n;
  a.hq = h->cfg.num_q_heads;
  a.rope = lt.rope;
  a.norm_q = lt.norm_q;
  a.norm_k = lt.norm_k;
  a.norm_v = lt.norm_v;
  a.q_scaled = lt.q_scaled;
  a.k_scaled = lt.k_scaled;
  a.eps = lt.eps;
  a.weight_offset = lt.weight_offset;
  HIP_OR_RETURN(launch_pre_attention(a, h->cfg.kv_dtype, h->cfg.io_dtype, h->stream, h->timing ? h->ev0 : nullptr,
                                     h->timing ? h->ev1 : nullptr));
  h->timed = h->timing;
  note_rows_written(h, layer, seq, pos, n);
  return stage_out_end(h, 1, q_out, q_bytes, error_msg);
}

int mi355_attn_kv_read(mi355_attn* h, int32_t layer, int32_t seq, int32_t pos, int32_t n, void* k_out, void* v_out,
                       char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (seq < 0 || seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  if (n < 0 || pos < 0 || (int64_t)pos + n > h->cfg.max_tokens)
    return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "rows [%d, %lld) outside [0, max_tokens=%d]", pos,
                (long long)pos + n, h->cfg.max_tokens);
  if (n == 0) return MI355_ATTN_OK;
  if (!k_out || !v_out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null k_out or v_out");
  HIP_OR_RETURN(hipSetDevice(h->device));
  const size_t bytes = (size_t)n * h->cfg.num_kv_heads * h->cfg.head_dim * kv_size(h);
  void *dk = nullptr, *dv = nullptr;
  if (int rc = stage_out_begin(h, 2, k_out, bytes, &dk, error_msg)) return rc;
  if (int rc = stage_out_begin(h, 3, v_out, bytes, &dv, error_msg)) return rc;
  KvCopyArgs a{};
  a.cache = h->cache;
  a.geom = h->geom;
  a.v_half = h->cfg.kv_dtype == MI355_ATTN_BF16;
  a.layer = layer;
  a.seq = seq;
  a.pos = pos;
  a.n = n;
  a.k = dk;
  a.v = dv;
  HIP_OR_RETURN(launch_kv_read(a, h->stream));
  if (int rc = stage_out_end(h, 2, k_out, bytes, error_msg)) return rc;
  return stage_out_end(h, 3, v_out, bytes, error_msg);
}

int mi355_attn_prefill(mi355_attn* h, int32_t layer, int32_t seq, int32_t q_pos0, int32_t n, const void* q,
                       void* out, char** error_msg) {
  return prefill_impl(h, layer, 1, seq, q_pos0, n, q, out, error_msg);
}

int mi355_attn_prefill_layers(mi355_attn* h, int32_t layer_begin, int32_t n_layers, int32_t seq, int32_t q_pos0,
                              int32_t n, const void* q, void* out, char** error_msg) {
  return prefill_impl(h, layer_begin, n_layers, seq, q_pos0, n, q, out, error_msg);
}

int mi355_attn_decode(mi355_attn* h, int32_t layer, const int32_t* seq_ids, const int32_t* kv_lens, int32_t batch,
                      const void* q, void* out, int32_t num_splits, char** error_msg) {
  return decode_impl(h, layer, 1, seq_ids, kv_lens, batch, q, out, num_splits, error_msg);
}

int mi355_attn_decode_layers(mi355_attn* h, int32_t layer_begin, int32_t n_layers, const int32_t* seq_ids,
                             const int32_t* kv_lens, int32_t batch, const void* q, void* out, int32_t num_splits,
                             char** error_msg) {
  return decode_impl(h, layer_begin, n_layers, seq_ids, kv_lens, batch, q, out, num_splits, error_msg);
}

int mi355_attn_prefill_plan_probe(int32_t n_layers, int32_t n, int32_t q_pos0, int32_t num_q_heads, int32_t num_kv_heads,
                                  const int32_t* layer_window, int32_t workgroups, int32_t compute_units,
                                  int32_t* items_per_wg, int32_t* blocks_per_wg, int32_t* items_off_home) {
  return mi355::prefill_plan_probe(n_layers, n, q_pos0, num_q_heads, num_kv_heads, layer_window, workgroups, compute_units,
                                   items_per_wg, blocks_per_wg, items_off_home);
}

int mi355_attn_prefill_route_probe(int32_t kv_dtype, int32_t n_layers, int32_t n, int32_t q_pos0, int32_t num_q_heads,
                                   int32_t num_kv_heads, const int32_t* layer_window, int32_t compute_units, int32_t* parts) {
  if (kv_dtype < MI355_ATTN_F32 || kv_dtype > MI355_ATTN_I8 || n_layers < 1 || n < 1 || q_pos0 < 0 || num_kv_heads < 1 ||
      num_q_heads < num_kv_heads || num_q_heads % num_kv_heads || num_q_heads / num_kv_heads > kMaxGroup || !layer_window ||
      compute_units < 1)
    return -1;
  if (parts) *parts = 1;
  if (kv_dtype == MI355_ATTN_I8 && n < kI8MinRows) return MI355_ATTN_ROUTE_ROWWISE;
  if (short_prefill_takes(n_layers, n) &&
      prefill_short_wanted(kv_dtype, num_q_heads, num_kv_heads, layer_window, n_layers, q_pos0, n)) {
    if (parts) *parts = prefill_short_call_parts(kv_dtype, num_q_heads / num_kv_heads, num_kv_heads, layer_window, n_layers, q_pos0, n);
    return MI355_ATTN_ROUTE_SHORT;
  }
  if (kv_dtype == MI355_ATTN_F32) return MI355_ATTN_ROUTE_ROWWISE;
  PrefillArgs a{};
  a.n_layers = n_layers;
  a.n = n;
  a.q_pos0 = q_pos0;
  a.hq = num_q_heads;
  a.group = num_q_heads / num_kv_heads;
  a.geom.hkv = num_kv_heads;
  a.host_window = layer_window;
  a.rows16 = -1;
  const PrefillSplit split = split_of(a, -1, compute_units);
  if (parts) *parts = split.smax;
  if (split.direct) return MI355_ATTN_ROUTE_DIRECT16;
  a.kchunk = split.kchunk;
  return prefill_takes_plan(a, prefill_work_items(a), compute_units) ? MI355_ATTN_ROUTE_PLANNED16 : MI355_ATTN_ROUTE_TILED32;
}

int mi355_attn_decode_plan_probe(int32_t kv_dtype, int32_t n_layers, int32_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                                 const int32_t* layer_window, int32_t max_len, int32_t min_len, int32_t num_splits,
                                 int32_t* merged_in_launch, int32_t* rows, int32_t* fixed_rows) {
  if (kv_dtype < MI355_ATTN_F32 || kv_dtype > MI355_ATTN_I8 || n_layers < 1 || batch < 1 || batch > 65535 || num_kv_heads < 1 ||
      num_q_heads < num_kv_heads || num_q_heads % num_kv_heads || num_q_heads / num_kv_heads > kMaxGroup || !layer_window ||
      min_len < 1 || max_len < min_len || num_splits < 0 || num_splits > kMaxSplits)
    return -1;
  const DecodeShape shape{layer_window, n_layers, batch, batch, num_q_heads, num_kv_heads, dtype_size(kv_dtype), max_len, min_len};
  const DecodePlan plan = plan_decode(shape, num_splits, SIZE_MAX);
  if (merged_in_launch) *merged_in_launch = plan.merges_itself;
  if (rows) *rows = (int32_t)std::min<size_t>(plan.rows, INT32_MAX);
  if (fixed_rows) *fixed_rows = (int32_t)kFixedRows;
  return plan.num_splits;
}

int mi355_attn_decode_step(mi355_attn* h, int32_t layer, const int32_t* seq_ids, const int32_t* kv_lens, int32_t batch,
                           const void* q, const void* k, const void* v, void* out, int32_t num_splits,
                           char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (batch <= kInlineItems) {
    const NewRows rows{k, v};
    return decode_impl(h, layer, 1, seq_ids, kv_lens, batch, q, out, num_splits, error_msg, /*no_alloc=*/false, &rows);
  }
  // More sequences than one launch carries in its argument block: launches of kInlineItems sequences each, queued
  // back to back. Everything that can be refused is checked for the whole batch first, so that a call either
  // runs all of its launches or none.
  if (int rc = check_layers(h, layer, 1, error_msg)) return rc;
  if (!kv_lens || !q || !k || !v || !out) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null kv_lens, q, k, v or out");
  if (batch > h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "batch %d outside [1, max_seqs=%d]", batch, h->cfg.max_seqs);
  if (num_splits < 0 || num_splits > kMaxSplits)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "num_splits %d outside [0, %d]", num_splits, kMaxSplits);
  std::vector<int32_t> ids(batch);
  std::vector<char> named(h->cfg.max_seqs, 0);
  for (int b = 0; b < batch; ++b) {
    const int seq = seq_ids ? seq_ids[b] : b;
    if (seq < 0 || seq >= h->cfg.max_seqs)
      return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq_ids[%d]=%d outside [0, %d)", b, seq, h->cfg.max_seqs);
    if (named[seq]) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq_ids names sequence %d twice (entry %d)", seq, b);
    named[seq] = 1;
    ids[b] = seq;
    const int len = kv_lens[b];
    if (len < 1 || len > h->cfg.max_tokens)
      return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "kv_lens[%d]=%d outside [1, max_tokens=%d]", b, len, h->cfg.max_tokens);
    if (len - 1 > h->filled[(size_t)layer * h->cfg.max_seqs + seq])
      return fail(error_msg, MI355_ATTN_OUT_OF_RANGE, "kv_lens[%d]=%d but only %d rows of layer %d, sequence %d were appended",
                  b, len, h->filled[(size_t)layer * h->cfg.max_seqs + seq], layer, seq);
  }
  const size_t q_row = (size_t)h->cfg.num_q_heads * h->cfg.head_dim * io_size(h);
  const size_t kv_row = (size_t)h->cfg.num_kv_heads * h->cfg.head_dim * io_size(h);
  WholeBatch whole{batch, 0, INT32_MAX};
  for (int b = 0; b < batch; ++b) {
    whole.max_len = std::max(whole.max_len, kv_lens[b]);
    whole.min_len = std::min(whole.min_len, kv_lens[b]);
  }
  for (int b0 = 0; b0 < batch; b0 += kInlineItems) {
    const int nb = std::min<int>(kInlineItems, batch - b0);
    const NewRows rows{static_cast<const uint8_t*>(k) + b0 * kv_row, static_cast<const uint8_t*>(v) + b0 * kv_row};
    if (int rc = decode_impl(h, layer, 1, ids.data() + b0, kv_lens + b0, nb, static_cast<const uint8_t*>(q) + b0 * q_row,
                             static_cast<uint8_t*>(out) + b0 * q_row, num_splits, error_msg, /*no_alloc=*/false, &rows,
                             &whole))
      return rc;
  }
  return MI355_ATTN_OK;
}

int mi355_attn_decode_noalloc(mi355_attn* h, int32_t layer, const int32_t* seq_ids, const int32_t* kv_lens,
                              int32_t batch, const void* q, void* out, int32_t num_splits, char** error_msg) {
  static_assert(kNoAllocHeadDim == 256, "the workspace is laid out for the one head_dim the library builds");
  return decode_impl(h, layer, 1, seq_ids, kv_lens, batch, q, out, num_splits, error_msg, /*no_alloc=*/true);
}

int mi355_attn_stream_probe(mi355_attn* h, uint64_t offset, uint64_t bytes, int32_t workgroups, int32_t waves,
                            char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (workgroups < 1 || waves < 1 || waves > 16 || bytes < 1)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "workgroups >= 1, 1 <= waves <= 16 and bytes >= 1");
  HIP_OR_RETURN(hipSetDevice(h->device));
  hipError_t e = launch_stream_probe(h->cache, (int64_t)h->cache_bytes, (int64_t)offset, (int64_t)bytes, workgroups, waves,
                                     reinterpret_cast<uint32_t*>(h->d_sched) + kPrefillSchedInts, h->stream,
                                     h->timing ? h->ev0 : nullptr, h->timing ? h->ev1 : nullptr);
  if (e == hipErrorInvalidValue)
    return fail(error_msg, MI355_ATTN_OUT_OF_RANGE,
                "%llu bytes from offset %llu in %d x %d shares of whole 32 KiB pieces do not fit the cache (%llu bytes), or "
                "the offset is not a multiple of 16",
                (unsigned long long)bytes, (unsigned long long)offset, workgroups, waves, (unsigned long long)h->cache_bytes);
  HIP_OR_RETURN(e);
  h->timed = h->timing;
  return MI355_ATTN_OK;
}

int mi355_attn_reset(mi355_attn* h, int32_t seq, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  if (seq >= h->cfg.max_seqs)
    return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "seq %d outside [0, %d)", seq, h->cfg.max_seqs);
  for (int l = 0; l < h->cfg.num_layers; ++l)
    for (int s = 0; s < h->cfg.max_seqs; ++s)
      if (seq < 0 || s == seq) h->filled[(size_t)l * h->cfg.max_seqs + s] = 0;
  return MI355_ATTN_OK;
}

int mi355_attn_sync(mi355_attn* h, char** error_msg) {
  if (!h) return fail(error_msg, MI355_ATTN_INVALID_ARGUMENT, "null handle");
  HIP_OR_RETURN(hipSetDevice(h->device));
  HIP_OR_RETURN(hipStreamSynchronize(h->stream));
  return MI355_ATTN_OK;
}

void* mi355_attn_stream(mi355_attn* h) { return h ? h->stream : nullptr; }

int mi355_attn_set_timing(mi355_attn* h, int32_t enabled) {
  if (!h) return MI355_ATTN_INVALID_ARGUMENT;
  h->timing = enabled != 0;
  h->timed = false;
  return MI355_ATTN_OK;
}

float mi355_attn_last_kernel_ms(mi355_attn* h) {
  if (!h || !h->timed) return -1.f;
  if (hipEventSynchronize(h->ev1) != hipSuccess) return -1.f;
  float ms = -1.f;
  if (hipEventElapsedTime(&ms, h->ev0, h->ev1) != hipSuccess) return -1.f;
  return ms;
}

int mi355_attn_set_option(mi355_attn* h, const char* name, int32_t value) {
  if (!h || !name) return MI355_ATTN_INVALID_ARGUMENT;
  if (!strcmp(name, "decode_waves")) {
    if (value != 0 && value != 1 && value != 2 && value != 4) return MI355_ATTN_INVALID_ARGUMENT;
    h->tuning.waves = value;
  } else if (!strcmp(name, "rowwise_prefill")) {
    h->rowwise_prefill = value != 0;
  } else if (!strcmp(name, "prefill_workgroups")) {
    if (value < 0) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_workgroups = value;
  } else if (!strcmp(name, "prefill_rows16")) {
    if (value < -1 || value > 1) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_rows16 = value;
  } else if (!strcmp(name, "prefill_i8_stage_mib")) {
    if (value < 1) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_i8_stage_mib = value;
  } else if (!strcmp(name, "prefill_i8_min_rows")) {
    if (value < 1) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_i8_min_rows = value;
  } else if (!strcmp(name, "prefill_short")) {
    if (value < -1 || value > 1) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_short = value;
  } else if (!strcmp(name, "prefill_key_split")) {
    if (value < -1 || value > 4096) return MI355_ATTN_INVALID_ARGUMENT;
    h->prefill_key_split = value;
  } else {
    return MI355_ATTN_INVALID_ARGUMENT;
  }
  return MI355_ATTN_OK;
}

uint64_t mi355_attn_cache_bytes(const mi355_attn* h) { return h ? h->cache_bytes : 0; }

}  // extern "C"
