// One-token decode attention over the KV cache (gfx950, wave64, MFMA).
//
// Grid: x = layer, y = sequence, z = split-KV partition x KV head.
// A workgroup of NW waves streams the K and V rows of its partition exactly
// once. Each wave owns every NW-th block of VB tokens and, per block, issues
// 32 wave-wide 1 KiB streaming loads (16 of K, 16 of V at head_dim 256); the
// K loads of the next block are issued as soon as the current scores exist and
// the V loads right after P.V, so memory stays busy during the arithmetic. Scores are
// S^T = K . Q^T on the matrix cores with the (at most 16) query heads of the KV
// head in the column dimension, so each lane keeps the running max / sum of
// one query head; the probabilities leave the first MFMA already in the
// operand layout of the second (O^T = V^T . P^T). Waves are merged through
// LDS; partitions write (max, sum, accumulator) partials to a workspace, which
// the workgroup that writes the last of a row (launches of up to one workgroup
// a compute unit) or a small second kernel merges by log-sum-exp.
//
// Replaces the decode-time attention that the reference reaches through
// compiled_model_.Run("decode", ...)
// (runtime/executor/llm_litert_compiled_model_executor.cc:407,522).
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "attn_params.h"
#include "kernels.h"
#include <hip/hip_ext.h>

#include "kv_blocks.h"
#include "mfma_util.h"
#include "pre_attn_rows.h"

namespace mi355 {
namespace {

// Q^T as the B operand, kept by every wave in its own LDS slice as [step][lane]
// 16-byte entries: entry (jj, lane) with n = lane%16, g = lane/16 holds the
// elements of query head n that pair with K chunk 4*jj + g (for an int8 cache:
// with one half of that chunk, pre-multiplied by the K scales). Heads
// n >= group are zero columns. A lane only ever reads the entries it wrote
// itself, so no barrier is needed; keeping Q out of the register file leaves
// room for two waves per SIMD next to the 128 registers of K/V data in flight.
// q_rows: the `group` query rows of this KV head, [group][D]; ks: its K scales (int8 cache only). (A kernel that has
// produced the rows itself reads the operands from them as they lie in LDS, kRowsQ.)
template <int KV, int D>
constexpr int query_steps() { return KV == kF32 ? D / 16 : D / 32; }

template <int KV, int IO, int D, int NQ>
__device__ __forceinline__ void load_q(u4 (&w)[NQ], const typename IoT<IO>::type* q_rows, const float* ks, int group,
                                       int lane) {
  const int n = lane & 15, g = lane >> 4;
  const bool live = n < group;
  const typename IoT<IO>::type* qrow = q_rows + (live ? n : 0) * D;
#pragma unroll
  for (int step = 0; step < NQ; ++step) w[step] = q_operand<KV, IO, D>(qrow, ks, step, g);
}

template <int NQ>
__device__ __forceinline__ void store_q(u4* sm_q, const u4 (&w)[NQ], int group, int lane) {
  const bool live = (lane & 15) < group;
#pragma unroll
  for (int step = 0; step < NQ; ++step) sm_q[step * 64 + lane] = live ? w[step] : u4{0, 0, 0, 0};
}

// One wave's share of a partition: blocks first, first + step, ... < blk_end of
// the K / V planes behind krsrc / vrsrc, through the online softmax. Leaves the
// reference max (exp2 domain), this lane's share of the sum (lane (n, g): head n,
// tokens 4 g .. 4 g + 3 of every 16) and the unnormalised accumulators (channels
// 16 * db + 4 * g .. + 3 of head n). Keys outside [vlo, p_hi) are masked.
// The caller has requested block `first` into kreg / vreg (request_first_block) and left the Q
// operands in sm_q while those loads were under way (QL: how they lie there, lane_q: byte offset of the lane's first).
// patch_blk: a block one of whose rows is not in the cache yet (-1: none); patch(kreg, vreg) puts that
// row into the block's registers once they are loaded.
//
// The loads are issued on every path (`first` is wave-uniform: the caller has taken it through readfirstlane, and it is
// the very value the block loop starts from): a wave that streams nothing comes with a resource of no bytes, from which
// the loads return zeros without a trip to memory. Behind a branch of their own, the waits for whatever was loaded
// before them would have to be waits for everything.
template <int D>
__device__ __forceinline__ void request_first_block(u4 (&kreg)[D / 16], u4 (&vreg)[D / 16], __amdgpu_buffer_rsrc_t krsrc,
                                                    __amdgpu_buffer_rsrc_t vrsrc, int first, int lane) {
  load_plane_block<D>(kreg, krsrc, first * (64 * D), lane * 16);
  load_plane_block<D>(vreg, vrsrc, first * (64 * D), lane * 16);
}

template <int KV, int QL, int D, class Patch>
__device__ __forceinline__ void stream_blocks(float sc, float softcap, __amdgpu_buffer_rsrc_t krsrc,
                                              __amdgpu_buffer_rsrc_t vrsrc, u4 (&kreg)[D / 16], u4 (&vreg)[D / 16],
                                              int first, int blk_end, int step, int vlo, int p_hi, const uint8_t* sm_q,
                                              int lane_q, int patch_blk, Patch&& patch, int lane, float& m_run, float& l_run,
                                              f4 (&acc)[D / 16]) {
  constexpr int VB = KvT<KV>::VB, NT = VB / 16, NL = D / 16;
  constexpr int kBlockBytes = 64 * D;
  const int g = lane >> 4;
  const int lane_off = lane * 16;
  // Rolling prefetch: the K registers are refilled with the next block as soon
  // as the QK^T product has consumed them, the V registers right after P.V, so
  // 16 to 32 KiB per wave are in flight while it computes.
  int blk = first;  // (wave-uniform: the caller's readfirstlane)

  m_run = -INFINITY;
  l_run = 0.f;
#pragma unroll
  for (int i = 0; i < NL; ++i) acc[i] = f4{0.f, 0.f, 0.f, 0.f};

  while (blk < blk_end) {
    // The offset is made opaque so the Q reads stay inside the loop: hoisted
    // they would occupy 32 to 64 registers for the whole kernel.
    int q_off = lane_q;
    asm volatile("" : "+v"(q_off));
    if (blk == patch_blk) patch(kreg, vreg);
    f4 s[NT];
    qk_block<KV, D, QL>(kreg, sm_q + q_off, s);
    const int nxt = blk + step;
    if (nxt < blk_end) load_plane_block<D>(kreg, krsrc, nxt * kBlockBytes, lane_off);

    // scores in the exp2 domain; soft-capping and the range mask are uniform
    // branches taken only by the layers / boundary blocks that need them
    if (softcap > 0.f) {
      const float inv_cap = sc / softcap, cap2 = softcap * kLog2e;
#pragma unroll
      for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[T][i] = cap2 * fast_tanh(s[T][i] * inv_cap);
    } else {
      const float sc2 = sc * kLog2e;
#pragma unroll
      for (int T = 0; T < NT; ++T) s[T] *= sc2;
    }
    if (blk * VB < vlo || (blk + 1) * VB > p_hi) {
      const int tok0 = blk * VB + 4 * g;
#pragma unroll
      for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tok = tok0 + 16 * T + i;
          s[T][i] = (tok >= vlo && tok < p_hi) ? s[T][i] : -INFINITY;
        }
    }
    float bm = -INFINITY;
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int i = 0; i < 4; ++i) bm = fmaxf(bm, s[T][i]);
    bm = wave_xor_max<16>(bm);
    bm = wave_xor_max<32>(bm);
    const float m_new = fmaxf(m_run, bm);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float lsum = 0.f;
#pragma unroll
    for (int T = 0; T < NT; ++T) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pv = fast_exp2(s[T][i] - m_use);
        s[T][i] = pv;
        lsum += pv;
      }
    }
    l_run = l_run * alpha + lsum;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < NL; ++i) acc[i] *= alpha;
    pv_block<KV, D>(vreg, s, acc);
    if (nxt < blk_end) load_plane_block<D>(vreg, vrsrc, nxt * kBlockBytes, lane_off);
    blk = nxt;
  }

  // The four lanes (g = 0..3) of a head each summed their own tokens.
}

// What a workgroup works on: its sequence's slot, length and row in q / out, its layer's window and partition size.
struct Place { int seq, kv_len, row, window, per; };
template <int ITEMS, int LAYERS>
__device__ __forceinline__ void item_of(const DecodeWork<ITEMS, LAYERS>& work, int j, Place& p) {
  const DecodeItem it = work.item[j];
  p.seq = it.seq;
  p.kv_len = it.row_len & ((1u << kDecodeLenBits) - 1);
  p.row = it.row_len >> kDecodeLenBits;
}
// Everything in the argument blocks, at addresses that depend on the block index only: one round of scalar loads.
template <int ITEMS, int LAYERS>
__device__ __forceinline__ Place inline_place(const DecodeWork<ITEMS, LAYERS>& work, int li, int j) {
  Place p;
  item_of(work, j, p);
  const auto& t = work.layers;
  if constexpr (LAYERS == 1) {
    p.window = t.window[0];
    p.per = t.per[0];
  } else {
    const int code = (t.code[li >> 4] >> (2 * (li & 15))) & 3;
    p.window = code < 2 ? (code == 0 ? t.window[0] : t.window[1]) : (code == 2 ? t.window[2] : t.window[3]);
    p.per = code < 2 ? (code == 0 ? t.per[0] : t.per[1]) : (code == 2 ? t.per[2] : t.per[3]);
  }
  return p;
}
__device__ __forceinline__ Place table_place(const DecodeArgs& a, const DecodeWork<kInlineItems, kInlineLayers>& work,
                                             const DecodeTables& tab, int li, int j) {
  Place p;
  p.row = j;
  if (!tab.kv_lens) {
    item_of(work, j, p);
  } else {
    p.seq = tab.seq_ids ? tab.seq_ids[j] : j;
    p.kv_len = tab.kv_lens[j];
    if (tab.rows) p.row = tab.rows[j];
  }
  p.window = tab.layer_window ? tab.layer_window[a.layer_begin + li] : inline_place(work, li, 0).window;
  p.row = __builtin_amdgcn_readfirstlane(p.row);
  p.seq = __builtin_amdgcn_readfirstlane(p.seq);
  p.kv_len = __builtin_amdgcn_readfirstlane(p.kv_len);
  p.window = __builtin_amdgcn_readfirstlane(p.window);
  p.per = decode_partition_tokens(tab.max_kv_len, p.window, a.num_splits, a.align);
  return p;
}
// The blocks of a kernel's arguments behind DecodeArgs: DecodeTables where the DecodeWork does not hold everything (INL
// false), DecodePre where the kernel runs the step before attention (PRE).
struct NoBlock {};
template <bool INL>
using TableBlock = std::conditional_t<INL, NoBlock, DecodeTables>;
template <int PRE>
using PreBlock = std::conditional_t<PRE != 0, DecodePre, NoBlock>;

constexpr int kMergeRows = 16;  // partitions of a wave at a time
MI355_HD int merge_waves(int num_splits) { return num_splits >= 49 ? 4 : (num_splits + kMergeRows - 1) / kMergeRows; }

// Log-sum-exp merge of the split-KV partials: grid (query head, sequence, layer), a wave for every 16 partitions (up to
// four) that adds up their rows with four channels per lane. A launch of its own for decode launches of more workgroups than
// compute units or of more than 64 partitions, where it takes 4 to 5 us and the workgroups of the attention have their slots
// for the next ones; smaller launches merge themselves (decode_attn_kernel). What neither does is write back and invalidate
// an L2, the other way to make partials visible to another XCD: a fence pair per workgroup made the launch several times
// slower.
//
// Bound: latency. A launch moves a few hundred KiB to a few MiB; its time is its trips to memory one behind the other, so
// there are two, the arguments, then all (max, sum) pairs and rows at once, and the instructions of a single wave, so it is
// straight-line code (rows that hold nothing are read as zeros through a resource that ends in front of them, and weigh 0).
// More than 64 partitions come in further trips of 64.
// INL and the argument loads in front of the first read of the partials: as in decode_attn_kernel.
template <int KV, int IO, int D, int ITEMS, int LAYERS, bool INL>
__global__ void __launch_bounds__(256)
decode_merge_kernel(const DecodeArgs a, const DecodeWork<ITEMS, LAYERS> work, const TableBlock<INL> tab) {
  using io_t = typename IoT<IO>::type;
  static_assert(D == 4 * 64, "four channels per lane");
  __shared__ f4 sm_part[3][64];
  const int head = blockIdx.x, j = blockIdx.y, li = blockIdx.z;  // j: dispatch slot of the sequence
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int batch = a.batch, layer_begin = a.layer_begin, num_splits = a.num_splits, align = a.align, hq = a.hq;
  const float* ws_ml = a.ws_ml;
  const float* ws_acc = a.ws_acc;
  void* out = a.out;
  Place at{};
  if constexpr (INL) at = inline_place(work, li, j);
  asm volatile("" : "+s"(batch), "+s"(layer_begin), "+s"(num_splits), "+s"(align), "+s"(hq), "+s"(ws_ml), "+s"(ws_acc), "+s"(out),
               "+s"(at.seq), "+s"(at.kv_len), "+s"(at.row), "+s"(at.window), "+s"(at.per));
  if constexpr (!INL) at = table_place(a, work, tab, li, j);
  const int kv_len = at.kv_len, per = at.per;
  const int item = li * batch + at.row;
  const int layer = layer_begin + li;
  int vlo, start;
  decode_visible_range(kv_len, at.window, align, &vlo, &start);
  const int64_t slot0 = ((int64_t)item * hq + head) * num_splits;
  const float2* const mlp = reinterpret_cast<const float2*>(ws_ml) + slot0;
  // Partitions s0 .. s0 + 63, lane u of this wave partition s0 + (u + 16 wave) % 64, so that its own are in lanes 0 to 15;
  // a partition holds something if it starts in front of kv_len.
  auto live = [&](int s) { return s < num_splits && start + s * per < kv_len; };
  auto pairs = [&](int s0) {
    const int s = s0 + ((lane + kMergeRows * wave) & 63);
    return live(s) ? mlp[s] : float2{-INFINITY, 0.f};
  };
  f4 v[kMergeRows];
  auto rows = [&](int s0) {
    const int end = s0 + __popcll(__ballot(live(s0 + lane)));  // of these 64 partitions
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ws_acc + slot0 * D), 0, end * (D * 4), 0x00020000);
#pragma unroll
    for (int u = 0; u < kMergeRows; ++u)
      v[u] = bit_cast<f4>(__builtin_amdgcn_raw_buffer_load_b128(rsrc, lane * 16 + (s0 + kMergeRows * wave + u) * (D * 4), 0, 0));
  };
  float2 ml = pairs(0);
  rows(0);
  f4 vscale = {1.f, 1.f, 1.f, 1.f};
  if constexpr (KV == kI8)
    vscale = *reinterpret_cast<const f4*>(a.scales + ((((int64_t)layer * a.max_seqs + at.seq) * 2 + 1) * a.hkv + head / a.group) * D + 4 * lane);
  __builtin_amdgcn_sched_barrier(0);  // (everything is asked for before the pairs are waited for)
  float M = wave_max(ml.x);
  for (int s0 = 64; s0 < num_splits; s0 += 64) M = fmaxf(M, wave_max(pairs(s0).x));
  const float m_use = (M == -INFINITY) ? 0.f : M;
  f4 A = {0.f, 0.f, 0.f, 0.f};
  float L = 0.f;
  for (int s0 = 0;;) {
    const float wgt = fast_exp2(ml.x - m_use);
    L += wave_sum(wgt * ml.y);
#pragma unroll
    for (int u = 0; u < kMergeRows; ++u) A += lane_value(wgt, u) * v[u];
    s0 += 64;
    if (s0 >= num_splits) break;
    ml = pairs(s0);
    rows(s0);
  }
  const int waves = merge_waves(num_splits);
  if (waves > 1) {
    if (wave > 0) sm_part[wave - 1][lane] = A;
    __syncthreads();
    if (wave > 0) return;
    for (int w = 1; w < waves; ++w) A += sm_part[w - 1][lane];
  }
  io_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x = L > 0.f ? A[e] / L : 0.f;
    if constexpr (KV == kI8) x *= vscale[e];
    o[e] = (io_t)x;
  }
  io_t* orow = reinterpret_cast<io_t*>(out) + ((int64_t)item * hq + head) * D + 4 * lane;
  if constexpr (sizeof(io_t) == 4) *reinterpret_cast<u4*>(orow) = *reinterpret_cast<const u4*>(o);
  else *reinterpret_cast<u2*>(orow) = *reinterpret_cast<const u2*>(o);
}

// INL: lengths, sequence ids and windows travel in the argument block (inline_place; the host
// knows: DecodeLaunch::inline_items and inline_layers). Then everything in front of the first
// loads is one round of scalar loads at addresses that depend on the block index only. (With
// both sources in one kernel, behind a condition per value, the compiler selects a pointer and
// issues vector loads, one after the other, and a wave spent 2 to 4 us before its first K/V load.)
//
// PRE (with INL, one layer): the kernel runs the step before attention for the one new token of its
// sequence itself (row t = kv_len - 1): every workgroup norms and rotates the query rows of its KV
// head into LDS; the workgroup whose partition ends at kv_len also norms / rotates the key and value
// rows, stores them into the cache planes for later calls, and keeps them in LDS in the planes' element
// format: the wave that streams the block of row t loads it like any other block (the row's bytes are
// stale, or change under the load) and overwrites the row's bytes in its registers from LDS before the
// block is used. The MFMAs see the operands that a load after pre_attention_kernel would have
// delivered, so the results are the same bit for bit, and nothing waits for a store. No other
// workgroup reads that block (partitions are whole blocks). Same arithmetic, lane for lane, as
// pre_attention_kernel.
// The rows are serial work for a wave (a norm with its cross-lane sums per row, two full-precision sincosf per lane). In a
// launch of up to one workgroup a compute unit (kOwnWaves) four waves more have them, and the NW others request their first
// block at once. (With the block behind the rows in the same waves, the compute unit's path to memory, 16 cycles for a load
// of 1 KiB, 32 of them for each wave, brought the rows 1.2 us later.) Larger launches need the compute units' wave slots
// for the attention (64 sequences of 1,000 tokens, 8 heads on 2: 40 us instead of 29): there four waves, or the NW, do both
// (kSharedWaves), and those beyond NW leave after the rows.
enum { kNoPre = 0, kOwnWaves = 1, kSharedWaves = 2 };
constexpr int kRowWaves = 4;
template <int NW, int PRE>
constexpr int decode_wg_waves() { return PRE == kSharedWaves ? (NW < kRowWaves ? kRowWaves : NW) : NW + kRowWaves; }  // at most

// Query rows of a PRE workgroup in LDS, as the matrix cores take them: half, bfloat16 or float32, 64 bytes of padding (the
// operand reads of up to four rows then meet no bank conflict).
template <int KV>
constexpr int pre_row_bytes() { return kRowD * (KV == kF32 ? 4 : 2) + 64; }

// One float of padding per four lanes: the accumulator rows of different heads start in different banks.
constexpr int kAccStride = kRowD + 4;

// What bounds this kernel in a launch of a few short partitions (a decode step of one sequence) is the way to the first
// block: arguments, then the rows, the first K / V block and everything else that comes from memory in ONE further trip,
// and as few instructions as can be in front of it (one wave issues an instruction every four or five cycles at best: a
// hundred of them are a quarter of a microsecond). Measured on one layer's step at 1,152 tokens, from the first instruction:
// rows there at 1.3 us, attention done at 5.2; with a wait for each row in front of its norm's weights, two further rounds of
// arguments, two integer divisions and the rows in the attention's waves 2.9 and 7.0. What then ends such a launch is the
// merge below: 2.3 us, against 3 for a launch of its own and its gap, and 3 us of the host's time saved (26 layers in turn,
// 1,152 tokens: 252 us with two launches a layer, 222 with one).
template <int KV, int IO, int D, int NW, int ITEMS, int LAYERS, bool INL, int PRE>
__global__ void __launch_bounds__((decode_wg_waves<NW, PRE>()) * 64, 2)
decode_attn_kernel(const DecodeArgs a, const DecodeWork<ITEMS, LAYERS> work, const TableBlock<INL> tab, const PreBlock<PRE> pre) {
  static_assert(!PRE || INL, "the fused step needs the items in the argument block");
  constexpr int kFirstRowWave = PRE == kSharedWaves ? 0 : NW;
  constexpr int kRowStep = PRE == kSharedWaves ? decode_wg_waves<NW, PRE>() : kRowWaves;
  constexpr int VB = KvT<KV>::VB, NL = D / 16;
  constexpr int NQ = query_steps<KV, D>();
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: block addresses stay scalar
  const int n = lane & 15, g = lane >> 4;
  // Grid (layer, sequence slot, partition x KV head): partitions vary slowest in
  // dispatch order, so with ragged lengths the empty ones (sequences shorter than
  // the longest) come last instead of between the full ones; inside a partition
  // index the host has put the longest sequences first (all their layers, then the
  // next sequence), so that the short ones fill the end of the launch.
  const int li = blockIdx.x, j = blockIdx.y;
  // What the kernel needs from the argument block is read here in one go (left alone, the compiler sinks each scalar load
  // behind the branch that needs it: several dependent round trips instead of one).
  int hkv = a.hkv, batch = a.batch, layer_begin = a.layer_begin, max_seqs = a.max_seqs, num_splits = a.num_splits, align = a.align;
  uint32_t hkv_inverse = a.hkv_inverse;
  int64_t plane_bytes = a.plane_bytes;
  const uint8_t* cache = a.cache;
  int hq = a.hq, G = a.group;
  float* ws_acc = a.ws_acc;
  float* ws_ml = a.ws_ml;
  uint32_t* tickets = a.tickets;
  void* out = a.out;
  const float* scales = a.scales;
  float sc = a.scale, softcap = a.softcap;
  const void* q = a.q;
  Place at{};
  if constexpr (INL) at = inline_place(work, li, j);
  const void *pre_q = nullptr, *pre_k = nullptr, *pre_v = nullptr;
  const float* pre_constants = nullptr;
  int pre_rope = 0, norm_q = 0, norm_k = 0, norm_v = 0, q_scaled = 0, k_scaled = 0;
  float pre_eps = 0.f, pre_offset = 0.f;
  asm volatile("" : "+s"(hkv), "+s"(batch), "+s"(layer_begin), "+s"(max_seqs), "+s"(num_splits), "+s"(align), "+s"(hkv_inverse),
               "+s"(plane_bytes), "+s"(cache), "+s"(at.seq), "+s"(at.kv_len), "+s"(at.row), "+s"(at.window), "+s"(at.per));
  if constexpr (PRE) {
    pre_q = pre.q; pre_k = pre.k; pre_v = pre.v; pre_constants = pre.constants;
    pre_rope = pre.rope; norm_q = pre.norm_q; norm_k = pre.norm_k; norm_v = pre.norm_v;
    q_scaled = pre.q_scaled; k_scaled = pre.k_scaled;
    pre_eps = pre.eps; pre_offset = pre.weight_offset;
    if constexpr (PRE == kOwnWaves)
      asm volatile("" : "+s"(pre_q), "+s"(pre_k), "+s"(pre_v), "+s"(pre_constants), "+s"(pre_rope), "+s"(norm_q),
                 "+s"(norm_k), "+s"(norm_v), "+s"(q_scaled), "+s"(k_scaled), "+s"(pre_eps), "+s"(pre_offset), "+s"(hq),
                 "+s"(G), "+s"(scales), "+s"(sc), "+s"(softcap), "+s"(ws_acc), "+s"(ws_ml), "+s"(tickets), "+s"(out));
  }
  // blockIdx.z / hkv through the host's 2^32 / hkv, rounded up (0: one KV head), exact below 2^16 each
  const int split = hkv_inverse ? (int)__umulhi(blockIdx.z, hkv_inverse) : (int)blockIdx.z, kvh = blockIdx.z - split * hkv;
  const int layer = layer_begin + li;
  if constexpr (!INL) at = table_place(a, work, tab, li, j);
  const int seq = at.seq, kv_len = at.kv_len, window = at.window, per = at.per, b = at.row;
  const int item = li * batch + b;  // row of q, out and the partials
  int vlo, start;
  decode_visible_range(kv_len, window, align, &vlo, &start);
  const int p_lo = start + split * per;
  const int p_hi = min(kv_len, p_lo + per);
  if (p_lo >= p_hi) return;  // empty partition: uniform over the workgroup

  const uint8_t* kplane = cache + ((((int64_t)layer * max_seqs + seq) * hkv + kvh) * 2) * plane_bytes;  // geom.plane_offset
  const int blk_end = (p_hi + VB - 1) / VB;
  const int first_blk = __builtin_amdgcn_readfirstlane(p_lo / VB + wave);
  const int64_t streamed = wave < NW && first_blk < blk_end ? plane_bytes : 0;
  const __amdgpu_buffer_rsrc_t krsrc = plane_resource(kplane, streamed);
  const __amdgpu_buffer_rsrc_t vrsrc = plane_resource(kplane + plane_bytes, streamed);

  // LDS: the accumulators, maxima and sums of the waves (NW > 1), behind them the queries
  float* sm_acc = reinterpret_cast<float*>(smem);
  float2* sm_ml = reinterpret_cast<float2*>(sm_acc + (NW > 1 ? NW * G * kAccStride : 0));
  uint8_t* const sm_q0 = reinterpret_cast<uint8_t*>(sm_ml + (NW > 1 ? (NW * G + 1) / 2 * 2 : 0));
  float m_run, l_run;
  f4 acc[NL];
  using io_t = typename IoT<IO>::type;
  u4 kreg[NL], vreg[NL];
  if constexpr (PRE) {
    static_assert(D == kRowD, "row helpers are written for head_dim 256");
    constexpr int ESZ = KV == kF32 ? 4 : (KV == kI8 ? 1 : 2);
    constexpr int NT = VB / 16, KPT = NL / NT;
    constexpr int kRowBytes = pre_row_bytes<KV>();
    // [G] query rows as matrix operands, then the new key and value row as the planes hold them
    uint8_t* const sm_krow = sm_q0 + G * kRowBytes;
    uint8_t* const sm_vrow = sm_krow + D * ESZ;
    const int t = kv_len - 1;
    const bool owns_row = p_hi == kv_len;  // exactly one partition per sequence and KV head
    if (wave < kFirstRowWave) {
      request_first_block<D>(kreg, vreg, krsrc, vrsrc, first_blk, lane);
    } else {
      const int nrows = G + (owns_row ? 2 : 0);  // G query rows, then the key and the value row
      constexpr int kMaxRows = (kMaxGroup + 2 + kRowStep - 1) / kRowStep;
      const int d0 = 2 * lane, d1 = D / 2 + 2 * lane;
      typename RawPair<IO>::type lo[kMaxRows], hi[kMaxRows];
      float2 w0[kMaxRows], w1[kMaxRows], freq = {0.f, 0.f};
      float2 ks0, ks1, vs0, vs1;  // int8 cache: scales of the lane's channels
      ks0 = ks1 = vs0 = vs1 = float2{0.f, 0.f};
      // every row of this wave, its norm's weights, the scales and the frequencies in flight before the first is waited for
#pragma unroll
      for (int r = 0; r < kMaxRows; ++r) {
        const int row = wave - kFirstRowWave + r * kRowStep;
        w0[r] = w1[r] = float2{0.f, 0.f};
        if (row < nrows) {
          const void* src = row < G ? pre_q : (row == G ? pre_k : pre_v);
          const int64_t base = (int64_t)(row < G ? b * hq + kvh * G + row : b * hkv + kvh) * D;
          lo[r] = load_raw_pair<IO>(src, base + d0);
          hi[r] = load_raw_pair<IO>(src, base + d1);
          const float* weights = row_weights(pre_constants, row < G ? 0 : (row == G ? 1 : 2), q_scaled != 0, k_scaled != 0);
          if (weights) {
            w0[r] = *reinterpret_cast<const float2*>(weights + d0);
            w1[r] = *reinterpret_cast<const float2*>(weights + d1);
          }
        }
      }
      if (pre_rope) freq = *reinterpret_cast<const float2*>(pre_constants + d0);
      if constexpr (KV == kI8) {
        const float* ks = scales + (((int64_t)layer * max_seqs + seq) * 2 * hkv + kvh) * D;  // geom.scale_offset
        ks0 = *reinterpret_cast<const float2*>(ks + d0);
        ks1 = *reinterpret_cast<const float2*>(ks + d1);
        vs0 = *reinterpret_cast<const float2*>(ks + hkv * D + d0);
        vs1 = *reinterpret_cast<const float2*>(ks + hkv * D + d1);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PRE == kSharedWaves) {
        // The block behind the rows: a chip full of workgroups has the memory's queues full of blocks, and rows that wait in
        // line with them keep the next workgroup's wave slots.
#pragma unroll
        for (int r = 0; r < kMaxRows; ++r)
          asm volatile("" : "+v"(lo[r]), "+v"(hi[r]), "+v"(w0[r].x), "+v"(w0[r].y), "+v"(w1[r].x), "+v"(w1[r].y));
        asm volatile("" : "+v"(freq.x), "+v"(freq.y));
        if constexpr (KV == kI8)
          asm volatile("" : "+v"(ks0.x), "+v"(ks0.y), "+v"(ks1.x), "+v"(ks1.y), "+v"(vs0.x), "+v"(vs0.y), "+v"(vs1.x), "+v"(vs1.y));
        if (wave < NW) request_first_block<D>(kreg, vreg, krsrc, vrsrc, first_blk, lane);
        __builtin_amdgcn_sched_barrier(0);
      }
      const RowAngles ang = row_angles(pre_rope != 0, freq, t);
#pragma unroll
      for (int r = 0; r < kMaxRows; ++r) {
        const int row = wave - kFirstRowWave + r * kRowStep;
        if (row < nrows) {
          const int kind = row < G ? 0 : (row == G ? 1 : 2);
          const bool norm = kind == 0 ? norm_q != 0 : (kind == 1 ? norm_k != 0 : norm_v != 0);
          const bool weighted = kind == 0 ? q_scaled != 0 : (kind == 1 && k_scaled != 0);
          float x[4];
          unpack_pair<IO>(lo[r], x[0], x[1]);
          unpack_pair<IO>(hi[r], x[2], x[3]);
          transform_row(x, norm, weighted, w0[r], w1[r], pre_offset, pre_eps, pre_rope != 0 && kind != 2, ang);
          if (kind == 0) {
            // rounded to the io type, as a query that pre_attention_kernel has written out, then to the operand type
            uint8_t* dst = sm_q0 + row * kRowBytes;
            if constexpr (KV == kI8) {
              float y[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) y[e] = (float)(io_t)x[e];
              y[0] *= ks0.x; y[1] *= ks0.y; y[2] *= ks1.x; y[3] *= ks1.y;
#pragma unroll
              for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(y[e]));  // (a product of its own, rounded once more to half, as in q_operand)
              store_pair<kF16>(dst + d0 * 2, y[0], y[1]);
              store_pair<kF16>(dst + d1 * 2, y[2], y[3]);
            } else {
              store_pair<KV>(dst + d0 * ESZ, x[0], x[1]);
              store_pair<KV>(dst + d1 * ESZ, x[2], x[3]);
            }
          } else {
            const int is_v = kind - 1;
            uint8_t* plane = const_cast<uint8_t*>(kplane) + is_v * plane_bytes;
            const float2 s0 = is_v ? vs0 : ks0, s1 = is_v ? vs1 : ks1;
            store_cache_row<KV, false>(plane, s0, s1, is_v, t, x, lane);
            store_cache_row<KV, true>(is_v ? sm_vrow : sm_krow, s0, s1, is_v, t, x, lane);
          }
        }
      }
    }
    // (a barrier for LDS alone: __syncthreads() would also wait for the block under way)
    lds_barrier();
    if (wave >= NW && !tickets) return;  // a row wave has done its share
    // lane (n, g) reads row n as it lies (columns n >= G, which nobody looks at, get row 0)
    const int lane_q = (n < G ? n : 0) * kRowBytes + g * (KV == kI8 ? 32 : 16);
    // Row t in the registers of its block. K: chunk c of the row is the 16 bytes of lane (t % 16, g) in load
    // (t % VB) / 16 * KPT + j with c = 4 j + g. V: element d of the row sits in lane (d % 16, (t % 16) / 4), load
    // d / 16, at element slot 4 * ((t % VB) / 16) + t % 4 of the lane's 16 bytes.
    auto patch = [&](u4 (&kr)[NL], u4 (&vr)[NL]) __attribute__((always_inline)) {
      const int tb = t % VB;
      const int tile = tb >> 4;
      const bool k_lane = (lane & 15) == (tb & 15);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        if (T == tile) {
#pragma unroll
          for (int j = 0; j < KPT; ++j) {
            const u4 fresh = *reinterpret_cast<const u4*>(sm_krow + (4 * j + g) * 16);
            kr[T * KPT + j] = k_lane ? fresh : kr[T * KPT + j];
          }
        }
      }
      const int byte0 = (4 * tile + (tb & 3)) * ESZ;  // of the lane's 16 bytes
      const unsigned in_word = ESZ == 4 ? 0xffffffffu : ((ESZ == 2 ? 0xffffu : 0xffu) << (8 * (byte0 & 3)));
      const bool v_lane = g == ((tb & 15) >> 2);
      // The row's element slot in the lane's 16 bytes, as whole-vector operations on purpose. Written element
      // by element (vr[db][w] = ... for one w) this compiler's register allocator gave registers of the patched
      // group to the softmax as temporaries before the matrix instruction that reads the group: a sixteenth of
      // the outputs came out wrong (first seen as "wrong unless a lambda is forced inline": any change of the
      // code's shape moved it). check_decode_kernels.py looks for that pattern in every build.
      u4 mask;
#pragma unroll
      for (int w = 0; w < 4; ++w) mask[w] = (v_lane && w == (byte0 >> 2)) ? in_word : 0u;
      const u4 keep = ~mask;
#pragma unroll
      for (int db = 0; db < NL; ++db) {
        const uint8_t* src = sm_vrow + (16 * db + n) * ESZ;
        unsigned e;
        if constexpr (ESZ == 4) e = *reinterpret_cast<const unsigned*>(src);
        else if constexpr (ESZ == 2) e = *reinterpret_cast<const uint16_t*>(src);
        else e = *src;
        e <<= 8 * (byte0 & 3);
        const u4 ev = {e, e, e, e};
        vr[db] = (vr[db] & keep) | (ev & mask);
      }
    };
    if (wave < NW)
      stream_blocks<KV, kRowsQ, D>(sc, softcap, krsrc, vrsrc, kreg, vreg, first_blk, blk_end, NW, vlo, p_hi, sm_q0, lane_q,
                                   owns_row ? t / VB : -1, patch, lane, m_run, l_run, acc);
  } else if (wave < NW) {
    u4* const sm_q = reinterpret_cast<u4*>(sm_q0) + wave * (NQ * 64);
    // The queries are asked for first, the first block right behind them: loads complete in the order they were issued, so
    // the queries are staged while the block is still on its way.
    const io_t* q_rows = reinterpret_cast<const io_t*>(q) + ((int64_t)item * hq + kvh * G) * D;
    const float* ks = KV == kI8 ? scales + (((int64_t)layer * max_seqs + seq) * 2 * hkv + kvh) * D : nullptr;  // geom.scale_offset
    u4 qw[NQ];
    // (queries that are converted on the way would be waited for before the block is asked for: the block goes first)
    if constexpr (KV == IO) load_q<KV, IO, D>(qw, q_rows, ks, G, lane);
    __builtin_amdgcn_sched_barrier(0);
    request_first_block<D>(kreg, vreg, krsrc, vrsrc, first_blk, lane);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KV != IO) load_q<KV, IO, D>(qw, q_rows, ks, G, lane);
    store_q(sm_q, qw, G, lane);
    auto patch = [](u4 (&)[NL], u4 (&)[NL]) {};
    stream_blocks<KV, kStagedQ, D>(sc, softcap, krsrc, vrsrc, kreg, vreg, first_blk, blk_end, NW, vlo, p_hi,
                                   reinterpret_cast<const uint8_t*>(sm_q), lane * 16, -1, patch, lane, m_run, l_run, acc);
  }
  // Lane (n, g) holds channels 16 * db + 4 * g .. + 3 of head n; in rows of the output and of the partials:
  const int64_t head0 = (int64_t)item * hq + kvh * G;
  const float* vs = nullptr;
  if constexpr (KV == kI8) vs = scales + ((((int64_t)layer * max_seqs + seq) * 2 + 1) * hkv + kvh) * D;  // geom.scale_offset
  auto store_out = [&](int hn, f4 A, float L, f4 vscale) {  // a row, four channels per lane
    io_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = L > 0.f ? A[e] / L : 0.f;
      if constexpr (KV == kI8) x *= vscale[e];
      o[e] = (io_t)x;
    }
    io_t* orow = reinterpret_cast<io_t*>(out) + (head0 + hn) * D + 4 * lane;
    if constexpr (sizeof(io_t) == 4) *reinterpret_cast<u4*>(orow) = *reinterpret_cast<const u4*>(o);
    else *reinterpret_cast<u2*>(orow) = *reinterpret_cast<const u2*>(o);
  };
  auto load_vscale = [&]() {
    f4 r = {1.f, 1.f, 1.f, 1.f};
    if constexpr (KV == kI8) r = *reinterpret_cast<const f4*>(vs + 4 * lane);
    return r;
  };
  // The partials of this KV head, [G][num_splits] rows and pairs; written through to memory where another workgroup of the
  // launch reads them.
  const __amdgpu_buffer_rsrc_t acc_rsrc = __builtin_amdgcn_make_buffer_rsrc(ws_acc + head0 * num_splits * D, 0, G * num_splits * (D * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t ml_rsrc = __builtin_amdgcn_make_buffer_rsrc(ws_ml + head0 * num_splits * 2, 0, G * num_splits * 8, 0x00020000);
  auto store_part = [&](int hn, int d, f4 x) {
    const int at_byte = ((hn * num_splits + split) * D + d) * 4;
    if (tickets) __builtin_amdgcn_raw_buffer_store_b128(bit_cast<u4>(x), acc_rsrc, at_byte, 0, kDeviceScope);
    else __builtin_amdgcn_raw_buffer_store_b128(bit_cast<u4>(x), acc_rsrc, at_byte, 0, 0);
  };
  auto store_pair_ml = [&](int hn, float m, float l) {
    const u2 x = {__float_as_uint(m), __float_as_uint(l)};
    const int at_byte = (hn * num_splits + split) * 8;
    if (tickets) __builtin_amdgcn_raw_buffer_store_b64(x, ml_rsrc, at_byte, 0, kDeviceScope);
    else __builtin_amdgcn_raw_buffer_store_b64(x, ml_rsrc, at_byte, 0, 0);
  };
  if (wave < NW) {
    float l_tot = wave_xor_add<16>(l_run);
    l_tot = wave_xor_add<32>(l_tot);
    if constexpr (NW == 1) {
      // One wave: nothing to merge.
      if (n < G) {
        if (num_splits == 1) {
          const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
          io_t* orow = reinterpret_cast<io_t*>(out) + (head0 + n) * D + 4 * g;
#pragma unroll
          for (int db = 0; db < NL; ++db) {
            io_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float x = acc[db][e] * inv;
              if constexpr (KV == kI8) x *= vs[16 * db + 4 * g + e];
              o[e] = (io_t)x;
            }
            if constexpr (sizeof(io_t) == 4) *reinterpret_cast<u4*>(orow + 16 * db) = *reinterpret_cast<const u4*>(o);
            else *reinterpret_cast<u2*>(orow + 16 * db) = *reinterpret_cast<const u2*>(o);
          }
        } else {
#pragma unroll
          for (int db = 0; db < NL; ++db) store_part(n, 16 * db + 4 * g, acc[db]);
          if (g == 0) store_pair_ml(n, m_run, l_tot);
        }
      }
    } else {
      // Merge the waves through LDS, then a wave per head and four channels per lane.
      if (n < G) {
        float* dst = sm_acc + (wave * G + n) * kAccStride + 4 * g;
#pragma unroll
        for (int db = 0; db < NL; ++db) *reinterpret_cast<f4*>(dst + 16 * db) = acc[db];
        if (g == 0) sm_ml[wave * G + n] = float2{m_run, l_tot};
      }
      lds_barrier();
      for (int hn = wave; hn < G; hn += NW) {
        f4 v[NW];
        float2 ml[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          ml[w] = sm_ml[w * G + hn];
          v[w] = *reinterpret_cast<const f4*>(sm_acc + (w * G + hn) * kAccStride + 4 * lane);
        }
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[w].x);
        const float m_use = (M == -INFINITY) ? 0.f : M;
        f4 A = {0.f, 0.f, 0.f, 0.f};
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          const float wgt = fast_exp2(ml[w].x - m_use);
          A += wgt * v[w];
          L += wgt * ml[w].y;
        }
        if (num_splits == 1) {
          store_out(hn, A, L, load_vscale());
        } else {
          store_part(hn, 4 * lane, A);
          if (lane == 0) store_pair_ml(hn, M, L);
        }
      }
    }
  } else if constexpr (NW > 1) {
    lds_barrier();  // (a wave that is here for the merge of the partials)
  }
  if (!tickets) return;

  // The merge of the partials by the workgroup that writes the last of them: every workgroup adds its share of the keys to the
  // ticket once its stores have been acknowledged (device scope: they and the loads below go through to memory, the
  // workgroups of a row sit on different XCDs, whose L2s are different ones; no cache is written back or invalidated).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_barrier();
  uint32_t* const sm_last = reinterpret_cast<uint32_t*>(smem);
  if (threadIdx.x == 0) {
    uint32_t* ticket = tickets + item * hkv + kvh;
    const uint32_t mine = ticket_share(split, p_hi - p_lo, kv_len - start);
    *sm_last = __hip_atomic_fetch_add(ticket, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine == 0;
  }
  lds_barrier();
  if (!__builtin_amdgcn_readfirstlane((int)*sm_last)) return;
  const f4 vscale = load_vscale();
  for (int hn = wave; hn < G; hn += NW + kRowWaves) {
    // as in decode_merge_kernel, sum for sum, with up to two of its waves' rows under way together
    const bool live = lane < num_splits && start + lane * per < kv_len;
    const int nparts = __popcll(__ballot(live));
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(ws_acc + (head0 + hn) * num_splits * D, 0, nparts * (D * 4), 0x00020000);
    const u2 pair = __builtin_amdgcn_raw_buffer_load_b64(ml_rsrc, (hn * num_splits + (live ? lane : 0)) * 8, 0, kDeviceScope);
    f4 v[2 * kMergeRows];
    auto load_rows = [&](int u0, int s0) {
#pragma unroll
      for (int u = 0; u < kMergeRows; ++u)
        v[u0 + u] = bit_cast<f4>(__builtin_amdgcn_raw_buffer_load_b128(rows, lane * 16 + (s0 + u) * (D * 4), 0, kDeviceScope));
    };
    load_rows(0, 0);
    load_rows(kMergeRows, kMergeRows);
    __builtin_amdgcn_sched_barrier(0);
    const float m = live ? __uint_as_float(pair[0]) : -INFINITY;
    const float M = wave_max(m);
    const float m_use = (M == -INFINITY) ? 0.f : M;
    const float wgt = fast_exp2(m - m_use);
    const float L = wave_sum(wgt * (live ? __uint_as_float(pair[1]) : 0.f));
    f4 A = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nparts; s0 += 2 * kMergeRows) {
      if (s0 > 0) {
        load_rows(0, s0);
        load_rows(kMergeRows, s0 + kMergeRows);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kMergeRows; ++u) sum += lane_value(wgt, s0 + h * kMergeRows + u) * v[h * kMergeRows + u];
        A = s0 + h == 0 ? sum : A + sum;
      }
    }
    store_out(hn, A, L, vscale);
  }
}

template <int KV, int IO, int D, int NW, int ITEMS, int LAYERS, bool INL, int PRE = kNoPre>
hipError_t launch_inl(const DecodeLaunch& l, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  const DecodeArgs& a = l.args;
  const dim3 grid(l.n_layers, a.batch, a.num_splits * a.hkv);
  constexpr int NQ = query_steps<KV, D>();
  const size_t merge = NW > 1 ? (size_t)NW * a.group * kAccStride * sizeof(float) + (size_t)(NW * a.group + 1) / 2 * 2 * sizeof(float2) : 0;
  const size_t lds = merge + (PRE ? (size_t)a.group * pre_row_bytes<KV>() + 2 * (size_t)D * l.esize : (size_t)NW * NQ * 64 * 16);
  DecodeWork<ITEMS, LAYERS> work;
  std::copy(l.work.item, l.work.item + ITEMS, work.item);
  if constexpr (LAYERS == 1) {
    work.layers.window[0] = l.work.layers.window[0];
    work.layers.per[0] = l.work.layers.per[0];
  } else {
    work.layers = l.work.layers;
  }
  TableBlock<INL> tab{};
  if constexpr (!INL) {
    tab = l.tables;
    tab.max_kv_len = l.max_kv_len;
    if (l.inline_layers) tab.layer_window = nullptr;
    if (l.inline_items) tab.kv_lens = nullptr;
  }
  PreBlock<PRE> pre{};
  if constexpr (PRE) pre = l.pre;
  // (a launch that merges its own partials has waves that are there for that, as the fused step has for its rows)
  const int waves = PRE || a.tickets ? decode_wg_waves<NW, PRE>() : NW;
  // ev0/ev1 are attached to the dispatch itself: they carry the kernel's own
  // begin and end timestamps, not the host-side launch latency around it.
  hipExtLaunchKernelGGL((decode_attn_kernel<KV, IO, D, NW, ITEMS, LAYERS, INL, PRE>), grid, dim3(waves * 64), lds, stream, ev0,
                        ev1, 0, a, work, tab, pre);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || a.num_splits == 1 || a.tickets) return err;
  hipLaunchKernelGGL((decode_merge_kernel<KV, IO, D, ITEMS, LAYERS, INL>), dim3(a.hq, a.batch, l.n_layers),
                     dim3(64 * merge_waves(a.num_splits)), 0, stream, a, work, tab);
  return hipGetLastError();
}

template <int KV, int IO, int D, int NW>
hipError_t launch_variant(const DecodeLaunch& l, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  const bool few = l.args.batch <= kFewItems;
  if (l.fused) {
    if (!l.inline_items || !l.inline_layers || l.n_layers != 1) return hipErrorInvalidValue;
    if ((int64_t)l.rule_batch * l.args.hkv * l.args.num_splits > kLatencyWorkgroups)
      return launch_inl<KV, IO, D, NW, kInlineItems, 1, true, kSharedWaves>(l, stream, ev0, ev1);
    return few ? launch_inl<KV, IO, D, NW, kFewItems, 1, true, kOwnWaves>(l, stream, ev0, ev1)
               : launch_inl<KV, IO, D, NW, kInlineItems, 1, true, kOwnWaves>(l, stream, ev0, ev1);
  }
  if (!l.inline_items || !l.inline_layers) return launch_inl<KV, IO, D, NW, kInlineItems, kInlineLayers, false>(l, stream, ev0, ev1);
  return few ? launch_inl<KV, IO, D, NW, kFewItems, kInlineLayers, true>(l, stream, ev0, ev1)
             : launch_inl<KV, IO, D, NW, kInlineItems, kInlineLayers, true>(l, stream, ev0, ev1);
}

template <int KV, int IO, int D>
hipError_t launch_typed(const DecodeLaunch& l, const DecodeTuning& t, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  const DecodeArgs& a = l.args;
  int waves = t.waves;
  if (waves == 0) {
    // Measured on MI355X (head_dim 256, 4096-token context): with several
    // workgroups per CU one wave each is as fast or faster (fewer LDS merges),
    // with less than one per CU more waves per workgroup hide the latency:
    // one for every block of a partition, up to four (a step of one sequence of
    // 1,152 tokens in partitions of two blocks: 8.8 us with two waves, 9.4 with
    // one, 9.2 with four; of one block: 7.8, 8.1 with two).
    constexpr int VB = KvT<KV>::VB;
    const int heads = l.n_layers * l.rule_batch * a.hkv, wgs = heads * a.num_splits;
    const int blocks = decode_partition_tokens(l.max_kv_len, l.widest_window, a.num_splits, a.align) / VB;
    if (wgs <= kLatencyWorkgroups) waves = blocks >= 3 ? 4 : blocks;
    else waves = heads * l.rule_splits >= 768 || blocks <= 2 ? 1 : 2;
    // ... and four waves for a big launch of whole sequences of unequal lengths: the wave slots of
    // the chip then hold a quarter of the workgroups at a time instead of all of them, and the short
    // sequences, dispatched last, fill in behind the long ones (16 layers x 64 sequences of 256 to
    // 4096 tokens: 6.5 instead of 6.1 TB/s; sequences of equal length lose 1 % and keep one wave).
    if (a.num_splits == 1 && wgs >= 1024 && l.min_kv_len * 4 < l.max_kv_len * 3) waves = 4;
  }
  if (waves == 1) return launch_variant<KV, IO, D, 1>(l, s, e0, e1);
  if (waves == 2) return launch_variant<KV, IO, D, 2>(l, s, e0, e1);
  return launch_variant<KV, IO, D, 4>(l, s, e0, e1);
}

}  // namespace

bool decode_supported(int kv_dtype, int io_dtype, int head_dim) {
  if (head_dim != 256) return false;
  if (io_dtype != kF32 && io_dtype != kF16 && io_dtype != kBF16) return false;
  if (kv_dtype == kI8) return true;                      // int8 cache: any activation type
  return kv_dtype == io_dtype || (io_dtype == kF32 && (kv_dtype == kF16 || kv_dtype == kBF16));
}

hipError_t launch_decode(const DecodeLaunch& l, int kv_dtype, int io_dtype, const DecodeTuning& tuning,
                         hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  switch (kv_dtype * 4 + io_dtype) {
    case kF32 * 4 + kF32: return launch_typed<kF32, kF32, 256>(l, tuning, stream, ev0, ev1);
    case kF16 * 4 + kF16: return launch_typed<kF16, kF16, 256>(l, tuning, stream, ev0, ev1);
    case kF16 * 4 + kF32: return launch_typed<kF16, kF32, 256>(l, tuning, stream, ev0, ev1);
    case kBF16 * 4 + kBF16: return launch_typed<kBF16, kBF16, 256>(l, tuning, stream, ev0, ev1);
    case kBF16 * 4 + kF32: return launch_typed<kBF16, kF32, 256>(l, tuning, stream, ev0, ev1);
    case kI8 * 4 + kF16: return launch_typed<kI8, kF16, 256>(l, tuning, stream, ev0, ev1);
    case kI8 * 4 + kBF16: return launch_typed<kI8, kBF16, 256>(l, tuning, stream, ev0, ev1);
    case kI8 * 4 + kF32: return launch_typed<kI8, kF32, 256>(l, tuning, stream, ev0, ev1);
  }
  return hipErrorInvalidValue;
}

}  // namespace mi355
