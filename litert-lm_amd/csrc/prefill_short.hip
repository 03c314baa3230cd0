// Prefill attention for calls that are too small to fill the chip with whole query tiles (gfx950, wave64, MFMA).
//
// A workgroup takes the 16 MFMA columns of one KV head that hold R consecutive positions x all `group` query heads
// (R = the largest power of two with R * group <= 16, stretches aligned to R positions) and walks all key blocks
// that those positions see; its eight waves deal the blocks out among themselves, each wave streaming its blocks
// from the planes straight into registers (the decode kernel's loads and products, kv_blocks.h), and merge through
// LDS at the end. Against the tiled kernels of prefill_attn.hip, where a workgroup takes 32 positions and a short
// call is cut over the keys into work items whose float32 parts travel through HBM to a merge launch, this has 8
// times as many workgroups of an eighth of the keys per wave, no parts in HBM and one launch.
//
// Bound: a 16-column tile reads 32 KiB of K and V per 32 matrix instructions, so beyond one tile per compute unit
// the path from the L2 (64 bytes per clock and compute unit) sets the time, and the tiled kernels, which feed 128
// columns from every block they bring in, take over (prefill_short_wanted has the line and what was measured).
//
// Replaces, like prefill_attn.hip, the attention behind compiled_model_.Run(prefill_signature, ...)
// (runtime/executor/llm_litert_compiled_model_executor.cc:271).
#include <atomic>
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <math.h>

#include "attn_params.h"
#include "kernels.h"
#include "kv_blocks.h"
#include "mfma_util.h"

namespace mi355 {
namespace {

constexpr int kCols = 16;
constexpr int kAccStride = 4;  // floats of padding per accumulator row in LDS (16 rows a power of two apart share their banks)

// Launches of up to this many workgroups use eight waves each (one workgroup a compute unit), larger ones four.
constexpr long kWideWorkgroups = 256;

int short_tiles(int q_pos0, int n, int rows_log2) { return ((q_pos0 + n - 1) >> rows_log2) - (q_pos0 >> rows_log2) + 1; }

template <int KV, int D>
constexpr int query_steps() { return KV == kF32 ? D / 16 : D / 32; }

// LDS: query operands [steps][64 lanes] of 16 bytes, accumulators [waves][columns][D + pad], (max, sum) [waves][columns]
template <int KV, int D, int NW>
constexpr int lds_bytes() {
  return query_steps<KV, D>() * 1024 + NW * kCols * (D + kAccStride) * 4 + NW * kCols * 8;
}

// NW waves per workgroup; either way eight waves a compute unit, two per SIMD, which is all that 256 registers per
// lane leave room for.
template <int KV, int IO, int D, int NW, bool CAP>
__global__ void __launch_bounds__(NW * 64, 2) prefill_short_kernel(const PrefillShortArgs a) {
  using io_t = typename IoT<IO>::type;
  constexpr int VB = KvT<KV>::VB, NT = VB / 16, NL = D / 16;
  constexpr int NQ = query_steps<KV, D>();
  constexpr int kBlockBytes = 64 * D;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  u4* const sm_q = reinterpret_cast<u4*>(smem);
  float* const sm_acc = reinterpret_cast<float*>(smem + NQ * 1024);
  float2* const sm_ml = reinterpret_cast<float2*>(sm_acc + NW * kCols * (D + kAccStride));

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // Grid (layer x KV head, tile): units vary fastest, so that tiles are dispatched from the longest key range down.
  const int unit = blockIdx.x;
  const int li = unit / a.geom.hkv, kvh = unit - li * a.geom.hkv;
  const int layer = a.layer_begin + li;
  const int window = a.window[li];
  const int tile = (int)gridDim.y - 1 - (int)blockIdx.y;
  const int rows_log2 = a.rows_log2, rows = 1 << rows_log2;
  const int pos_end = a.q_pos0 + a.n;
  const int tile_pos = ((a.q_pos0 >> rows_log2) + tile) << rows_log2;  // may lie in front of q_pos0, rows behind pos_end
  const int first_pos = max(tile_pos, a.q_pos0), last_pos = min(tile_pos + rows, pos_end) - 1;
  const int lo_first = window > 0 ? max(0, first_pos - window + 1) : 0;
  const int lo_last = window > 0 ? max(0, last_pos - window + 1) : 0;
  const int blk0 = lo_first / VB, blk_end = last_pos / VB + 1;

  // this lane's column: head and position (columns without a row of the call hold zero queries and are not stored)
  const int head = c >> rows_log2;  // column = head * rows + row, so that a row's heads need no division
  const int pos = tile_pos + (c & (rows - 1));
  const bool live = head < a.group && pos >= first_pos && pos <= last_pos;
  const int vlo = window > 0 ? max(0, pos - window + 1) : 0;
  const int64_t row = live ? pos - a.q_pos0 : 0;
  const int64_t q_elem = (((int64_t)li * a.n + row) * a.hq + kvh * a.group + (live ? head : 0)) * D;

  const uint8_t* kplane = a.cache + a.geom.plane_offset(layer, a.seq, kvh, 0);
  int blk = blk0 + wave;
  // (a wave without a block has a resource of no bytes: its first loads return zeros without a trip to memory; behind a
  // branch, the wait for the queries would have to be a wait for everything)
  const int64_t streamed = blk < blk_end ? a.geom.plane_bytes : 0;
  const __amdgpu_buffer_rsrc_t krsrc = plane_resource(kplane, streamed);
  const __amdgpu_buffer_rsrc_t vrsrc = plane_resource(kplane + a.geom.plane_bytes, streamed);

  // This wave's share of the query operands goes first, then its first K and V blocks: the wait for the former leaves
  // the latter under way. (Queries that are converted on the way would be waited for before the blocks are asked for:
  // then the blocks go first.)
  static_assert(NQ % NW == 0, "every wave stages the same number of operands");
  constexpr int kQPerWave = NQ / NW;
  u4 qw[kQPerWave];
  auto load_queries = [&]() {
    const float* ks = KV == kI8 ? a.scales + a.geom.scale_offset(layer, a.seq, 0, kvh) : nullptr;
    const io_t* qrow = reinterpret_cast<const io_t*>(a.q) + q_elem;
#pragma unroll
    for (int s = 0; s < kQPerWave; ++s) qw[s] = q_operand<KV, IO, D>(qrow, ks, wave * kQPerWave + s, g);
  };
  if constexpr (KV == IO) load_queries();
  __builtin_amdgcn_sched_barrier(0);
  u4 kreg[NL], vreg[NL];
  load_plane_block<D, kCachedLoad>(kreg, krsrc, blk * kBlockBytes, lane * 16);
  load_plane_block<D, kCachedLoad>(vreg, vrsrc, blk * kBlockBytes, lane * 16);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (KV != IO) load_queries();
#pragma unroll
  for (int s = 0; s < kQPerWave; ++s) sm_q[(wave * kQPerWave + s) * 64 + lane] = live ? qw[s] : u4{0, 0, 0, 0};
  // (a barrier for LDS alone: __syncthreads() would also wait for the blocks under way)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  float m_run = -INFINITY, l_run = 0.f;
  f4 acc[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) acc[i] = f4{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale, softcap = a.softcap;
  while (blk < blk_end) {
    int qi = lane;  // opaque, so that the operand reads stay in the loop (hoisted they would fill the registers)
    asm volatile("" : "+v"(qi));
    f4 s[NT];
    qk_block<KV, D>(kreg, sm_q, qi, s);
    const int nxt = blk + NW;
    if (nxt < blk_end) load_plane_block<D, kCachedLoad>(kreg, krsrc, nxt * kBlockBytes, lane * 16);
    if constexpr (CAP) {
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
    // the blocks at the edges of the tile's key range hold keys that some of its positions do not see
    if (blk * VB < lo_last || (blk + 1) * VB > first_pos + 1) {
      const int tok0 = blk * VB + 4 * g;
#pragma unroll
      for (int T = 0; T < NT; ++T)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tok = tok0 + 16 * T + i;
          s[T][i] = (tok >= vlo && tok <= pos) ? s[T][i] : -INFINITY;
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
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pv = fast_exp2(s[T][i] - m_use);
        s[T][i] = pv;
        lsum += pv;
      }
    l_run = l_run * alpha + lsum;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < NL; ++i) acc[i] *= alpha;
    pv_block<KV, D>(vreg, s, acc);
    if (nxt < blk_end) load_plane_block<D, kCachedLoad>(vreg, vrsrc, nxt * kBlockBytes, lane * 16);
    blk = nxt;
  }
  float l_tot = wave_xor_add<16>(l_run);
  l_tot = wave_xor_add<32>(l_tot);

  // Merge the waves that had a block: accumulators and (max, sum) through LDS, then a wave per column and 4 channels
  // per lane, so that whole rows leave.
  const int nw = min(NW, blk_end - blk0);
  if (wave < nw) {
    float* dst = sm_acc + (wave * kCols + c) * (D + kAccStride) + 4 * g;
#pragma unroll
    for (int db = 0; db < NL; ++db) *reinterpret_cast<f4*>(dst + 16 * db) = acc[db];
    if (g == 0) sm_ml[wave * kCols + c] = float2{m_run, l_tot};
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kCols / NW; ++k) {
    const int col = k * NW + wave;
    const int h = col >> rows_log2, p = tile_pos + (col & (rows - 1));
    if (h >= a.group || p < first_pos || p > last_pos) continue;  // (uniform over the wave)
    float M = -INFINITY;
    for (int w = 0; w < nw; ++w) M = fmaxf(M, sm_ml[w * kCols + col].x);
    const float m_use = (M == -INFINITY) ? 0.f : M;
    f4 A = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
    for (int w = 0; w < nw; ++w) {
      const float2 ml = sm_ml[w * kCols + col];
      const float wgt = fast_exp2(ml.x - m_use);
      A += wgt * *reinterpret_cast<const f4*>(sm_acc + (w * kCols + col) * (D + kAccStride) + 4 * lane);
      L += wgt * ml.y;
    }
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = L > 0.f ? A[e] / L : 0.f;
    if constexpr (KV == kI8)
      o *= *reinterpret_cast<const f4*>(a.scales + a.geom.scale_offset(layer, a.seq, 1, kvh) + 4 * lane);
    io_t* orow = reinterpret_cast<io_t*>(a.out) + (((int64_t)li * a.n + (p - a.q_pos0)) * a.hq + kvh * a.group + h) * D + 4 * lane;
    io_t w4[4] = {(io_t)o[0], (io_t)o[1], (io_t)o[2], (io_t)o[3]};
    if constexpr (sizeof(io_t) == 4) *reinterpret_cast<u4*>(orow) = *reinterpret_cast<const u4*>(w4);
    else *reinterpret_cast<u2*>(orow) = *reinterpret_cast<const u2*>(w4);
  }
}

template <int KV, int IO, int D, int NW, bool CAP>
hipError_t launch_variant(const PrefillShortArgs& a, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  constexpr int kLds = lds_bytes<KV, D, NW>();
  // more than 64 KiB of LDS has to be requested once per kernel (idempotent: callers on several threads may both ask)
  static std::atomic<bool> configured{false};
  if (!configured.load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_short_kernel<KV, IO, D, NW, CAP>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    configured.store(true, std::memory_order_release);
  }
  const int tiles = short_tiles(a.q_pos0, a.n, a.rows_log2);
  hipExtLaunchKernelGGL((prefill_short_kernel<KV, IO, D, NW, CAP>), dim3(a.n_layers * a.geom.hkv, tiles), dim3(NW * 64), kLds,
                        stream, ev0, ev1, 0, a);
  return hipGetLastError();
}

template <int KV, int IO>
hipError_t launch_typed(const PrefillShortArgs& a, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  const int tiles = short_tiles(a.q_pos0, a.n, a.rows_log2);
  if ((long)tiles * a.n_layers * a.geom.hkv > kWideWorkgroups)
    return a.softcap > 0.f ? launch_variant<KV, IO, 256, 4, true>(a, stream, ev0, ev1)
                           : launch_variant<KV, IO, 256, 4, false>(a, stream, ev0, ev1);
  return a.softcap > 0.f ? launch_variant<KV, IO, 256, 8, true>(a, stream, ev0, ev1)
                         : launch_variant<KV, IO, 256, 8, false>(a, stream, ev0, ev1);
}

}  // namespace

int prefill_short_rows_log2(int group) {
  int r = 0;
  while ((2 << r) * group <= kCols) ++r;
  return r;
}

// Whether the short kernel is expected to finish a call before the tiled kernels of prefill_attn.hip, by the times in
// microseconds that both were measured to take (head_dim 256, MI355X, calls queued back to back, 64 to 2,048 rows behind
// 0 to 4,096 cached ones, 1 to 40 layers; the two formulas are within some 15 % of the measured times, and the short
// kernel has to come out ahead by as much). Examples, tiled / short, bfloat16, 4 query heads on 1 KV head: one layer of 64
// rows 9.9 / 5.1 us, 256 rows 15.9 / 8.0, 1,024 rows 29.5 / 14.1, 2,048 rows 41.2 / 29.6; four layers of 1,024 rows with
// a window of 512 41 / 27, eight 32 / 47, 26 of 256 rows 20 / 28; 64 rows behind 4,096 (8 heads on 2) 32 / 38. int8 cache,
// 300 rows 24 / 10, 256 rows behind 3,072 47 / 31. A float32 cache always takes the short kernel: the alternative is
// one decode item per row, which reads every key once per position instead of once per 16 columns (300 rows 36 / 17,
// 300 behind 2,000 305 / 81).
// The activation type is not part of the rule, so that calls that differ in nothing else run the same arithmetic.
bool prefill_short_wanted(int kv_dtype, int hq, int hkv, const int32_t* window, int n_layers, int q_pos0, int n) {
  constexpr int kCus = 256;  // (what the times were measured on; the launches themselves ask the device)
  if (kv_dtype == kF32) return true;
  const int group = hq / hkv, rows_log2 = prefill_short_rows_log2(group);
  const int vb = kv_dtype == kI8 ? 64 : 32;
  const double wgs = (double)n_layers * hkv * short_tiles(q_pos0, n, rows_log2);
  if (wgs > 16 * kCus) return false;
  const int hpb = group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);
  const int tile_rows = 32 * (4 / hpb), tiles = (n + tile_rows - 1) / tile_rows;
  const double items = (double)n_layers * hkv * (group / hpb) * tiles;
  // key blocks of a stretch of `rows` positions: mean over the call (the count is linear in the position but for the
  // corner at the window, so a few samples do) and most
  auto blocks = [&](int w, int first, int rows, int block) {
    const int last = first + rows - 1;
    const int lo = w > 0 && first - w + 1 > 0 ? first - w + 1 : 0;
    return (double)(last / block - lo / block + 1);
  };
  constexpr int kSamples = 9;
  double short_mean = 0, short_most = 0, tiled_mean = 0, tiled_most = 0;
  for (int li = 0; li < n_layers; ++li)
    for (int k = 0; k < kSamples; ++k) {
      const int at = q_pos0 + (int)((int64_t)(n - 1) * k / (kSamples - 1));
      const double bs = blocks(window[li], at >> rows_log2 << rows_log2, 1 << rows_log2, vb);
      const double bt = blocks(window[li], at, n < tile_rows ? n : tile_rows, 32);
      short_mean += bs;
      tiled_mean += bt;
      if (bs > short_most) short_most = bs;
      if (bt > tiled_most) tiled_most = bt;
    }
  short_mean /= kSamples * n_layers;
  tiled_mean /= kSamples * n_layers;

  const double per_block = kv_dtype == kI8 ? 1.75 : 1.0;  // (64 keys instead of 32, and a conversion)
  double t_short;
  if (wgs <= kWideWorkgroups) {
    t_short = 4.5 + 0.28 * per_block * short_most;
  } else {
    const double longest = 0.36 * per_block * short_most, rate = 0.32 * per_block * short_mean * wgs / kCus + 2.7 * wgs / (2 * kCus);
    t_short = 5.0 + (longest > rate ? longest : rate);
  }
  double t_tiled;
  int want = items * 4 >= 3 * kCus ? 1 : (int)((kCus + items - 1) / items);
  if (want > 8) want = 8;
  if (want > tiled_most / 4) want = (int)(tiled_most / 4);
  if (want > 1) {  // keys split over work items, parts merged by a second launch (plan_prefill_split)
    const double chunk = tiled_most / want;
    const double part_bytes = tiled_mean / chunk * n_layers * n * hq * 1024;
    t_tiled = 9.0 + 1.5 * chunk + 2 * part_bytes / 4.7e6;
  } else if (items < 2 * kCus) {
    const double rounds = (double)(((long)items + kCus - 1) / kCus) * (4.0 + 1.6 * tiled_mean), longest = 4.0 + 1.6 * tiled_most;
    t_tiled = 4.0 + (rounds > longest ? rounds : longest);
  } else {
    const double rate = 1.25 * tiled_mean * items / kCus, longest = 1.75 * tiled_most;
    t_tiled = 7.0 + (rate > longest ? rate : longest);
  }
  if (kv_dtype == kI8) t_tiled += 5.5;  // the staging pass
  return t_short * 1.15 < t_tiled;
}

hipError_t launch_prefill_short(const PrefillShortArgs& a, int kv_dtype, int io_dtype, hipStream_t stream, hipEvent_t ev0,
                                hipEvent_t ev1) {
  if (a.n_layers < 1 || a.n_layers > kInlineLayers || a.group < 1 || a.group > kCols || a.n < 1 || a.geom.head_dim != 256)
    return hipErrorInvalidValue;
  const int tiles = short_tiles(a.q_pos0, a.n, a.rows_log2);
  if (tiles > 65535) return hipErrorInvalidValue;
  switch (kv_dtype * 4 + io_dtype) {
    case kF32 * 4 + kF32: return launch_typed<kF32, kF32>(a, stream, ev0, ev1);
    case kF16 * 4 + kF16: return launch_typed<kF16, kF16>(a, stream, ev0, ev1);
    case kF16 * 4 + kF32: return launch_typed<kF16, kF32>(a, stream, ev0, ev1);
    case kBF16 * 4 + kBF16: return launch_typed<kBF16, kBF16>(a, stream, ev0, ev1);
    case kBF16 * 4 + kF32: return launch_typed<kBF16, kF32>(a, stream, ev0, ev1);
    case kI8 * 4 + kF16: return launch_typed<kI8, kF16>(a, stream, ev0, ev1);
    case kI8 * 4 + kBF16: return launch_typed<kI8, kBF16>(a, stream, ev0, ev1);
    case kI8 * 4 + kF32: return launch_typed<kI8, kF32>(a, stream, ev0, ev1);
  }
  return hipErrorInvalidValue;
}

}  // namespace mi355
