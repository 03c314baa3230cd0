// Prefill attention for calls that are too small to fill the chip with whole query tiles (gfx950, wave64, MFMA).
//
// A workgroup takes the 16 MFMA columns of one KV head that hold R consecutive positions x all `group` query heads
// (R = the largest power of two with R * group <= 16, stretches aligned to R positions) and walks all key blocks
// that those positions see; its eight waves deal the blocks out among themselves, each wave streaming its blocks
// from the planes straight into registers (the decode kernel's loads and products, kv_blocks.h), and merge through
// LDS at the end. Against the tiled kernels of prefill_attn.hip, where a workgroup takes 32 positions and a short
// call is cut over the keys into work items whose float32 parts travel through HBM to a merge launch, this has 8
// times as many workgroups of an eighth of the keys per wave and one launch; a call that leaves half of the compute units
// without a tile cuts its tiles over the keys too, into parts that the launch merges itself.
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

#include <algorithm>
#include <type_traits>

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

constexpr int kMinPartBlocks = 4;  // key blocks of a part of a split tile, at least

int short_tiles(int q_pos0, int n, int rows_log2) { return ((q_pos0 + n - 1) >> rows_log2) - (q_pos0 >> rows_log2) + 1; }

template <int KV, int D>
constexpr int query_steps() { return KV == kF32 ? D / 16 : D / 32; }

// LDS: query operands [steps][64 lanes] of 16 bytes, accumulators [waves][columns][D + pad], (max, sum) [waves][columns]
template <int KV, int D, int NW>
constexpr int lds_bytes() {
  return query_steps<KV, D>() * 1024 + NW * kCols * (D + kAccStride) * 4 + NW * kCols * 8;
}

// NW waves per workgroup, eight waves a compute unit either way, two per SIMD, which is all that 256 registers per lane
// leave room for; but for a float32 cache in launches of four waves, whose 81.5 KiB of LDS let one workgroup run on a
// compute unit instead of two.
//
// A call of few tiles cuts each of them into up to `parts` stretches of its key blocks, a workgroup each (grid z). A part
// leaves its unnormalised sums, maxima and totals in the workspace by device-scope stores, adds its share of the blocks to the
// tile's ticket, and the workgroup that completes the tile adds the parts up in order (as decode_attn_kernel does).
template <int KV, int IO, int D, int NW, bool CAP, int LAYERS>
__global__ void __launch_bounds__(NW * 64, 2) prefill_short_kernel(const PrefillShortArgs a, const PrefillWindows<LAYERS> windows) {
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
  // Grid (layer x KV head, tile, part): units vary fastest, so that tiles are dispatched from the longest key range down.
  // Everything in front of the first load comes in one round of scalar loads (left alone, each is sunk to its use).
  const int unit = blockIdx.x;
  int hkv = a.hkv, max_seqs = a.max_seqs, hq = a.hq, group = a.group, layer_begin = a.layer_begin, seq = a.seq;
  int q_pos0 = a.q_pos0, rows_n = a.n, rows_log2 = a.rows_log2, tiles = a.tiles;
  uint32_t hkv_inverse = a.hkv_inverse, parts_inverse = a.parts_inverse;
  int64_t plane_bytes = a.plane_bytes;
  const uint8_t* cache = a.cache;
  const float* scales = a.scales;
  const void* q = a.q;
  // (with one layer its window comes in the same round, else behind the unit's layer)
  int window = LAYERS == 1 ? windows.of[0] : 0;
  asm volatile("" : "+s"(hkv), "+s"(max_seqs), "+s"(hq), "+s"(group), "+s"(layer_begin), "+s"(seq), "+s"(q_pos0), "+s"(rows_n),
               "+s"(rows_log2), "+s"(tiles), "+s"(hkv_inverse), "+s"(parts_inverse), "+s"(plane_bytes), "+s"(cache), "+s"(scales),
               "+s"(q), "+s"(window));
  const int li = LAYERS == 1 ? 0 : (hkv_inverse ? (int)__umulhi(unit, hkv_inverse) : unit), kvh = unit - li * hkv;
  if constexpr (LAYERS > 1) window = windows.of[li];
  const int layer = layer_begin + li;
  const int tile = tiles - 1 - (int)blockIdx.y;
  const int rows = 1 << rows_log2;
  const int pos_end = q_pos0 + rows_n;
  const int tile_pos = ((q_pos0 >> rows_log2) + tile) << rows_log2;  // may lie in front of q_pos0, rows behind pos_end
  const int first_pos = max(tile_pos, q_pos0), last_pos = min(tile_pos + rows, pos_end) - 1;
  const int lo_first = window > 0 ? max(0, first_pos - window + 1) : 0;
  const int lo_last = window > 0 ? max(0, last_pos - window + 1) : 0;
  int blk0 = lo_first / VB, blk_end = last_pos / VB + 1;
  // this part of the tile's blocks
  const int tile_blocks = blk_end - blk0;
  int per_part = tile_blocks;
  if (parts_inverse) {
    // (ceil(blocks / parts) through the host's inverse, exact for what a plane holds)
    per_part = max(kMinPartBlocks, (int)__umulhi(tile_blocks + a.parts - 1, parts_inverse));
    blk0 += (int)blockIdx.z * per_part;
    blk_end = min(blk_end, blk0 + per_part);
    if (blk0 >= blk_end) return;  // (uniform over the workgroup)
  }

  // this lane's column: head and position (columns without a row of the call hold zero queries and are not stored)
  const int head = c >> rows_log2;  // column = head * rows + row, so that a row's heads need no division
  const int pos = tile_pos + (c & (rows - 1));
  const bool live = head < group && pos >= first_pos && pos <= last_pos;
  const int vlo = window > 0 ? max(0, pos - window + 1) : 0;
  const int64_t row = live ? pos - q_pos0 : 0;
  const int64_t q_elem = (((int64_t)li * rows_n + row) * hq + kvh * group + (live ? head : 0)) * D;

  const uint8_t* kplane = cache + ((((int64_t)layer * max_seqs + seq) * hkv + kvh) * 2) * plane_bytes;  // geom.plane_offset
  const float* ks = KV == kI8 ? scales + (((int64_t)layer * max_seqs + seq) * 2 * hkv + kvh) * D : nullptr;  // geom.scale_offset
  int blk = blk0 + wave;
  // (a wave without a block has a resource of no bytes: its first loads return zeros without a trip to memory; behind a
  // branch, the wait for the queries would have to be a wait for everything)
  const int64_t streamed = blk < blk_end ? plane_bytes : 0;
  const __amdgpu_buffer_rsrc_t krsrc = plane_resource(kplane, streamed);
  const __amdgpu_buffer_rsrc_t vrsrc = plane_resource(kplane + plane_bytes, streamed);

  // This wave's share of the query operands goes first, then its first K block: the wait for the former leaves the latter
  // under way. (Queries that are converted on the way would be waited for before the block is asked for: then the block goes
  // first.) The V block is requested behind the barrier that the queries need: the compute unit takes 16 cycles for a load
  // of 1 KiB, so the V blocks of eight waves are a microsecond in which no wave could reach the barrier (26 layers of 1,024
  // rows in turn: 410 us with both blocks in front of it, 390 so).
  static_assert(NQ % NW == 0, "every wave stages the same number of operands");
  constexpr int kQPerWave = NQ / NW;
  u4 qw[kQPerWave];
  auto load_queries = [&]() {
    const io_t* qrow = reinterpret_cast<const io_t*>(q) + q_elem;
#pragma unroll
    for (int s = 0; s < kQPerWave; ++s) qw[s] = q_operand<KV, IO, D>(qrow, ks, wave * kQPerWave + s, g);
  };
  if constexpr (KV == IO) load_queries();
  __builtin_amdgcn_sched_barrier(0);
  u4 kreg[NL], vreg[NL];
  load_plane_block<D, kCachedLoad>(kreg, krsrc, blk * kBlockBytes, lane * 16);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (KV != IO) load_queries();
#pragma unroll
  for (int s = 0; s < kQPerWave; ++s) sm_q[(wave * kQPerWave + s) * 64 + lane] = live ? qw[s] : u4{0, 0, 0, 0};
  lds_barrier();  // (__syncthreads() would also wait for the blocks under way)
  load_plane_block<D, kCachedLoad>(vreg, vrsrc, blk * kBlockBytes, lane * 16);
  __builtin_amdgcn_sched_barrier(0);

  float m_run = -INFINITY, l_run = 0.f;
  f4 acc[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) acc[i] = f4{0.f, 0.f, 0.f, 0.f};
  const float sc = a.scale, softcap = a.softcap;
  while (blk < blk_end) {
    int q_off = lane * 16;  // opaque, so that the operand reads stay in the loop (hoisted they would fill the registers)
    asm volatile("" : "+v"(q_off));
    f4 s[NT];
    qk_block<KV, D>(kreg, smem + q_off, s);
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

  // Merge the waves that had a block: accumulators and (max, sum) through LDS, then kCols / NW columns a wave with 4 channels
  // per lane, so that whole rows leave. All LDS reads of a column go out together: one after the other, wave by wave, they
  // were 2 us of a 10 us launch.
  const int nw = min(NW, blk_end - blk0);
  if (wave < nw) {
    float* dst = sm_acc + (wave * kCols + c) * (D + kAccStride) + 4 * g;
#pragma unroll
    for (int db = 0; db < NL; ++db) *reinterpret_cast<f4*>(dst + 16 * db) = acc[db];
    if (g == 0) sm_ml[wave * kCols + c] = float2{m_run, l_tot};
  }
  f4 vscale = {1.f, 1.f, 1.f, 1.f};
  if constexpr (KV == kI8) vscale = *reinterpret_cast<const f4*>(ks + hkv * D + 4 * lane);
  lds_barrier();
  constexpr int kColsPerWave = kCols / NW;
  f4 A[kColsPerWave];
  float M[kColsPerWave], L[kColsPerWave];
  // (all: every wave had a block. Conditions around the reads, or idle waves that bring zeros, would cost the others more)
  auto merge_column = [&](int k, auto all) {
    constexpr bool kAll = decltype(all)::value;
    const int col = k * NW + wave;
    const float2* mlp = sm_ml + col;
    const float* accp = sm_acc + col * (D + kAccStride) + 4 * lane;
    float2 ml[NW];
    f4 v[NW];
    if constexpr (kAll) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        ml[w] = mlp[w * kCols];
        v[w] = *reinterpret_cast<const f4*>(accp + w * kCols * (D + kAccStride));
      }
    }
    M[k] = -INFINITY;
#pragma unroll kAll ? NW : 1
    for (int w = 0; w < (kAll ? NW : nw); ++w) M[k] = fmaxf(M[k], kAll ? ml[w].x : mlp[w * kCols].x);
    const float m_use = (M[k] == -INFINITY) ? 0.f : M[k];
    A[k] = f4{0.f, 0.f, 0.f, 0.f};
    L[k] = 0.f;
#pragma unroll kAll ? NW : 1
    for (int w = 0; w < (kAll ? NW : nw); ++w) {
      const float2 x = kAll ? ml[w] : mlp[w * kCols];
      const f4 y = kAll ? v[w] : *reinterpret_cast<const f4*>(accp + w * kCols * (D + kAccStride));
      const float wgt = fast_exp2(x.x - m_use);
      A[k] += wgt * y;
      L[k] += wgt * x.y;
    }
  };
  if (nw == NW) {
#pragma unroll
    for (int k = 0; k < kColsPerWave; ++k) merge_column(k, std::true_type{});
  } else {
#pragma unroll
    for (int k = 0; k < kColsPerWave; ++k) merge_column(k, std::false_type{});
  }
  if (per_part < tile_blocks) {
    // a part: its columns to the workspace, and the last part of the tile adds them up
    const int64_t slot0 = ((int64_t)unit * tiles + tile) * a.parts;
    const __amdgpu_buffer_rsrc_t acc_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(a.ws_acc + slot0 * (kCols * D), 0, a.parts * (kCols * D * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t ml_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(a.ws_ml + slot0 * (kCols * 2), 0, a.parts * (kCols * 8), 0x00020000);
#pragma unroll
    for (int k = 0; k < kColsPerWave; ++k) {
      const int at = (int)blockIdx.z * kCols + k * NW + wave;
      __builtin_amdgcn_raw_buffer_store_b128(bit_cast<u4>(A[k]), acc_rsrc, at * (D * 4) + lane * 16, 0, kDeviceScope);
      if (lane == 0) __builtin_amdgcn_raw_buffer_store_b64(u2{__float_as_uint(M[k]), __float_as_uint(L[k])}, ml_rsrc, at * 8, 0, kDeviceScope);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    uint32_t* const sm_last = reinterpret_cast<uint32_t*>(smem);
    if (threadIdx.x == 0) {
      uint32_t* ticket = a.tickets + unit * tiles + tile;
      const uint32_t mine = ticket_share(blockIdx.z, blk_end - blk0, tile_blocks);
      *sm_last = __hip_atomic_fetch_add(ticket, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine == 0;
    }
    lds_barrier();
    if (!__builtin_amdgcn_readfirstlane((int)*sm_last)) return;
    f4 v[kColsPerWave][kShortParts];
    u2 ml[kColsPerWave][kShortParts];
#pragma unroll
    for (int k = 0; k < kColsPerWave; ++k)
#pragma unroll
      for (int p = 0; p < kShortParts; ++p) {
        // (a part that does not exist is read as zeros behind the resource's end, and weighs 0)
        const int at = p * per_part < tile_blocks ? p * kCols + k * NW + wave : kShortParts * kCols;
        ml[k][p] = __builtin_amdgcn_raw_buffer_load_b64(ml_rsrc, at * 8, 0, kDeviceScope);
        v[k][p] = bit_cast<f4>(__builtin_amdgcn_raw_buffer_load_b128(acc_rsrc, at * (D * 4) + lane * 16, 0, kDeviceScope));
      }
#pragma unroll
    for (int k = 0; k < kColsPerWave; ++k) {
      float m[kShortParts];
      M[k] = -INFINITY;
#pragma unroll
      for (int p = 0; p < kShortParts; ++p) {
        m[p] = p * per_part < tile_blocks ? __uint_as_float(ml[k][p][0]) : -INFINITY;
        M[k] = fmaxf(M[k], m[p]);
      }
      const float m_use = (M[k] == -INFINITY) ? 0.f : M[k];
      A[k] = f4{0.f, 0.f, 0.f, 0.f};
      L[k] = 0.f;
#pragma unroll
      for (int p = 0; p < kShortParts; ++p) {
        const float wgt = fast_exp2(m[p] - m_use);
        A[k] += wgt * v[k][p];
        L[k] += wgt * __uint_as_float(ml[k][p][1]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kColsPerWave; ++k) {
    const int col = k * NW + wave;
    const int h = col >> rows_log2, p = tile_pos + (col & (rows - 1));
    if (h >= group || p < first_pos || p > last_pos) continue;  // (uniform over the wave)
    f4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = L[k] > 0.f ? A[k][e] / L[k] : 0.f;
    if constexpr (KV == kI8) o *= vscale;
    io_t* orow = reinterpret_cast<io_t*>(a.out) + (((int64_t)li * rows_n + (p - q_pos0)) * hq + kvh * group + h) * D + 4 * lane;
    io_t w4[4] = {(io_t)o[0], (io_t)o[1], (io_t)o[2], (io_t)o[3]};
    if constexpr (sizeof(io_t) == 4) *reinterpret_cast<u4*>(orow) = *reinterpret_cast<const u4*>(w4);
    else *reinterpret_cast<u2*>(orow) = *reinterpret_cast<const u2*>(w4);
  }
}

template <int KV, int IO, int D, int NW, bool CAP, int LAYERS>
hipError_t launch_variant(const PrefillShortArgs& a, const int32_t* window, int n_layers, hipStream_t stream, hipEvent_t ev0,
                          hipEvent_t ev1) {
  constexpr int kLds = lds_bytes<KV, D, NW>();
  // more than 64 KiB of LDS has to be requested once per kernel (idempotent: callers on several threads may both ask)
  static std::atomic<bool> configured{false};
  if (!configured.load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_short_kernel<KV, IO, D, NW, CAP, LAYERS>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    configured.store(true, std::memory_order_release);
  }
  PrefillWindows<LAYERS> windows{};
  std::copy(window, window + n_layers, windows.of);
  hipExtLaunchKernelGGL((prefill_short_kernel<KV, IO, D, NW, CAP, LAYERS>), dim3(n_layers * a.hkv, a.tiles, a.parts), dim3(NW * 64),
                        kLds, stream, ev0, ev1, 0, a, windows);
  return hipGetLastError();
}

template <int KV, int IO, int NW, bool CAP>
hipError_t launch_layers(const PrefillShortArgs& a, const int32_t* window, int n_layers, hipStream_t stream, hipEvent_t ev0,
                         hipEvent_t ev1) {
  return n_layers == 1 ? launch_variant<KV, IO, 256, NW, CAP, 1>(a, window, 1, stream, ev0, ev1)
                       : launch_variant<KV, IO, 256, NW, CAP, kInlineLayers>(a, window, n_layers, stream, ev0, ev1);
}

template <int KV, int IO>
hipError_t launch_typed(const PrefillShortArgs& a, const int32_t* window, int n_layers, hipStream_t stream, hipEvent_t ev0,
                        hipEvent_t ev1) {
  if ((long)a.tiles * n_layers * a.hkv > kWideWorkgroups)
    return a.softcap > 0.f ? launch_layers<KV, IO, 4, true>(a, window, n_layers, stream, ev0, ev1)
                           : launch_layers<KV, IO, 4, false>(a, window, n_layers, stream, ev0, ev1);
  return a.softcap > 0.f ? launch_layers<KV, IO, 8, true>(a, window, n_layers, stream, ev0, ev1)
                         : launch_layers<KV, IO, 8, false>(a, window, n_layers, stream, ev0, ev1);
}

}  // namespace

int prefill_short_rows_log2(int group) {
  int r = 0;
  while ((2 << r) * group <= kCols) ++r;
  return r;
}

// Parts of the tiles of a call of `wgs` tiles, the longest of `most` key blocks: as few as end the launch first by the
// times measured (us: a key block of a workgroup 0.72 over a float32 cache, 0.40 over an int8 one, 0.184 otherwise; the parts'
// way through the workspace 3), a workgroup a compute unit. Whole tiles / parts, us a call back to back: 300 rows over a float32
// cache, 4 heads on 1: three parts, 16.6 / 13.6; 100 rows behind 1,000: eight, 42.0 / 15.3; 64 behind 3,000, int8, 8 on 2: eight,
// 28.2 / 14.4; 26 behind 6,843, fp16, 8 on 1: eight, 66.8 / 16.7, and 38.1 on the tiled kernels.
int prefill_short_parts(int kv_dtype, long wgs, int most) {
  if (wgs > kShortPartSlots / 2) return 1;
  const double block = kv_dtype == kF32 ? 0.72 : (kv_dtype == kI8 ? 0.40 : 0.184), merge = 3.0;
  int best = 1;
  double t = block * most;
  for (int p = 2; p <= kShortParts && p * wgs <= kShortPartSlots; ++p) {
    const double tp = block * std::max((most + p - 1) / p, kMinPartBlocks) + merge;
    if (tp < t - 0.2) {
      best = p;
      t = tp;
    }
  }
  return best;
}

int prefill_short_call_parts(int kv_dtype, int group, int hkv, const int32_t* window, int n_layers, int q_pos0, int n) {
  const int rows_log2 = prefill_short_rows_log2(group);
  const int vb = kv_dtype == kF32 ? 16 : (kv_dtype == kI8 ? 64 : 32);
  int most = 0;
  for (int l = 0; l < n_layers; ++l) {
    // (a tile at the end of the call sees the most blocks, but where the window cuts them all alike)
    const int last = q_pos0 + n - 1, lo = window[l] > 0 ? std::max(0, (last >> rows_log2 << rows_log2) - window[l] + 1) : 0;
    most = std::max(most, last / vb - lo / vb + 1);
  }
  return prefill_short_parts(kv_dtype, (long)short_tiles(q_pos0, n, rows_log2) * n_layers * hkv, most);
}

// Whether the short kernel is expected to finish a call before the tiled kernels of prefill_attn.hip: both sides by
// formulas fitted to measured times (head_dim 256, MI355X, calls queued back to back, 1,140 shapes spread at random over
// 16 to 4,096 rows behind 0 to 12,000 cached ones, 1 to 34 layers with and without windows, sixteen head counts; the formula
// of calls of up to 256 tiles again, with their parts, to 133). On 296 other shapes of both kernels what they choose takes 0.3 %
// longer than the better side in the mean, three of them by 10 to 31 % (the worst 26 layers of 34 rows behind 249, 16 heads
// on 2: 25 / 19). Examples, tiled / short, us: bfloat16, 4 query heads on 1 KV head, one layer of 256 rows 17.2 / 7.0, 1,024
// rows 25.8 / 12.0; 8 heads on 2, 2 layers of 1,768 behind 693 83 / 96. int8 cache, 300 rows 21.8 / 9.5, 64 rows behind 3,000
// 31.2 / 14.4. A float32 cache always takes the short kernel: the alternative is one decode item per row, which reads every
// key once per position instead of once per 16 columns (300 rows 36 / 13.6, 300 behind 2,000 305 / 33.5).
//
// What decides for the short kernel beside the key blocks themselves is where its workgroups run. They go round the eight
// XCDs and, within each, round its four engines of eight compute units, with the units (layer x KV head) varying fastest:
// if the number of units shares a factor f with 32, all tiles of a unit are the work of 32 / f engines. With 8 units the
// only global layer among windowed ones has a single XCD (8 layers of 1,686 rows behind 1,059, window 512: 204 us, tiled
// 92), with 32 a single engine (16 layers of 108 rows behind 3,058, window 1,024: 103 us, tiled 63). And units whose
// planes do not fit an XCD's L2 (4 MiB) together are read from behind it again and again.
//
// The activation type is not part of the rule, so that calls that differ in nothing else run the same arithmetic.
bool prefill_short_wanted(int kv_dtype, int hq, int hkv, const int32_t* window, int n_layers, int q_pos0, int n) {
  constexpr int kCus = 256, kXcds = 8, kEngines = 32;  // what the times were measured on
  if (kv_dtype == kF32) return true;
  const bool i8 = kv_dtype == kI8;
  const int group = hq / hkv, rows_log2 = prefill_short_rows_log2(group);
  const int vb = i8 ? 64 : 32;
  const int units = n_layers * hkv;
  const double tiles = short_tiles(q_pos0, n, rows_log2), wgs = units * tiles;
  if (wgs > 16 * kCus) return false;
  const int hpb = group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);
  const int tile_rows = prefill_tile_rows(group);
  const long items = (long)n_layers * hkv * (group / hpb) * ((n + tile_rows - 1) / tile_rows);
  const int classes = std::min(units & -units, kEngines);  // of units that share engines
  const int xcd_classes = std::min(classes, kXcds);
  // key blocks of a stretch of `rows` positions: mean over the call (the count is linear in the position but for the
  // corner at the window, so a few samples do) and most
  auto blocks = [&](int w, int first, int rows, int block) {
    const int last = first + rows - 1;
    const int lo = w > 0 && first - w + 1 > 0 ? first - w + 1 : 0;
    return (double)(last / block - lo / block + 1);
  };
  constexpr int kSamples = 9;
  double short_mean = 0, short_most = 0, short_least = 1e9, tiled_mean = 0, tiled_most = 0, tiled_least = 1e9;
  double load[kEngines] = {};  // of a class: key blocks per compute unit
  double planes[kXcds] = {};   // MiB of K and V that an XCD sees
  double sum_s = 0, sum_t = 0;                  // of the layer (kept from the layer before where the window is the same)
  int seen = 0;
  bool mixed = false;  // layers with different windows
  for (int li = 0; li < n_layers; ++li) {
    if (li == 0 || window[li] != window[li - 1]) {
      mixed = li > 0;
      sum_s = sum_t = 0;
      for (int k = 0; k < kSamples; ++k) {
        const int at = q_pos0 + (int)((int64_t)(n - 1) * k / (kSamples - 1));
        const double bs = blocks(window[li], at >> rows_log2 << rows_log2, 1 << rows_log2, vb);
        const double bt = blocks(window[li], at, n < tile_rows ? n : tile_rows, 32);
        sum_s += bs;
        sum_t += bt;
        short_most = fmax(short_most, bs);
        short_least = fmin(short_least, bs);
        tiled_most = fmax(tiled_most, bt);
        tiled_least = fmin(tiled_least, bt);
      }
      const int lo = window[li] > 0 && q_pos0 - window[li] + 1 > 0 ? q_pos0 - window[li] + 1 : 0;
      seen = (q_pos0 + n - 1) / vb - lo / vb + 1;
    }
    short_mean += sum_s / (kSamples * n_layers);
    tiled_mean += sum_t / (kSamples * n_layers);
    for (int h = 0; h < hkv; ++h) {
      const int c = (li * hkv + h) % classes;
      load[c] += sum_s / kSamples * tiles * classes / kCus;
      planes[c % xcd_classes] += seen / 32.0;  // (a block is 32 KiB of K and V)
    }
  }
  // Up to two rounds over the compute units, longest first: the one that gets the longest of the second round as well.
  auto two_rounds = [&](double count, double from, double to) { return to + from + (to - from) * (1 - kCus / count); };

  double planes_mean = 0;
  for (int c = 0; c < xcd_classes; ++c) planes_mean += planes[c] / xcd_classes;
  double t_short;
  if (wgs <= kWideWorkgroups) {
    const int parts = prefill_short_parts(kv_dtype, (long)wgs, (int)short_most);
    const double walked = parts > 1 ? fmax(ceil(short_most / parts), kMinPartBlocks) : short_most;
    t_short = i8 ? 6.4 + 0.40 * walked + 0.66 * planes_mean + (parts > 1 ? 3.3 : 0)
                 : 5.4 + 0.184 * walked + 0.68 * planes_mean + (parts > 1 ? 3.0 : 0);
  } else {
    // The compute units of the busiest engine, in blocks each, with what an L2 too small costs (the workgroups of a unit
    // walk its blocks together while all run at once, and less and less so in more rounds or beside shorter layers) ...
    double busiest = 0;
    const double rounds = wgs / (2 * kCus), apart = fmin(1.0, fmax(0.0, (rounds - 1) / (i8 ? 2.2 : 1.3)));
    for (int c = 0; c < classes; ++c) {
      const double over = fmax(0.0, planes[c % xcd_classes] - 4);
      const double slow = mixed ? fmin(i8 ? 1.07 : 1.57, (i8 ? 0.16 : 0.117) * over)
                                : apart * fmin(i8 ? 0.9 : 3.0, (i8 ? 0.027 : 0.064) * over);
      busiest = fmax(busiest, load[c] * (1 + slow));
    }
    // ... and in rounds of two workgroups a compute unit, longest first: what is left for the last one is a round all the same
    const double full = floor(rounds), rest = wgs - full * 2 * kCus;
    if (rounds <= 1) busiest = fmax(busiest, two_rounds(wgs, short_least, short_most));
    else busiest = fmax(busiest, 2 * full * short_mean + (rest > kCus ? 2 : (rest > 0 ? (i8 ? 0.65 : 1.26) : 0)) * short_least);
    t_short = (i8 ? 4.7 : 3.6) + fmax((i8 ? 0.45 : 0.28) * short_most, (i8 ? 0.42 : 0.212) * busiest) +
              (i8 ? 5.6 : 4.4) * rounds + (i8 ? 0.65 : 0.95) * planes_mean;
  }

  const int most = prefill_most_key_blocks(window, n_layers, q_pos0, n, tile_rows);
  const PrefillParts split = choose_prefill_parts(items, most, n_layers, n, hq, kCus, true);
  double t_tiled;
  if (split.parts > 1) {
    const long slots = split.direct ? 2 * kCus : kCus;
    const double walked = (double)((most + split.parts - 1) / split.parts) * ((items * split.parts + slots - 1) / slots);
    const double part_bytes = (double)split.parts * tiled_mean / most * n_layers * n * hq * 1024;
    t_tiled = (split.direct ? 7.9 + 1.4 * walked : 10.5 + 0.89 * walked) + 2.8 + 1.17 * 2 * part_bytes / 4.7e6;
  } else if (items < 2 * kCus) {
    double walked = fmax(tiled_mean * items / kCus, tiled_most);
    if (items > kCus) walked = fmax(walked, two_rounds(items, tiled_least, tiled_most));
    t_tiled = 6.8 + 0.85 * walked + 6.8 * items / kCus;
  } else {
    t_tiled = 14.2 + fmax(1.1 * tiled_mean * items / kCus, 1.2 * tiled_most);
  }
  // (the staging pass of an int8 cache: planes read and written as halves, queries in 16 bits)
  if (i8) t_tiled += 3.0 + 0.14e-6 * 256 * ((double)units * 2 * (q_pos0 + n) * 3 + (double)n_layers * n * hq * 4);
  // (16-bit caches: 5 % for the pass that rounds float32 queries, which the times above are without. An int8 cache in
  // launches of up to two workgroups a compute unit: the tiled times come out some 5 % too long around the tie of 1,024
  // rows behind 3,072, 60 / 62 us)
  return t_short < (i8 ? (wgs > kWideWorkgroups && wgs <= 2 * kCus ? 0.95 : 1.0) : 1.05) * t_tiled;
}

hipError_t launch_prefill_short(PrefillShortArgs a, const int32_t* window, int n_layers, int kv_dtype, int io_dtype,
                                hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  if (n_layers < 1 || n_layers > kInlineLayers || a.group < 1 || a.group > kCols || a.n < 1) return hipErrorInvalidValue;
  a.rows_log2 = prefill_short_rows_log2(a.group);
  a.tiles = short_tiles(a.q_pos0, a.n, a.rows_log2);
  if (a.tiles > 65535) return hipErrorInvalidValue;
  a.parts = prefill_short_call_parts(kv_dtype, a.group, a.hkv, window, n_layers, a.q_pos0, a.n);
  auto inverse = [](int d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
  a.parts_inverse = inverse(a.parts);
  a.hkv_inverse = inverse(a.hkv);
  switch (kv_dtype * 4 + io_dtype) {
    case kF32 * 4 + kF32: return launch_typed<kF32, kF32>(a, window, n_layers, stream, ev0, ev1);
    case kF16 * 4 + kF16: return launch_typed<kF16, kF16>(a, window, n_layers, stream, ev0, ev1);
    case kF16 * 4 + kF32: return launch_typed<kF16, kF32>(a, window, n_layers, stream, ev0, ev1);
    case kBF16 * 4 + kBF16: return launch_typed<kBF16, kBF16>(a, window, n_layers, stream, ev0, ev1);
    case kBF16 * 4 + kF32: return launch_typed<kBF16, kF32>(a, window, n_layers, stream, ev0, ev1);
    case kI8 * 4 + kF16: return launch_typed<kI8, kF16>(a, window, n_layers, stream, ev0, ev1);
    case kI8 * 4 + kBF16: return launch_typed<kI8, kBF16>(a, window, n_layers, stream, ev0, ev1);
    case kI8 * 4 + kF32: return launch_typed<kI8, kF32>(a, window, n_layers, stream, ev0, ev1);
  }
  return hipErrorInvalidValue;
}

}  // namespace mi355
