// The step right before attention, in one pass over the new rows: per-head RMS
// norm of the query / key (/ value) projections, rotary position embedding of
// query and key, the query written out for the attention kernels and the key /
// value rows written straight into the cache planes in MFMA operand order
// (quantised with the plane's fixed scales for an int8 cache).
//
// Replaces, in the reference's NPU flow, the RoPE signature that turns
// `input_pos` into cos / sin tables and the cache-update signature that merges
// the new `kv_slice_{k,v}_i` rows at `input_pos`
// (runtime/executor/llm_litert_npu_compiled_model_executor.cc:82-110,1209-1219,
// 1294-1333); in the CPU/GPU executor the same work sits inside the graph behind
// compiled_model_.Run (llm_litert_compiled_model_executor.cc:271,407,522). The
// int8 write follows the quantise idiom of
// llm_litert_npu_compiled_model_executor.cc:116-148 (reciprocal scale,
// std::round, clamp).
//
// Bound: HBM for long calls, launch latency for short ones. Each row of 256 channels is read once and written once. A wave
// owns a row, a lane the channel pairs (2l, 2l+1) and (128+2l, 128+2l+1), so both members of every rotated pair (d, d+128)
// are in the same lane and the only cross-lane step is the sum of squares of the norm. Value rows that fill blocks of the
// V plane go by workgroups of their own (value_block; kBlockRowsI8 has the rule and the times), the ends of the range a
// row a wave like the others: by one workgroup a block, the up to 63 rows of an int8 end were up to sixteen dependent
// trips to memory (63 rows, 4 heads on 1: 13.8 us of kernel time, 4.1 now). (Several rows of a token per wave, so that its
// two full-precision sincosf are paid once: 26 calls of 1,024 rows take 41 us more, the launch is not bound by
// arithmetic.)
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "attn_params.h"
#include "kernels.h"
#include "mfma_util.h"
#include "pre_attn_rows.h"

namespace mi355 {
namespace {

constexpr int kD = kRowD;
constexpr int kRowsPerWg = 4;  // waves per workgroup

// Tokens of a block of the V plane: 16 KiB, whose 16-byte chunks hold several tokens of one channel each.
template <int KV>
constexpr int v_block_tokens() { return KV == kF32 ? 16 : (KV == kI8 ? 64 : 32); }

// Where the value rows of a call go: `blocks` whole blocks of each V plane from block `block0` on by a workgroup each
// (value_block), the rows in front of them (`front` tokens) and behind them by a wave each.
struct ValueRows {
  int block0, blocks, front;
};

// Channels of a value row, normed and stored, for a row that a wave writes by itself and for the rows of a block: both
// ways leave the same bytes.
template <int IO>
__device__ __forceinline__ void load_value(const PreAttentionArgs& a, int i, int head, int lane, float (&x)[4]) {
  const int64_t base = ((int64_t)i * a.geom.hkv + head) * kD;
  load_pair<IO>(a.v, base + 2 * lane, x[0], x[1]);
  load_pair<IO>(a.v, base + kD / 2 + 2 * lane, x[2], x[3]);
}
__device__ __forceinline__ void norm_value(const PreAttentionArgs& a, float (&x)[4]) {
  const RowAngles none{0.f, 1.f, 0.f, 1.f};
  transform_row(x, a.norm_v != 0, false, float2{0.f, 0.f}, float2{0.f, 0.f}, a.weight_offset, a.eps, false, none);
  // (the products stay float32 numbers, rounded once more by the store: left alone, the compiler turns product and
  // rounding into v_fma_mixlo_f16, which rounds once, in one of the two ways and not in the other)
  if (a.norm_v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(x[e]));
  }
}

// The value rows of one block of a V plane, by a workgroup. A chunk mixes tokens, so a row written by itself is 256
// stores of single elements into 256 chunks; the rows of a block that the call covers as a whole meet in LDS instead and
// leave as chunks, 1 KiB of consecutive bytes per store instruction.
template <int IO, int KV>
__device__ __forceinline__ void value_block(const PreAttentionArgs& a, int head, int block, uint8_t* sm) {
  constexpr int VB = v_block_tokens<KV>(), ESZ = KV == kF32 ? 4 : (KV == kI8 ? 1 : 2), EPC = 16 / ESZ;
  constexpr int kStride = kD * ESZ + 4 * ESZ;  // (4 rows a multiple of 256 bytes + 16 elements apart: no bank conflicts below)
  constexpr int kRows = VB / kRowsPerWg;       // of a wave: w, w + 4, ...
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t0 = block * VB;
  uint8_t* plane = a.cache + a.geom.plane_offset(a.layer, a.seq, head, 1);
  const float* sc = KV == kI8 ? a.scales + a.geom.scale_offset(a.layer, a.seq, 1, head) : nullptr;
  // (no condition around the loads: behind one, each would be waited for and converted before the next; sixteen float32
  // rows at once would be the registers that take the kernel from eight waves per SIMD to five, the row waves included)
  constexpr int kAtOnce = kRows * (IO == kF32 ? 2 : 1) > 16 ? kRows / 2 : kRows;
#pragma unroll 1
  for (int r0 = 0; r0 < kRows; r0 += kAtOnce) {
    float x[kAtOnce][4];
#pragma unroll
    for (int r = 0; r < kAtOnce; ++r) load_value<IO>(a, t0 + wave + (r0 + r) * kRowsPerWg - a.pos, head, lane, x[r]);
#pragma unroll
    for (int r = 0; r < kAtOnce; ++r) {
      norm_value(a, x[r]);
      store_cache_row<KV, true>(sm + (wave + (r0 + r) * kRowsPerWg) * kStride, sc, 1, 0, x[r], lane);
    }
  }
  __syncthreads();
  uint8_t* const out = plane + (int64_t)block * (64 * kD);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = k * 64 * kRowsPerWg + (int)threadIdx.x;  // chunk (d / 16 * 4 + g) * 16 + d % 16
    const int d = (c >> 6) * 16 + (c & 15), g = (c >> 4) & 3;
    const uint8_t* src = sm + 4 * g * kStride + d * ESZ;
    u4 w;
    if constexpr (ESZ == 4) {
#pragma unroll
      for (int s = 0; s < EPC; ++s) w[s] = *reinterpret_cast<const uint32_t*>(src + s * kStride);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 4 / ESZ; ++e) {
          const int s = q * (4 / ESZ) + e;  // slot -> token 16 * (s / 4) + 4 * g + s % 4
          const uint8_t* p = src + (16 * (s >> 2) + (s & 3)) * kStride;
          if constexpr (ESZ == 2) word |= (uint32_t)*reinterpret_cast<const uint16_t*>(p) << (16 * e);
          else word |= (uint32_t)*p << (8 * e);
        }
        w[q] = word;
      }
    }
    *reinterpret_cast<u4*>(out + (int64_t)c * 16) = w;
  }
}

// The first blocks x KV heads workgroups take a block of value rows each, the others a row per wave: the query and key
// rows token by token, behind them the value rows outside the blocks.
template <int IO, int KV>
__global__ void __launch_bounds__(64 * kRowsPerWg) pre_attention_kernel(const PreAttentionArgs a, const ValueRows v) {
  constexpr int VB = v_block_tokens<KV>(), ESZ = KV == kF32 ? 4 : (KV == kI8 ? 1 : 2);
  __shared__ __attribute__((aligned(16))) uint8_t sm[VB * (kD + 4) * ESZ];
  const int v_groups = v.blocks * a.geom.hkv;
  if ((int)blockIdx.x < v_groups) {
    value_block<IO, KV>(a, (int)blockIdx.x % a.geom.hkv, v.block0 + (int)blockIdx.x / a.geom.hkv, sm);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int rows_per_token = a.hq + a.geom.hkv, qk_rows = a.n * rows_per_token;
  const int row = ((int)blockIdx.x - v_groups) * kRowsPerWg + (int)(threadIdx.x >> 6);
  if (row >= qk_rows + (a.n - v.blocks * VB) * a.geom.hkv) return;  // whole waves leave; no barrier below
  if (row >= qk_rows) {  // a value row (a path of its own: the query and key rows are not to pay for the third kind)
    int i = (row - qk_rows) / a.geom.hkv;
    const int head = row - qk_rows - i * a.geom.hkv;
    if (i >= v.front) i += v.blocks * VB;
    float x[4];
    load_value<IO>(a, i, head, lane, x);
    norm_value(a, x);
    store_cache_row<KV>(a.cache + a.geom.plane_offset(a.layer, a.seq, head, 1),
                        KV == kI8 ? a.scales + a.geom.scale_offset(a.layer, a.seq, 1, head) : nullptr, 1, a.pos + i, x, lane);
    return;
  }
  const int i = row / rows_per_token;
  const int j = row - i * rows_per_token;
  const int kind = j < a.hq ? 0 : 1;  // 0 = query, 1 = key
  const int head = kind == 0 ? j : j - a.hq;
  const void* src = kind == 0 ? a.q : a.k;
  const int heads = kind == 0 ? a.hq : a.geom.hkv;
  const int64_t base = ((int64_t)i * heads + head) * kD;
  const int d0 = 2 * lane, d1 = kD / 2 + 2 * lane;  // the lane's channels: d0, d0+1, d1, d1+1

  float x[4];
  load_pair<IO>(src, base + d0, x[0], x[1]);
  load_pair<IO>(src, base + d1, x[2], x[3]);

  // everything the row needs comes in one trip to memory: its channels, the norm's weights, the rotary frequencies
  const int t = a.pos + i;
  const bool rotate = a.rope != 0;
  const bool norm = kind == 0 ? a.norm_q != 0 : a.norm_k != 0;
  const float* weights = row_weights(a.constants, kind, a.q_scaled != 0, a.k_scaled != 0);
  float2 w0 = {0.f, 0.f}, w1 = {0.f, 0.f}, freq = {0.f, 0.f};
  if (weights) {
    w0 = *reinterpret_cast<const float2*>(weights + d0);
    w1 = *reinterpret_cast<const float2*>(weights + d1);
  }
  if (rotate) freq = *reinterpret_cast<const float2*>(a.constants + d0);
  const RowAngles ang = row_angles(rotate, freq, t);
  transform_row(x, norm, weights != nullptr, w0, w1, a.weight_offset, a.eps, rotate, ang);

  if (kind == 0) {
    uint8_t* out = reinterpret_cast<uint8_t*>(a.q_out);
    constexpr int IOSZ = IO == kF32 ? 4 : 2;
    store_pair<IO>(out + (base + d0) * IOSZ, x[0], x[1]);
    store_pair<IO>(out + (base + d1) * IOSZ, x[2], x[3]);
    return;
  }
  uint8_t* plane = a.cache + a.geom.plane_offset(a.layer, a.seq, head, 0);
  const float* sc = KV == kI8 ? a.scales + a.geom.scale_offset(a.layer, a.seq, 0, head) : nullptr;
  store_cache_row<KV>(plane, sc, 0, t, x, lane);
}

// Calls over an int8 cache of at least this many rows (queries, keys and values) write their value rows by blocks, other
// caches' always do. 8,192 waves are resident at once: up to there every row has a wave of its own from the start, and
// the sixteen rows that a wave of an int8 block takes one after the other only make the launch longer. Kernel time by
// rows / by blocks, us, bfloat16 and float32 activations: 1,024 rows of 4 heads on 1 (6,144 in all) 4.6 / 5.0 and
// 4.8 / 5.8, 512 of 8 on 4 (8,192) 5.8 / 5.7 and 6.3 / 6.0, 2,048 of 4 on 1 (12,288) 7.1 / 6.3 and 7.7 / 6.9. For half,
// bfloat16 and float32 caches (4 or 8 rows a wave) blocks are level up to 6,144 rows (1,024 of 4 on 1: 4.6 / 4.5) and
// ahead from there (1,024 of 8 on 4: 9.6 / 6.8).
constexpr int64_t kBlockRowsI8 = 8192;

template <int IO, int KV>
hipError_t launch_typed(const PreAttentionArgs& a, hipStream_t stream, hipEvent_t ev0, hipEvent_t ev1) {
  constexpr int VB = v_block_tokens<KV>();
  ValueRows v{0, 0, a.n};
  if (KV != kI8 || (int64_t)a.n * (a.hq + 2 * a.geom.hkv) >= kBlockRowsI8) {
    const int first = (a.pos + VB - 1) / VB, end = (a.pos + a.n) / VB;
    if (end > first) v = ValueRows{first, end - first, first * VB - a.pos};
  }
  const int64_t rows = (int64_t)a.n * (a.hq + a.geom.hkv) + (int64_t)(a.n - v.blocks * VB) * a.geom.hkv;
  const int64_t groups = (int64_t)v.blocks * a.geom.hkv + (rows + kRowsPerWg - 1) / kRowsPerWg;
  if (rows > INT32_MAX - kRowsPerWg || groups > INT32_MAX) return hipErrorInvalidValue;
  hipExtLaunchKernelGGL((pre_attention_kernel<IO, KV>), dim3((unsigned)groups), dim3(64 * kRowsPerWg), 0, stream, ev0, ev1, 0,
                        a, v);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pre_attention(const PreAttentionArgs& a, int kv_dtype, int io_dtype, hipStream_t stream,
                                hipEvent_t ev0, hipEvent_t ev1) {
  if (a.n <= 0) return hipSuccess;
  if (a.geom.head_dim != kD) return hipErrorInvalidValue;
  switch (kv_dtype * 4 + io_dtype) {
    case kF32 * 4 + kF32: return launch_typed<kF32, kF32>(a, stream, ev0, ev1);
    case kF16 * 4 + kF16: return launch_typed<kF16, kF16>(a, stream, ev0, ev1);
    case kF16 * 4 + kF32: return launch_typed<kF32, kF16>(a, stream, ev0, ev1);
    case kBF16 * 4 + kBF16: return launch_typed<kBF16, kBF16>(a, stream, ev0, ev1);
    case kBF16 * 4 + kF32: return launch_typed<kF32, kBF16>(a, stream, ev0, ev1);
    case kI8 * 4 + kF16: return launch_typed<kF16, kI8>(a, stream, ev0, ev1);
    case kI8 * 4 + kBF16: return launch_typed<kBF16, kI8>(a, stream, ev0, ev1);
    case kI8 * 4 + kF32: return launch_typed<kF32, kI8>(a, stream, ev0, ev1);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mi355
