// Element types, plane loads and the two matrix products of one key block, for the kernels that stream K / V blocks
// from the cache planes straight into registers: decode attention and the prefill kernel for short calls.
#ifndef LITERT_LM_AMD_CSRC_KV_BLOCKS_H_
#define LITERT_LM_AMD_CSRC_KV_BLOCKS_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attn_params.h"
#include "mfma_util.h"

namespace mi355 {

constexpr float kLog2e = 1.4426950408889634f;

template <int KV>
struct KvT;
template <>
struct KvT<kF16> { static constexpr int EPC = 8, VB = 32; };
template <>
struct KvT<kBF16> { static constexpr int EPC = 8, VB = 32; };
template <>
struct KvT<kF32> { static constexpr int EPC = 4, VB = 16; };
template <>
struct KvT<kI8> { static constexpr int EPC = 16, VB = 64; };

template <int IO>
struct IoT;
template <>
struct IoT<kF32> { using type = float; };
template <>
struct IoT<kF16> { using type = _Float16; };
template <>
struct IoT<kBF16> { using type = __bf16; };

// A block of VB tokens is 64*D bytes in both planes, laid out so that load i
// of a wave is bytes [i*1024, (i+1)*1024) of the block. Buffer loads keep the
// plane base and the block offset in scalar registers (one VGPR of address per
// lane for all 32 loads) and are bounds-checked against the plane size.
constexpr int kStreamingLoad = 2;  // "nt": the rows are read once per call
constexpr int kCachedLoad = 0;     // the rows are read by several workgroups of a call
constexpr int kDeviceScope = 16;   // "sc1": through to memory, for what workgroups of one launch hand to each other

// Workgroup barrier that orders LDS traffic only (__syncthreads() would also wait for every load and store under way).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_resource(const uint8_t* plane, int64_t plane_bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(plane), 0, (int)plane_bytes, 0x00020000);
}

template <int D, int AUX = kStreamingLoad>
__device__ __forceinline__ void load_plane_block(u4 (&r)[D / 16], __amdgpu_buffer_rsrc_t rsrc, int block_off,
                                                 int lane_off) {
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    r[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_off + (i & 3) * 1024, block_off + (i >> 2) * 4096,
                                                 AUX);
}

// Eight consecutive query elements of the io type as float32 (two vectors of four: plain values, no array
// that could end up in scratch memory).
struct Q8 { f4 lo, hi; };
template <int IO>
__device__ __forceinline__ Q8 load_q8(const typename IoT<IO>::type* p) {
  Q8 r;
  if constexpr (IO == kF32) {
    r.lo = *reinterpret_cast<const f4*>(p);
    r.hi = *reinterpret_cast<const f4*>(p + 4);
  } else if constexpr (IO == kF16) {
    const h8 v = *reinterpret_cast<const h8*>(p);
    r.lo = f4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    r.hi = f4{(float)v[4], (float)v[5], (float)v[6], (float)v[7]};
  } else {
    const b8 v = *reinterpret_cast<const b8*>(p);
    r.lo = f4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    r.hi = f4{(float)v[4], (float)v[5], (float)v[6], (float)v[7]};
  }
  return r;
}

// The activation type (IO: queries in, attention out) need not be the cache's: a 16-bit cache serves float32
// activations (the reference's ActivationDataType::FLOAT32 over its fp16 GPU cache,
// runtime/executor/executor_settings_base.h:54-66), an int8 cache any of the three. The matrix cores take
// the queries in the cache's operand type, so float32 queries are rounded to it here (to nearest even), once
// per call; the output is written in the io type from the float32 accumulators.
//
// One 16-byte piece of a Q^T operand: the elements of query row `qrow` that pair with K chunk 4 * step + g (for an
// int8 cache: with one half of chunk 4 * (step / 2) + g, multiplied by the K scales `ks`).
template <int KV, int IO, int D>
__device__ __forceinline__ u4 q_operand(const typename IoT<IO>::type* qrow, const float* ks, int step, int g) {
  constexpr int EPC = KvT<KV>::EPC;
  if constexpr (KV == kI8) {
    const int d0 = (4 * (step >> 1) + g) * EPC + 8 * (step & 1);
    const Q8 x = load_q8<IO>(qrow + d0);
    const f4 s0 = *reinterpret_cast<const f4*>(ks + d0), s1 = *reinterpret_cast<const f4*>(ks + d0 + 4);
    const f4 y0 = x.lo * s0, y1 = x.hi * s1;
    const h8 o = {(_Float16)y0[0], (_Float16)y0[1], (_Float16)y0[2], (_Float16)y0[3],
                  (_Float16)y1[0], (_Float16)y1[1], (_Float16)y1[2], (_Float16)y1[3]};
    return bit_cast<u4>(o);
  } else if constexpr (KV == IO) {
    return *reinterpret_cast<const u4*>(qrow + (4 * step + g) * EPC);
  } else {
    static_assert(IO == kF32 && (KV == kF16 || KV == kBF16), "float32 activations over a 16-bit cache");
    const Q8 x = load_q8<IO>(qrow + (4 * step + g) * EPC);
    if constexpr (KV == kF16) {
      const h8 o = {(_Float16)x.lo[0], (_Float16)x.lo[1], (_Float16)x.lo[2], (_Float16)x.lo[3],
                    (_Float16)x.hi[0], (_Float16)x.hi[1], (_Float16)x.hi[2], (_Float16)x.hi[3]};
      return bit_cast<u4>(o);
    } else {
      const b8 o = {(__bf16)x.lo[0], (__bf16)x.lo[1], (__bf16)x.lo[2], (__bf16)x.lo[3],
                    (__bf16)x.hi[0], (__bf16)x.hi[1], (__bf16)x.hi[2], (__bf16)x.hi[3]};
      return bit_cast<u4>(o);
    }
  }
}

// Where a lane's Q operands of the steps lie in LDS, relative to the lane's first. Staged: [step][64 lanes] of 16 bytes.
// Rows: whole query rows in the matrix cores' type, of which lane (n, g) reads chunk 4 * step + g (int8 cache: half
// `step` % 2 of chunk 4 * (step / 2) + g) of row n.
constexpr int kStagedQ = 0, kRowsQ = 1;
template <int KV, int QL>
__device__ __forceinline__ constexpr int q_step_bytes(int step) {
  return QL == kStagedQ ? step * 1024 : (KV == kI8 ? (step >> 1) * 128 + (step & 1) * 16 : step * 64);
}
template <int KV, int QL>
__device__ __forceinline__ u4 q_at(const uint8_t* lane_q, int step) {
  return *reinterpret_cast<const u4*>(lane_q + q_step_bytes<KV, QL>(step));
}

// S^T tiles of one block: s[T][i] is the raw score of token 16*T + 4*g + i
// against head n. lane_q: this lane's Q operands in LDS; each is read once and used for every tile of the block.
template <int KV, int D, int QL = kStagedQ>
__device__ __forceinline__ void qk_block(const u4 (&kreg)[D / 16], const uint8_t* lane_q, f4 (&s)[KvT<KV>::VB / 16]) {
  constexpr int NT = KvT<KV>::VB / 16;
  constexpr int KPT = (D / 16) / NT;  // K loads per 16-token tile
#pragma unroll
  for (int T = 0; T < NT; ++T) s[T] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    if constexpr (KV == kF16) {
      const h8 qv = bit_cast<h8>(q_at<KV, QL>(lane_q, j));
#pragma unroll
      for (int T = 0; T < NT; ++T) s[T] = mfma16_f16(bit_cast<h8>(kreg[T * KPT + j]), qv, s[T]);
    } else if constexpr (KV == kBF16) {
      const b8 qv = bit_cast<b8>(q_at<KV, QL>(lane_q, j));
#pragma unroll
      for (int T = 0; T < NT; ++T) s[T] = mfma16_bf16(bit_cast<b8>(kreg[T * KPT + j]), qv, s[T]);
    } else if constexpr (KV == kF32) {
      const f4 qf = bit_cast<f4>(q_at<KV, QL>(lane_q, j));
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        const f4 kf = bit_cast<f4>(kreg[T * KPT + j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[T] = mfma16_f32(kf[e], qf[e], s[T]);
      }
    } else {
      const h8 q0 = bit_cast<h8>(q_at<KV, QL>(lane_q, 2 * j)), q1 = bit_cast<h8>(q_at<KV, QL>(lane_q, 2 * j + 1));
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        h8 lo, hi;
        cvt_i8x16_to_h8x2(kreg[T * KPT + j], lo, hi);
        s[T] = mfma16_f16(lo, q0, s[T]);
        s[T] = mfma16_f16(hi, q1, s[T]);
      }
    }
  }
}

// O^T += V^T . P^T for one block; p[T][i] pairs with token 16*T + 4*g + i.
template <int KV, int D>
__device__ __forceinline__ void pv_block(const u4 (&vreg)[D / 16], const f4 (&p)[KvT<KV>::VB / 16], f4 (&acc)[D / 16]) {
  if constexpr (KV == kF16 || KV == kBF16) {
    // (the V planes of a bfloat16 cache hold IEEE half values, attn_params.h: both run on the fp16 MFMA)
    h8 pp;
#pragma unroll
    for (int e = 0; e < 4; ++e) { pp[e] = (_Float16)p[0][e]; pp[4 + e] = (_Float16)p[1][e]; }
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db] = mfma16_f16(bit_cast<h8>(vreg[db]), pp, acc[db]);
  } else if constexpr (KV == kF32) {
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      const f4 vf = bit_cast<f4>(vreg[db]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[db] = mfma16_f32(vf[e], p[0][e], acc[db]);
    }
  } else {
    h8 p01, p23;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p01[e] = (_Float16)p[0][e]; p01[4 + e] = (_Float16)p[1][e];
      p23[e] = (_Float16)p[2][e]; p23[4 + e] = (_Float16)p[3][e];
    }
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      h8 lo, hi;
      cvt_i8x16_to_h8x2(vreg[db], lo, hi);
      acc[db] = mfma16_f16(lo, p01, acc[db]);
      acc[db] = mfma16_f16(hi, p23, acc[db]);
    }
  }
}

}  // namespace mi355
#endif  // LITERT_LM_AMD_CSRC_KV_BLOCKS_H_
