// Vector types, MFMA wrappers and small device helpers for gfx950 (wave64).
//
// Operand layouts relied on (each verified on hardware by the parity tests):
//   mfma 16x16xK: A lane l supplies row l%16, K-slice group l/16;
//                 B lane l supplies column l%16, the same K-slice group;
//                 D lane l holds rows 4*(l/16)+i (i=0..3) of column l%16.
//   mfma 32x32xK: A lane l supplies row l%32, K-slice group l/32; B likewise
//                 for column l%32; D lane l holds rows 8*(i/4)+4*(l/32)+i%4
//                 (i=0..15) of column l%32.
#ifndef LITERT_LM_AMD_CSRC_MFMA_UTIL_H_
#define LITERT_LM_AMD_CSRC_MFMA_UTIL_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace mi355 {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

// Streaming 16-byte load: K/V rows are read once per call, so they bypass
// cache retention (measured: ~7.1 TB/s against ~6.0 TB/s for plain loads).
__device__ __forceinline__ u4 load_stream16(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
}

__device__ __forceinline__ f4 mfma16_f16(h8 a, h8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma16_bf16(b8 a, b8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma16_f32(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f16v mfma32_f16(h8 a, h8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f16v mfma32_bf16(b8 a, b8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <class To, class From>
__device__ __forceinline__ To bit_cast(const From& f) {
  static_assert(sizeof(To) == sizeof(From), "size mismatch");
  return __builtin_bit_cast(To, f);
}

// 16 two's-complement int8 (one 16-byte chunk) -> two h8, element order kept.
// byte ^ 0x80 = value + 128; 0x6400 | that = fp16(1024 + value + 128).
__device__ __forceinline__ void cvt_i8x16_to_h8x2(u4 w, h8& lo, h8& hi) {
  unsigned o[8];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const unsigned x = w[d] ^ 0x80808080u;
    o[2 * d] = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);      // bytes 0,1
    o[2 * d + 1] = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);  // bytes 2,3
  }
  const h8 bias = {1152, 1152, 1152, 1152, 1152, 1152, 1152, 1152};
  u4 a = {o[0], o[1], o[2], o[3]}, b = {o[4], o[5], o[6], o[7]};
  lo = bit_cast<h8>(a) - bias;
  hi = bit_cast<h8>(b) - bias;
}

// 8 two's-complement int8 (8 bytes) -> one h8, element order kept (half of cvt_i8x16_to_h8x2).
__device__ __forceinline__ h8 cvt_i8x8_to_h8(u2 w) {
  unsigned o[4];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const unsigned x = w[d] ^ 0x80808080u;
    o[2 * d] = __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u);
    o[2 * d + 1] = __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u);
  }
  const h8 bias = {1152, 1152, 1152, 1152, 1152, 1152, 1152, 1152};
  const u4 a = {o[0], o[1], o[2], o[3]};
  return bit_cast<h8>(a) - bias;
}

// bfloat16 bits -> the IEEE half that a V plane of a bfloat16 cache stores (exact for
// 2^-17 <= |v| <= 65504, finite values above saturate, nearest multiple of 2^-24 below), and back.
// NaN and +-infinity pass through as NaN and +-infinity (fminf / fmaxf would turn a NaN into a bound).
__device__ __forceinline__ uint16_t bf16_bits_to_half_bits(uint16_t b) {
  const float f = __uint_as_float((uint32_t)b << 16);
  const bool finite = (b & 0x7F80u) != 0x7F80u;
  const _Float16 h = (_Float16)(finite ? fminf(fmaxf(f, -65504.f), 65504.f) : f);
  return bit_cast<uint16_t>(h);
}
__device__ __forceinline__ uint16_t half_bits_to_bf16_bits(uint16_t hb) {
  const float f = (float)bit_cast<_Float16>(hb);  // at most 11 significant bits; what came from a bfloat16 has 8
  return bit_cast<uint16_t>((__bf16)f);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// tanh(y) = sign(y) * (1 - t) / (1 + t), t = exp(-2|y|): no overflow, no branch.
__device__ __forceinline__ float fast_tanh(float y) {
  const float t = __builtin_amdgcn_exp2f(-2.8853900817779268f * fabsf(y));
  const float r = (1.f - t) * __builtin_amdgcn_rcpf(1.f + t);
  return copysignf(r, y);
}

// Reductions over lanes a power of two apart, on the vector ALU: the DPP modes and the row swaps of gfx950 cost a few
// cycles each where a trip through the LDS crossbar (__shfl_xor) takes over a hundred. Every lane ends up with the same
// sum of the same two operands as with a xor shuffle, bit for bit. All 64 lanes must be active.
__device__ __forceinline__ float2 wave_swap16(float v) {  // {even row, odd row} of each pair of 16-lane rows
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return float2{__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ float2 wave_swap32(float v) {  // {lower half, upper half} of the wave
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return float2{__uint_as_float(r[0]), __uint_as_float(r[1])};
}
template <int MASK>
__device__ __forceinline__ float wave_xor_max(float v) {
  static_assert(MASK == 16 || MASK == 32, "rows or halves of a wave");
  const float2 r = MASK == 16 ? wave_swap16(v) : wave_swap32(v);
  return fmaxf(r.x, r.y);
}
template <int MASK>
__device__ __forceinline__ float wave_xor_add(float v) {
  static_assert(MASK == 16 || MASK == 32, "rows or halves of a wave");
  const float2 r = MASK == 16 ? wave_swap16(v) : wave_swap32(v);
  return r.x + r.y;
}
// The maximum over all lanes, in every lane.
__device__ __forceinline__ float wave_max(float v) {
  auto step = [](float x, auto ctrl) {
    return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true)));
  };
  v = step(v, std::integral_constant<int, 0xB1>{});   // (the moves of wave_sum)
  v = step(v, std::integral_constant<int, 0x4E>{});
  v = step(v, std::integral_constant<int, 0x141>{});
  v = step(v, std::integral_constant<int, 0x140>{});
  v = wave_xor_max<16>(v);
  return wave_xor_max<32>(v);
}
// The value of one lane, as a scalar.
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// The sum over all lanes, in every lane, in the order of a butterfly with xor distances 1, 2, 4, 8, 16, 32 (the mirrors
// pair a lane with one of the partner group, whose lanes all hold the same sum by then).
__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xB1>(v);   // quad_perm 1 0 3 2
  v = dpp_add<0x4E>(v);   // quad_perm 2 3 0 1
  v = dpp_add<0x141>(v);  // row_half_mirror
  v = dpp_add<0x140>(v);  // row_mirror
  v = wave_xor_add<16>(v);
  return wave_xor_add<32>(v);
}

}  // namespace mi355
#endif  // LITERT_LM_AMD_CSRC_MFMA_UTIL_H_
