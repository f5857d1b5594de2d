// gdnr_act16.h -- device helpers of the kernels that take 16-bit activations
// (gdnr_decode.hip, gdnr_ring.hip), compiled once per activation dtype
// (GDNR_ACT = 0 bf16, 1 f16): MFMA operands from ring rows and e4m3 codes,
// uniform loads, 16-lane row operations, gating inputs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gdnr_device.h"
#include "gdnr_internal.h"

namespace gdnr {
namespace {

constexpr int K = kKeyDim;
constexpr int NT = kStepRing;  // token rows of an operand (a ring of up to 16 tokens, or a chunk of a longer one)

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

#if GDNR_ACT == 0
using Act = ActBF16;
#define GDNR_SUFFIX(name) name##_bf16
#else
using Act = ActF16;
#define GDNR_SUFFIX(name) name##_f16
#endif
constexpr bool kBF16 = std::is_same<Act, ActBF16>::value;

__device__ __forceinline__ f32x4_t mfma16(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (kBF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                  0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma_bf16(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}
// 4 e4m3 codes -> 4 values of the activation type (exact), packed in pairs
__device__ __forceinline__ uint2 codes4(uint32_t w) { return kBF16 ? fp8x4_to_bf16x4(w) : fp8x4_to_f16x4(w); }
// the 8 codes of k-step m of a lane's 32 bytes of a row (c[0]: bytes
// [32 q4, +16), c[1]: [32 q4 + 16, +16); k-step m: bytes 32 q4 + 8 m + 0..7)
__device__ __forceinline__ u32x4_t codes8(const u32x4_t* c, int m) {
  const u32x4_t w = c[m >> 1];
  const uint32_t w0 = (m & 1) ? w[2] : w[0], w1 = (m & 1) ? w[3] : w[1];
  const uint2 lo = codes4(w0);
  const uint2 hi = codes4(w1);
  return u32x4_t{lo.x, lo.y, hi.x, hi.y};
}
// f32x4_to_fp8_ref with its constants formed where it runs (through empty
// asm statements, which stay in place): the flush's rare division path uses
// it, and constants hoisted out of the flush loop would hold registers for
// the whole loop
__device__ __forceinline__ uint32_t f32x4_to_fp8_ref_cold(float a, float b, float c, float d) {
  float lim = 448.0f;
  uint32_t k7f = 0x7Fu, kff = 0xFFu;
  asm volatile("" : "+v"(lim), "+v"(k7f), "+v"(kff));
  const float v[4] = {a, b, c, d};
  float cl[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cl[e] = (v[e] != v[e]) ? v[e] : fminf(fmaxf(v[e], -lim), lim);
  uint32_t w = f32x4_to_fp8(cl[0], cl[1], cl[2], cl[3]);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (v[e] != v[e]) w = (w & ~(kff << (8 * e))) | ((__float_as_uint(v[e]) >> 31 ? kff : k7f) << (8 * e));
  return w;
}
// activation value from 16 bits
__device__ __forceinline__ float act_val(uint32_t bits16) { return Act::from_bits(bits16 & 0xFFFFu); }
__device__ __forceinline__ uint32_t act_bits(float x) {
  if constexpr (kBF16) return f32_to_bf16(x);
  else return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x);
}

__device__ __forceinline__ float rdl(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
// a uniform value the compiler cannot see through: work derived from it
// stays after this point (is not hoisted into code shared by the roles,
// where it would wait for the argument block)
__device__ __forceinline__ int opaque_s(int x) {
  asm volatile("" : "+s"(x));
  return x;
}
__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// uniform loads through the scalar cache of data this kernel does not write
// before reading it (constant address space; they count in lgkmcnt)
typedef __attribute__((address_space(4))) const uint32_t const_u32;
__device__ __forceinline__ uint32_t ld_u32_uniform(const void* p) { return *(const_u32*)p; }
__device__ __forceinline__ uint32_t ld_u16_uniform(const uint8_t* p) {
  const uintptr_t ad = (uintptr_t)p;
  return (ld_u32_uniform((const void*)(ad & ~(uintptr_t)3)) >> (8u * (uint32_t)(ad & 2))) & 0xFFFFu;
}
__device__ __forceinline__ u32x4_t ld16(const uint8_t* p) { return *(const u32x4_t*)p; }
typedef __attribute__((address_space(1))) const u32x4_t g_u32x4;
typedef __attribute__((address_space(1))) u32x4_t g_u32x4_w;
__device__ __forceinline__ uint32_t ld32(const uint8_t* p) { return *(const uint32_t*)p; }
// A sequence's (slot's) base in a tensor, in 64 bits: the tensors of a slot
// cache may span more than 4 GiB; offsets inside one sequence stay 32-bit.
__device__ __forceinline__ uint8_t* sbase(const uint8_t* p, int seq, uint32_t stride) {
  return (uint8_t*)p + (uint64_t)(uint32_t)seq * stride;
}
// x + y for two 32-bit products, kept as two multiplies and an add: the fused
// form (v_mad_u64_u32, whose unused upper addend half the allocator may give
// a register an outstanding load is filling) makes the wave wait for every
// load issued before it
__device__ __forceinline__ uint32_t off_sum(uint32_t x, uint32_t y) {
  asm volatile("" : "+v"(x), "+v"(y));
  return x + y;
}
// DPP move within a 16-lane row; lanes whose source is outside the row get `fill`
template <int CTRL>
__device__ __forceinline__ float dpp_row(float x, float fill) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fill), __builtin_bit_cast(int, x),
                                                               CTRL, 0xF, 0xF, false));
}
// every lane of each 16-lane row gets lane n of its row (DPP row_newbcast)
template <int N>
__device__ __forceinline__ float row_bcast(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + N, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_bcast_n(float x, int n) {
  switch (n) {
    case 0: return row_bcast<0>(x);   case 1: return row_bcast<1>(x);   case 2: return row_bcast<2>(x);
    case 3: return row_bcast<3>(x);   case 4: return row_bcast<4>(x);   case 5: return row_bcast<5>(x);
    case 6: return row_bcast<6>(x);   case 7: return row_bcast<7>(x);   case 8: return row_bcast<8>(x);
    case 9: return row_bcast<9>(x);   case 10: return row_bcast<10>(x); case 11: return row_bcast<11>(x);
    case 12: return row_bcast<12>(x); case 13: return row_bcast<13>(x); case 14: return row_bcast<14>(x);
    default: return row_bcast<15>(x);
  }
}
__device__ __forceinline__ float row_prefix_prod(float x) {
  x *= dpp_row<0x111>(x, 1.f);
  x *= dpp_row<0x112>(x, 1.f);
  x *= dpp_row<0x114>(x, 1.f);
  x *= dpp_row<0x118>(x, 1.f);
  return x;
}
__device__ __forceinline__ float row_suffix_prod(float x) {
  x *= dpp_row<0x101>(x, 1.f);
  x *= dpp_row<0x102>(x, 1.f);
  x *= dpp_row<0x104>(x, 1.f);
  x *= dpp_row<0x108>(x, 1.f);
  return x;
}

// Sum over the four 16-lane rows of per-tile partials: p[i] is lane (nn, q4)'s
// partial of tile i; on return lane (nn, q4) holds the total of tile q4
// (v_permlane32_swap then v_permlane16_swap: a reduce-scatter in 3 swaps).
__device__ __forceinline__ float rows_reduce_scatter(float p0, float p1, float p2, float p3) {
  const auto r0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(p0), __float_as_uint(p2), false, false);
  const auto r1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(p1), __float_as_uint(p3), false, false);
  const float u0 = __uint_as_float(r0[0]) + __uint_as_float(r0[1]);
  const float u1 = __uint_as_float(r1[0]) + __uint_as_float(r1[1]);
  const auto r2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(u0), __float_as_uint(u1), false, false);
  return __uint_as_float(r2[0]) + __uint_as_float(r2[1]);
}

// max(m, |a|, |b|), NaN propagating (one v_maximum3_f32)
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(a)), __builtin_fabsf(b));
}

// raw bits of a gating input (f32, or the activation dtype) and their value
template <bool GATE_F32>
__device__ __forceinline__ uint32_t gate_bits(const uint8_t* p) {
  if constexpr (GATE_F32) return ld32(p);
  else return *(const uint16_t*)p;
}
template <bool GATE_F32>
__device__ __forceinline__ float gate_value(uint32_t bits) {
  if constexpr (GATE_F32) return __uint_as_float(bits);
  else return act_val(bits);
}

}  // namespace
}  // namespace gdnr
