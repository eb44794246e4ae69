// What the int4 projection kernels share: the packed record (its layout is
// described in gemv.hip), the unpack of its codes and the output store.
#pragma once

#include "kernels.h"

namespace rec {

constexpr int GV_SPAN = 128;        // elements per span
constexpr int GV_REC = 1024 + 128;  // bytes per (tile, span) record

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// Two floats as bf16, rounded to nearest even by the hardware conversion.
__device__ __forceinline__ int bf16_pair(float x, float y) {
  return (int)((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x) |
               ((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)y) << 16));
}

// The bits of bf16 128 twice, in a register the compiler takes for unknown, so
// that it forms (x & mask) | base as one v_and_or_b32 with the mask in a scalar
// register.  (Not the and_or of common.h: an instruction written as asm may be
// given the registers of a matrix product's unused results, which the product
// then writes late -- the compiler keeps its own instructions clear of that.)
__device__ __forceinline__ uint32_t code_base() {
  uint32_t b = 0x43004300u;
  asm volatile("" : "+v"(b));
  return b;
}

// Eight 4-bit codes of one word as eight bf16 values 128 + q, one and-or
// per pair: codes d and d + 4 (element order 0, 4, 1, 5, 2, 6, 3, 7, the
// order x is staged in).
__device__ __forceinline__ v8bf unpack_codes(uint32_t w, uint32_t base) {
  v4i o;
  o[0] = (int)((w & 0x000f000fu) | base);
  o[1] = (int)(((w >> 4) & 0x000f000fu) | base);
  o[2] = (int)(((w >> 8) & 0x000f000fu) | base);
  o[3] = (int)(((w >> 12) & 0x000f000fu) | base);
  return __builtin_bit_cast(v8bf, o);
}

// The same codes in their own order 0, 1, .., 7 (x as it lies in memory): two
// more instructions than above, one byte permute per pair.
__device__ __forceinline__ v8bf unpack_codes_in_order(uint32_t w, uint32_t base) {
  const uint32_t u = w >> 4;  // byte j: code 2j of w, code 2j + 1 of u
  v4i o;
  o[0] = (int)((__builtin_amdgcn_perm(u, w, 0x0c040c00u) & 0x000f000fu) | base);
  o[1] = (int)((__builtin_amdgcn_perm(u, w, 0x0c050c01u) & 0x000f000fu) | base);
  o[2] = (int)((__builtin_amdgcn_perm(u, w, 0x0c060c02u) & 0x000f000fu) | base);
  o[3] = (int)((__builtin_amdgcn_perm(u, w, 0x0c070c03u) & 0x000f000fu) | base);
  return __builtin_bit_cast(v8bf, o);
}

// Rows n0 .. n0 + 3 (below N) of output vector m.
__device__ __forceinline__ void q4_store(const Q4GemmArgs& a, int m, int64_t n0, const v4f& v) {
  if (a.out_dtype == DT_F32) {
    float* o = (float*)a.out + (int64_t)m * a.out_stride + n0;
    if (n0 + 3 < a.N) {
      *(v4f*)o = v;
    } else {
      for (int i = 0; i < 4; ++i)
        if (n0 + i < a.N) o[i] = v[i];
    }
  } else {
    uint16_t* o = (uint16_t*)a.out + (int64_t)m * a.out_stride + n0;
    const v2i h = {bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
    if (n0 + 3 < a.N) {
      *(v2i*)o = h;
    } else {
      for (int i = 0; i < 4; ++i)
        if (n0 + i < a.N) o[i] = (uint16_t)((uint32_t)h[i >> 1] >> (16 * (i & 1)));
    }
  }
}

// Rows n0 .. n0 + 7 (below N, n0 < N) of output vector m.
__device__ __forceinline__ void q4_store8(const Q4GemmArgs& a, int m, int64_t n0, const v4f& lo, const v4f& hi) {
  if (a.out_dtype == DT_F32 || n0 + 7 >= a.N) {
    q4_store(a, m, n0, lo);
    if (n0 + 4 < a.N) q4_store(a, m, n0 + 4, hi);
  } else {
    const v4i o = {bf16_pair(lo[0], lo[1]), bf16_pair(lo[2], lo[3]), bf16_pair(hi[0], hi[1]), bf16_pair(hi[2], hi[3])};
    *(v4i*)((uint16_t*)a.out + (int64_t)m * a.out_stride + n0) = o;
  }
}

}  // namespace rec
