// Quantize-on-append: one wavefront turns one (b, h, t) row of 128 values into
// cache codes and scales.  Restates the append step of
// engine/src/rec_mlx/model.py:77-81 (quantize the new rows, write them at
// [prev:offset]) for this library's int8 / uint4 formats.  The arithmetic is
// IEEE float32 (correctly rounded divide, round-half-even rint, fp16 RNE) so
// codes and scales are bit-identical to the CPU restatement.
#pragma once

#include "common.h"

namespace rec {

struct RowSrc {
  const void* p;
  int dtype;
  int64_t sb, sh, st;  // element strides for batch, head, token (dim stride 1)
  int vec;             // p is 16-byte aligned and every stride a multiple of 4 elements
};

// Elements i, i+1 (i even) of a row as floats: one load when src.vec.
__device__ __forceinline__ void load2_as_float(const RowSrc& s, int64_t i, float& x0, float& x1) {
  if (s.vec) {
    if (s.dtype == DT_F32) {
      const v2f v = *(const v2f*)((const float*)s.p + i);
      x0 = v[0];
      x1 = v[1];
    } else {
      const uint32_t w = *(const uint32_t*)((const uint16_t*)s.p + i);
      if (s.dtype == DT_F16) {
        x0 = half_bits_to_float(w & 0xffffu);
        x1 = half_bits_to_float(w >> 16);
      } else {
        x0 = __builtin_bit_cast(float, w << 16);
        x1 = __builtin_bit_cast(float, w & 0xffff0000u);
      }
    }
  } else {
    x0 = load_as_float(s.p, i, s.dtype);
    x1 = load_as_float(s.p, i + 1, s.dtype);
  }
}

__device__ __forceinline__ int64_t row_base(const RowSrc& s, int b, int h, int t) {
  return (int64_t)b * s.sb + (int64_t)h * s.sh + (int64_t)t * s.st;
}

// int8 symmetric, one fp16 scale per row.  Lane l owns dims 2l, 2l+1.
// Returns the two codes; the caller stores them in its layout.
__device__ __forceinline__ void quantize_i8_pair(float x0, float x1, int& q0, int& q1, uint16_t& sbits) {
  float amax = wave_max(fmaxf(fabsf(x0), fabsf(x1)));
  sbits = half_bits_saturate(amax / 127.0f);
  const float s = half_bits_to_float(sbits);
  q0 = 0;
  q1 = 0;
  if (s != 0.0f) {
    q0 = (int)fminf(fmaxf(__builtin_rintf(x0 / s), -127.0f), 127.0f);
    q1 = (int)fminf(fmaxf(__builtin_rintf(x1 / s), -127.0f), 127.0f);
  }
}

// uint4 asymmetric per 32-dim group (16 lanes).  Lane l owns dims 2l, 2l+1.
__device__ __forceinline__ void quantize_u4_pair(float x0, float x1, int& q0, int& q1, uint16_t& sbits,
                                                 uint16_t& zbits) {
  float mn = row16_min(fminf(x0, x1)), mx = row16_max(fmaxf(x0, x1));
  mn = fminf(mn, 0.0f);
  mx = fmaxf(mx, 0.0f);
  sbits = half_bits_saturate((mx - mn) / 15.0f);
  const float s = half_bits_to_float(sbits);
  q0 = 0;
  q1 = 0;
  float z = 0.0f;
  if (s != 0.0f) {
    z = fminf(fmaxf(__builtin_rintf(-mn / s), 0.0f), 15.0f) + 0.0f;  // +0, never -0
    q0 = (int)fminf(fmaxf(__builtin_rintf(x0 / s) + z, 0.0f), 15.0f);
    q1 = (int)fminf(fmaxf(__builtin_rintf(x1 / s) + z, 0.0f), 15.0f);
  }
  zbits = float_to_half_bits(z);
}

// MLX-style affine quantization of one group of 64 (32 lanes, 2 elements
// each; restates mx.quantize's affine_quantize, mlx 0.32.0): the range is
// [min w, max(0, max w)], the extreme of larger magnitude (the edge) is made
// exact by stretching the step, codes are round((w - bias) / scale) clamped to
// [0, 2^BITS - 1] (round = half away from zero), scale and bias are stored as
// bf16 (F16: fp16, the keys' dtype of an fp16 model), rounded to nearest even.
// Float32 arithmetic with correctly rounded division, so the codes and bits
// match the CPU restatement exactly.
template <int BITS, bool F16 = false>
__device__ __forceinline__ void quantize_affine_pair(float x0, float x1, int& q0, int& q1, uint16_t& sbits,
                                                     uint16_t& bbits) {
  constexpr float n_bins = (float)((1 << BITS) - 1);
  float a, b;
  float mn = row16_min(fminf(x0, x1)), mx = row16_max(fmaxf(x0, x1));
  pair16(mn, a, b);  // the two rows of the 32-lane group
  mn = fminf(a, b);
  mx = max_xor16(mx);
  mx = fmaxf(mx, 0.0f);
  float scale = fmaxf((mx - mn) / n_bins, 1e-7f);
  const bool side = fabsf(mn) > fabsf(mx);
  scale = side ? scale : -scale;
  const float edge = side ? mn : mx;
  const float qe = __builtin_roundf(edge / scale);
  const bool at_zero = qe == 0.0f;
  scale = at_zero ? scale : edge / qe;
  const float bias = at_zero ? 0.0f : edge;
  q0 = (int)fminf(fmaxf(__builtin_roundf((x0 - bias) / scale), 0.0f), n_bins);
  q1 = (int)fminf(fmaxf(__builtin_roundf((x1 - bias) / scale), 0.0f), n_bins);
  sbits = F16 ? float_to_half_bits(scale) : float_to_bf16_bits(scale);
  bbits = F16 ? float_to_half_bits(bias) : float_to_bf16_bits(bias);
}

// Cache addressing in elements (bytes for codes), see the layout table in common.h.
__device__ __forceinline__ int64_t blk_base(int64_t bh, int64_t cap, int64_t t, int block_elems) {
  return (bh * (cap / BLOCK_T) + (t >> 5)) * block_elems;
}
// int8 K: byte of dim d
__device__ __forceinline__ int64_t k8_off(int64_t bh, int64_t cap, int64_t t, int d) {
  return blk_base(bh, cap, t, 4096) + (d >> 6) * 2048 + (t & 31) * 64 + (d & 63);
}
// int4 K: byte holding dims d, d+1 (d even).  Row t of the block is 64 bytes:
// [4 dim-groups of 16 per half][half m][8 bytes], so the 16 bytes a lane reads
// (dims 16g..16g+15 of both halves) are contiguous.
__device__ __forceinline__ int64_t k4_off(int64_t bh, int64_t cap, int64_t t, int d) {
  const int b = (d & 63) >> 1;  // byte inside the half
  return blk_base(bh, cap, t, 2048) + (t & 31) * 64 + (b >> 3) * 16 + (d >> 6) * 8 + (b & 7);
}
// int8 V: byte of dim d.  For d = 16n + c and position p = 8kg + e the byte
// sits at [n/2][c][kg][n%2][e]: the 8 bytes of (d, kg) for n = 2h, 2h+1 are
// one 16-byte run, so a lane reads its 64 bytes with four 16-byte loads.
__device__ __forceinline__ int64_t v8_off(int64_t bh, int64_t cap, int64_t t, int d) {
  const int p = block_pos((int)(t & 31)), n = d >> 4, c = d & 15;
  return blk_base(bh, cap, t, 4096) + (n >> 1) * 1024 + (c * 4 + (p >> 3)) * 16 + (n & 1) * 8 + (p & 7);
}
// int4 V: byte holding token t (and its neighbour t^1) of dim d.  For dim
// d = 16n + c and position p = 8kg + e the byte sits at
// [n/4][c][kg][n%4][e/2]: the 4 bytes of (d, kg) for n = 4h..4h+3 are one
// 16-byte run, so a lane reads its 32 bytes with two 16-byte loads.
__device__ __forceinline__ int64_t v4_off(int64_t bh, int64_t cap, int64_t t, int d) {
  const int p = block_pos((int)(t & 31)), n = d >> 4, c = d & 15;
  return blk_base(bh, cap, t, 2048) + (n >> 2) * 1024 + (c * 4 + (p >> 3)) * 16 + (n & 3) * 4 + ((p & 7) >> 1);
}
// per-token scale (int8)
__device__ __forceinline__ int64_t s8_off(int64_t bh, int64_t cap, int64_t t) {
  return blk_base(bh, cap, t, 32) + block_pos((int)(t & 31));
}
// per-(token, group) scale / zero-point (int4), at slot s4_slot(position)
__device__ __forceinline__ int64_t s4_off(int64_t bh, int64_t cap, int64_t t, int g) {
  return blk_base(bh, cap, t, 128) + g * 32 + s4_slot(block_pos((int)(t & 31)));
}

// affine scale (which 0) or bias (which 1) of group g (0..1), at slot s4_slot(position)
__device__ __forceinline__ int64_t sa_off(int64_t bh, int64_t cap, int64_t t, int which, int g) {
  return blk_base(bh, cap, t, 128) + which * 64 + g * 32 + s4_slot(block_pos((int)(t & 31)));
}

// Quantize row (b, h, t_src) of `src` and store it at cache position `pos`.
// kind 0 = K (row-major codes), kind 1 = V (token-blocked codes).  uint4 V
// rows share bytes with their neighbour, so they go through append_v4_pair.
template <int BITS>
__device__ __forceinline__ void append_row(const RowSrc& src, int b, int h, int t_src, int kind, void* codes,
                                           uint16_t* scales, uint16_t* zeros, int64_t bh, int64_t cap,
                                           int64_t pos, int lane) {
  const int64_t base = row_base(src, b, h, t_src);
  float x0, x1;
  load2_as_float(src, base + 2 * lane, x0, x1);
  if constexpr (is_a8(BITS)) {  // affine 8-bit keys: uint8 codes in the int8 K layout
    int q0, q1;
    uint16_t sb, bb;
    quantize_affine_pair<8, meta_f16(BITS)>(x0, x1, q0, q1, sb, bb);
    *(uint16_t*)((uint8_t*)codes + k8_off(bh, cap, pos, 2 * lane)) = (uint16_t)(q0 | (q1 << 8));
    if ((lane & 31) == 0) {
      scales[sa_off(bh, cap, pos, 0, lane >> 5)] = sb;
      scales[sa_off(bh, cap, pos, 1, lane >> 5)] = bb;
    }
  } else if constexpr (BITS == 8) {
    int q0, q1;
    uint16_t sb;
    quantize_i8_pair(x0, x1, q0, q1, sb);
    int8_t* c = (int8_t*)codes;
    if (kind == 0) {
      *(uint16_t*)(c + k8_off(bh, cap, pos, 2 * lane)) = (uint16_t)((q0 & 0xff) | ((q1 & 0xff) << 8));
    } else {
      c[v8_off(bh, cap, pos, 2 * lane)] = (int8_t)q0;
      c[v8_off(bh, cap, pos, 2 * lane + 1)] = (int8_t)q1;
    }
    if (lane == 0) scales[s8_off(bh, cap, pos)] = sb;
  } else {
    int q0, q1;
    uint16_t sb, zb;
    quantize_u4_pair(x0, x1, q0, q1, sb, zb);
    ((uint8_t*)codes)[k4_off(bh, cap, pos, 2 * lane)] = (uint8_t)(q0 | (q1 << 4));
    if ((lane & 15) == 0) {
      const int g = lane >> 4;
      scales[s4_off(bh, cap, pos, g)] = sb;
      zeros[s4_off(bh, cap, pos, g)] = zb;
    }
  }
}

// uint4 V: the byte shared by tokens (2p, 2p+1) (block positions p', p'^1 with
// the even token in the low nibble).  Rows whose flag is false keep the nibble
// already in the cache; each byte is written once.
// AFFINE: MLX-style affine group 64 (scale and bias in `scales`, `zeros`
// unused), F16: stored as fp16 rather than bf16.
template <bool AFFINE = false, bool F16 = false>
__device__ __forceinline__ void append_v4_pair(const RowSrc& src, int b, int h, int t_even, bool has_even,
                                               bool has_odd, uint8_t* codes, uint16_t* scales, uint16_t* zeros,
                                               int64_t bh, int64_t cap, int64_t pos_even, int lane) {
  int qe0 = 0, qe1 = 0, qo0 = 0, qo1 = 0;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const bool has = r == 0 ? has_even : has_odd;
    if (!has) continue;  // wave-uniform
    const int64_t base = row_base(src, b, h, t_even + r);
    float x0, x1;
    load2_as_float(src, base + 2 * lane, x0, x1);
    int q0, q1;
    uint16_t sb, zb;
    if constexpr (AFFINE) {
      quantize_affine_pair<4, F16>(x0, x1, q0, q1, sb, zb);
      if ((lane & 31) == 0) {
        scales[sa_off(bh, cap, pos_even + r, 0, lane >> 5)] = sb;
        scales[sa_off(bh, cap, pos_even + r, 1, lane >> 5)] = zb;
      }
    } else {
      quantize_u4_pair(x0, x1, q0, q1, sb, zb);
      if ((lane & 15) == 0) {
        const int g = lane >> 4;
        scales[s4_off(bh, cap, pos_even + r, g)] = sb;
        zeros[s4_off(bh, cap, pos_even + r, g)] = zb;
      }
    }
    if (r == 0) { qe0 = q0; qe1 = q1; } else { qo0 = q0; qo1 = q1; }
  }
  const int64_t a0 = v4_off(bh, cap, pos_even, 2 * lane);
  const int64_t a1 = v4_off(bh, cap, pos_even, 2 * lane + 1);
  uint8_t o0 = 0, o1 = 0;
  if (!(has_even && has_odd)) { o0 = codes[a0]; o1 = codes[a1]; }
  const int lo0 = has_even ? qe0 : (o0 & 15), hi0 = has_odd ? qo0 : (o0 >> 4);
  const int lo1 = has_even ? qe1 : (o1 & 15), hi1 = has_odd ? qo1 : (o1 >> 4);
  codes[a0] = (uint8_t)(lo0 | (hi0 << 4));
  codes[a1] = (uint8_t)(lo1 | (hi1 << 4));
}

// ---- whole blocks: one wavefront per 32-token block ----
// Lane (kg, c) = (lane / 16, lane % 16) owns dims 8c .. 8c+7 of the eight
// tokens 4kg .. 4kg+3 and 16+4kg .. 16+4kg+3, which are the block's positions
// 8kg .. 8kg+7: a row's 16-byte runs load as one contiguous row per 16 lanes, a
// quantization group lies in 16 (int8), 4 (uint4) or 8 (affine) adjacent lanes,
// and every code it makes leaves in runs of 64 contiguous bytes per 8 or 16
// lanes without an exchange between lanes.

// a / b for several a of one b, in fewer instructions than the IEEE sequence.
// y = RN(1/b).  q0 = RN(a y) is within 2 ulp of a/b, q1 = RN(q0 + (a - b q0) y)
// within one, and q2 = RN(q1 + (a - b q1) y) is RN(a/b) (Markstein 1990: y
// correctly rounded, q1 faithful, the residual exact in an fma) while nothing
// overflows or turns subnormal, which the callers see to.
//
// EASY: a and b have at most 11 significant bits (fp16 or bf16 inputs, an fp16
// step) and only the rounding of a/b to an integer matters.  A quotient that
// is not half an odd integer is at least 2^-14 away from the next one that is
// (a 2^k / b - m / 2 with 11-bit integers a, b), far beyond q1's error; one that
// is comes out of the residual step exactly.  So one step with the hardware's
// approximate reciprocal gives the same integer.
template <bool EASY>
struct Quotient {
  float b, y;
  __device__ __forceinline__ explicit Quotient(float b_) : b(b_), y(EASY ? __builtin_amdgcn_rcpf(b_) : 1.0f / b_) {}
  __device__ __forceinline__ float operator()(float a) const {
    float q = a * y;
    q = fmaf(fmaf(-q, b, a), y, q);
    if constexpr (!EASY) q = fmaf(fmaf(-q, b, a), y, q);
    return q;
  }
};
constexpr float QUOTIENT_MAX = 1e20f;  // magnitudes up to this keep every step above in range

template <int CTRL>
__device__ __forceinline__ float max_step(float x) { return fmaxf(x, dpp_f<CTRL>(x)); }
template <int CTRL>
__device__ __forceinline__ float min_step(float x) { return fminf(x, dpp_f<CTRL>(x)); }

// The codes of a lane's eight values of one token in the format of `BITS`,
// with the group's scale and zero-point / bias bits: the arithmetic of
// quantize_i8_pair, quantize_u4_pair and quantize_affine_pair.
template <int BITS, bool EASY>
__device__ __forceinline__ void quantize_eight(const float (&x)[8], int (&q)[8], uint16_t& sbits, uint16_t& zbits) {
  zbits = 0;
  if constexpr (BITS == 8) {
    float amax = fabsf(x[0]);
#pragma unroll
    for (int j = 1; j < 8; ++j) amax = fmaxf(amax, fabsf(x[j]));
    amax = row16_max(amax);
    sbits = half_bits_saturate(amax / 127.0f);
    const float s = half_bits_to_float(sbits);
    if (__any(!(amax <= QUOTIENT_MAX))) {  // (wave-uniform; infinities, NaN rows)
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = s != 0.0f ? (int)fminf(fmaxf(__builtin_rintf(x[j] / s), -127.0f), 127.0f) : 0;
    } else {
      const Quotient<EASY> d(s != 0.0f ? s : 1.0f);
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = s != 0.0f ? (int)fminf(fmaxf(__builtin_rintf(d(x[j])), -127.0f), 127.0f) : 0;
    }
  } else if constexpr (BITS == 4) {
    float mn = x[0], mx = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      mn = fminf(mn, x[j]);
      mx = fmaxf(mx, x[j]);
    }
    mn = min_step<DPP_XOR2>(min_step<DPP_XOR1>(mn));
    mx = max_step<DPP_XOR2>(max_step<DPP_XOR1>(mx));
    mn = fminf(mn, 0.0f);
    mx = fmaxf(mx, 0.0f);
    sbits = half_bits_saturate((mx - mn) / 15.0f);
    const float s = half_bits_to_float(sbits);
    float z = 0.0f;
    if (__any(!(mx - mn <= QUOTIENT_MAX))) {
      if (s != 0.0f) z = fminf(fmaxf(__builtin_rintf(-mn / s), 0.0f), 15.0f) + 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = s != 0.0f ? (int)fminf(fmaxf(__builtin_rintf(x[j] / s) + z, 0.0f), 15.0f) : 0;
    } else {
      const Quotient<EASY> d(s != 0.0f ? s : 1.0f);
      z = s != 0.0f ? fminf(fmaxf(__builtin_rintf(d(-mn)), 0.0f), 15.0f) + 0.0f : 0.0f;  // +0, never -0
#pragma unroll
      for (int j = 0; j < 8; ++j)
        q[j] = s != 0.0f ? (int)fminf(fmaxf(__builtin_rintf(d(x[j])) + z, 0.0f), 15.0f) : 0;
    }
    zbits = float_to_half_bits(z);
  } else {
    constexpr float n_bins = is_a8(BITS) ? 255.0f : 15.0f;
    float mn = x[0], mx = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
      mn = fminf(mn, x[j]);
      mx = fmaxf(mx, x[j]);
    }
    mn = min_step<DPP_HALF_MIRROR>(min_step<DPP_XOR2>(min_step<DPP_XOR1>(mn)));
    mx = max_step<DPP_HALF_MIRROR>(max_step<DPP_XOR2>(max_step<DPP_XOR1>(mx)));
    mx = fmaxf(mx, 0.0f);
    float scale = fmaxf((mx - mn) / n_bins, 1e-7f);
    const bool side = fabsf(mn) > fabsf(mx);
    scale = side ? scale : -scale;
    const float edge = side ? mn : mx;
    const float qe = __builtin_roundf(edge / scale);
    const bool at_zero = qe == 0.0f;
    scale = at_zero ? scale : edge / qe;
    const float bias = at_zero ? 0.0f : edge;
    if (__any(!(mx - mn <= QUOTIENT_MAX))) {
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = (int)fminf(fmaxf(__builtin_roundf((x[j] - bias) / scale), 0.0f), n_bins);
    } else {
      const Quotient<false> d(scale);  // at least about 1e-7 in magnitude, 24 bits
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = (int)fminf(fmaxf(__builtin_roundf(d(x[j] - bias)), 0.0f), n_bins);
    }
    sbits = meta_f16(BITS) ? float_to_half_bits(scale) : float_to_bf16_bits(scale);
    zbits = meta_f16(BITS) ? float_to_half_bits(bias) : float_to_bf16_bits(bias);
  }
}

// Eight consecutive elements of a row, as loaded.
template <bool F32>
struct Eight {
  v4i w[F32 ? 2 : 1];
  __device__ __forceinline__ void load(const RowSrc& s, int64_t i) {
    if constexpr (F32) {
      w[0] = *(const v4i*)((const float*)s.p + i);
      w[1] = *(const v4i*)((const float*)s.p + i + 4);
    } else {
      w[0] = *(const v4i*)((const uint16_t*)s.p + i);
    }
  }
  __device__ __forceinline__ void values(int dtype, float (&x)[8]) const {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (F32) {
        const int u = w[j >> 2][j & 3];
        x[j] = __builtin_bit_cast(float, u);
      } else {
        const uint32_t u = (uint32_t)w[0][j >> 1];
        if (dtype == DT_F16) x[j] = half_bits_to_float((j & 1) ? u >> 16 : u & 0xffffu);
        else x[j] = __builtin_bit_cast(float, (j & 1) ? u & 0xffff0000u : u << 16);
      }
    }
  }
};

// Quantize tokens t_src .. t_src + 31 of row (b, h) of `src` into the 32-token
// block at cache position `pos` (a multiple of 32).  IS_V: the V layouts.
template <int BITS, bool IS_V, bool F32>
__device__ __forceinline__ void append_block(const RowSrc& src, int b, int h, int t_src, void* codes, uint16_t* scales,
                                             uint16_t* zeros, int64_t bh, int64_t cap, int64_t pos, int lane) {
  const int kg = lane >> 4, c = lane & 15;
  const int64_t base = row_base(src, b, h, t_src) + 8 * c;
  Eight<F32> in[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) in[e].load(src, base + (int64_t)((e >> 2) * 16 + 4 * kg + (e & 3)) * src.st);
  uint16_t sb[8], zb[8];  // by position e
  uint32_t v[8][2];       // V codes of dim j: bytes (int8) or nibbles (4-bit) by position
  constexpr bool BYTE = BITS == 8 || is_a8(BITS);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float x[8];
    int q[8];
    in[e].values(src.dtype, x);
    quantize_eight<BITS, !F32>(x, q, sb[e], zb[e]);
    if constexpr (!IS_V) {
      const int64_t t = pos + (e >> 2) * 16 + 4 * kg + (e & 3);
      if constexpr (BYTE) {
        v2i o;
#pragma unroll
        for (int i = 0; i < 2; ++i)
          o[i] = (q[4 * i] & 0xff) | ((q[4 * i + 1] & 0xff) << 8) | ((q[4 * i + 2] & 0xff) << 16) | (q[4 * i + 3] << 24);
        *(v2i*)((uint8_t*)codes + k8_off(bh, cap, t, 8 * c)) = o;
      } else {
        uint32_t o = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) o |= (uint32_t)q[j] << (4 * j);
        *(uint32_t*)((uint8_t*)codes + k4_off(bh, cap, t, 8 * c)) = o;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if constexpr (BYTE) {
          const uint32_t o = (uint32_t)(q[j] & 0xff) << (8 * (e & 3));
          v[j][e >> 2] = (e & 3) ? v[j][e >> 2] | o : o;
        } else {
          const uint32_t o = (uint32_t)q[j] << (4 * e);
          v[j][0] = e ? v[j][0] | o : o;
        }
      }
    }
  }
  if constexpr (IS_V) {  // token 4kg is position 8kg of the block
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (BYTE)
        *(v2i*)((uint8_t*)codes + v8_off(bh, cap, pos + 4 * kg, 8 * c + j)) = (v2i){(int)v[j][0], (int)v[j][1]};
      else
        *(uint32_t*)((uint8_t*)codes + v4_off(bh, cap, pos + 4 * kg, 8 * c + j)) = v[j][0];
    }
  }
  // one lane per group stores the eight positions' scales: int8 in order, the
  // others in slot order (s4_slot: positions 0 4 1 5 2 6 3 7)
  constexpr int GROUP_LANES = BITS == 8 ? 16 : (is_affine(BITS) ? 8 : 4);
  if (c % GROUP_LANES == 0) {
    const int g = c / GROUP_LANES;
    v4i so, zo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int lo = BITS == 8 ? 2 * i : i, hi = BITS == 8 ? 2 * i + 1 : i + 4;
      so[i] = (int)(sb[lo] | ((uint32_t)sb[hi] << 16));
      zo[i] = (int)(zb[lo] | ((uint32_t)zb[hi] << 16));
    }
    if constexpr (BITS == 8) {
      *(v4i*)(scales + s8_off(bh, cap, pos + 4 * kg)) = so;
    } else if constexpr (is_affine(BITS)) {
      *(v4i*)(scales + sa_off(bh, cap, pos + 4 * kg, 0, g)) = so;
      *(v4i*)(scales + sa_off(bh, cap, pos + 4 * kg, 1, g)) = zo;
    } else {
      *(v4i*)(scales + s4_off(bh, cap, pos + 4 * kg, g)) = so;
      *(v4i*)(zeros + s4_off(bh, cap, pos + 4 * kg, g)) = zo;
    }
  }
}

}  // namespace rec
