// Quantize-on-append of L new K/V rows into the cache (gfx950).
//
// Restates MixedQuantizedKVCache.update_and_fetch's write step
// (engine/src/rec_mlx/model.py:76-81): rows [0, L) of the new keys/values are
// quantized and stored at cache positions [offset, offset + L).  One wavefront
// per whole 32-token block, and per row (4-bit V: per byte pair of positions)
// of the partial blocks at the ends, four per workgroup.  Formats: int8 / uint4
// (this library's), and MLX-style affine 8-bit K with 4-bit V.
#include <type_traits>

#include "kernels.h"

namespace rec {


// Workgroups per launch of the row kernels, at most: they stride over the
// rows, so any row count stays inside the dispatch's 32-bit thread count.
constexpr int64_t ROW_GRID_MAX = 1 << 20;

__host__ __device__ inline unsigned row_grid(int64_t rows) {
  const int64_t wgs = (rows + 3) / 4;
  return (unsigned)(wgs < ROW_GRID_MAX ? (wgs > 0 ? wgs : 1) : ROW_GRID_MAX);
}

// Which whole 32-token blocks the rows [offset, offset + L) cover: [first,
// end) in tokens (first == end: none).
struct BlockRange {
  int64_t first, end;
};
__host__ __device__ inline BlockRange whole_blocks(const AppendArgs& a) {
  const int64_t first = (a.offset + BLOCK_T - 1) / BLOCK_T * BLOCK_T, end = (a.offset + a.L) / BLOCK_T * BLOCK_T;
  return end > first ? BlockRange{first, end} : BlockRange{a.offset, a.offset};
}

// blockIdx.y: 0 = K, 1 = V.  A wavefront takes the whole blocks first, one
// each, then what is left at both ends, one row (4-bit V: byte pair) each.
// BLOCKS: 0 none (a kernel of its own, whose 28 registers leave room for eight
// waves per SIMD), 1 from 16-bit rows, 2 from fp32 rows.
template <int KB, int VB, int BLOCKS>
__global__ __launch_bounds__(256) void append_kernel(const AppendArgs a) {
  const int lane = threadIdx.x & 63;
  const int kind = blockIdx.y;
  constexpr bool V_PAIRS = VB != 8;
  const BlockRange r = BLOCKS ? whole_blocks(a) : BlockRange{a.offset, a.offset};
  // unit counts fit 32 bits: 2^32 rows of 256 bytes are more than the memory
  const uint32_t nblk = (uint32_t)((r.end - r.first) / BLOCK_T);
  // row units: `head` of them before the blocks
  const bool pairs = kind == 1 && V_PAIRS;
  const uint32_t head = nblk == 0 ? 0 : (uint32_t)(pairs ? r.first / 2 - (a.offset >> 1) : r.first - a.offset);
  const uint32_t skip = (pairs ? BLOCK_T / 2 : BLOCK_T) * nblk;
  const uint32_t rows = (uint32_t)(pairs ? a.v_units : (int64_t)a.L) - skip;
  const uint32_t blk_units = (uint32_t)a.B * a.Hkv * nblk, total = blk_units + (uint32_t)a.B * a.Hkv * rows;
  for (uint32_t unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); unit < total;
       unit += gridDim.x * 4) {
    if constexpr (BLOCKS != 0) {
      if (unit < blk_units) {
        constexpr bool F32 = BLOCKS == 2;
        const uint32_t bh = unit / nblk;
        const int64_t pos = r.first + (int64_t)(unit - bh * nblk) * BLOCK_T;
        const int b = (int)(bh / a.Hkv), h = (int)(bh % a.Hkv), t = (int)(pos - a.offset);
        if (kind == 0) append_block<KB, false, F32>(a.k, b, h, t, a.kq, a.ks, a.kz, bh, a.cap, pos, lane);
        else append_block<VB, true, F32>(a.v, b, h, t, a.vq, a.vs, a.vz, bh, a.cap, pos, lane);
        continue;
      }
    }
    const uint32_t i = unit - blk_units, bh = i / rows;
    int64_t u = i - bh * rows;
    if (u >= head) u += skip;
    const int b = (int)(bh / a.Hkv), h = (int)(bh % a.Hkv);
    if (kind == 0) {
      append_row<KB>(a.k, b, h, (int)u, 0, a.kq, a.ks, a.kz, bh, a.cap, a.offset + u, lane);
    } else if constexpr (VB == 8) {
      append_row<8>(a.v, b, h, (int)u, 1, a.vq, a.vs, nullptr, bh, a.cap, a.offset + u, lane);
    } else {
      const int64_t pos_even = ((a.offset >> 1) + u) * 2;
      const bool has_even = pos_even >= a.offset && pos_even < a.offset + a.L;
      const bool has_odd = pos_even + 1 >= a.offset && pos_even + 1 < a.offset + a.L;
      append_v4_pair<is_a4(VB), meta_f16(VB)>(a.v, b, h, (int)(pos_even - a.offset), has_even, has_odd,
                                              (uint8_t*)a.vq, a.vs, a.vz, bh, a.cap, pos_even, lane);
    }
  }
}

// Dequantize cache rows [0, T) to bf16 (B, Hkv, T, 128) tensors: the
// reference's prefill branch dequantizes the cache to the query dtype before
// its attention (engine/src/rec_mlx/model.py:194-195).  One wavefront per row,
// lane l owns dims 2l, 2l+1; x̂ is formed in float32 exactly as the CPU
// restatement does (int8 q·s, uint4 (q - z)·s, affine q·s + b), then rounded
// to bf16.  blockIdx.y: 0 = K, 1 = V.
template <int BITS>
__device__ __forceinline__ void dequant_pair(const void* codes, const uint16_t* scales, const uint16_t* zeros,
                                             bool is_v, int64_t bh, int64_t cap, int64_t t, int lane, float& x0,
                                             float& x1) {
  const int d = 2 * lane;
  if constexpr (BITS == 8) {
    const int8_t* c = (const int8_t*)codes;
    const int q0 = is_v ? c[v8_off(bh, cap, t, d)] : c[k8_off(bh, cap, t, d)];
    const int q1 = is_v ? c[v8_off(bh, cap, t, d + 1)] : c[k8_off(bh, cap, t, d + 1)];
    const float s = half_bits_to_float(scales[s8_off(bh, cap, t)]);
    x0 = (float)q0 * s;
    x1 = (float)q1 * s;
  } else if constexpr (BITS == 4) {
    const uint8_t* c = (const uint8_t*)codes;
    int q0, q1;
    if (is_v) {
      const int p = block_pos((int)(t & 31));
      const uint8_t b0 = c[v4_off(bh, cap, t, d)], b1 = c[v4_off(bh, cap, t, d + 1)];
      q0 = (p & 1) ? b0 >> 4 : b0 & 15;
      q1 = (p & 1) ? b1 >> 4 : b1 & 15;
    } else {
      const uint8_t b = c[k4_off(bh, cap, t, d)];
      q0 = b & 15;
      q1 = b >> 4;
    }
    const int g = d >> 5;
    const float s = half_bits_to_float(scales[s4_off(bh, cap, t, g)]);
    const float z = half_bits_to_float(zeros[s4_off(bh, cap, t, g)]);
    x0 = ((float)q0 - z) * s;
    x1 = ((float)q1 - z) * s;
  } else {  // affine: 8-bit keys (uint8 in the int8 K layout), 4-bit values (uint4 in the int4 V layout)
    const uint8_t* c = (const uint8_t*)codes;
    int q0, q1;
    if constexpr (is_a8(BITS)) {
      q0 = c[k8_off(bh, cap, t, d)];
      q1 = c[k8_off(bh, cap, t, d + 1)];
    } else {
      const int p = block_pos((int)(t & 31));
      const uint8_t b0 = c[v4_off(bh, cap, t, d)], b1 = c[v4_off(bh, cap, t, d + 1)];
      q0 = (p & 1) ? b0 >> 4 : b0 & 15;
      q1 = (p & 1) ? b1 >> 4 : b1 & 15;
    }
    const int g = d >> 6;
    const float s = meta_bits<meta_f16(BITS)>(scales[sa_off(bh, cap, t, 0, g)]);
    const float b = meta_bits<meta_f16(BITS)>(scales[sa_off(bh, cap, t, 1, g)]);
    x0 = (float)q0 * s + b;
    x1 = (float)q1 * s + b;
  }
}

template <int KB, int VB>
__global__ __launch_bounds__(256) void dequant_kernel(const DequantArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t total = (int64_t)a.B * a.Hkv * a.T;
  const bool is_v = blockIdx.y == 1;
  for (int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); row < total; row += (int64_t)gridDim.x * 4) {
    const int64_t bh = row / a.T, t = row % a.T;
    float x0, x1;
    if (!is_v) dequant_pair<KB>(a.kq, a.ks, a.kz, false, bh, a.cap, t, lane, x0, x1);
    else dequant_pair<VB>(a.vq, a.vs, a.vz, true, bh, a.cap, t, lane, x0, x1);
    uint16_t* o = (is_v ? a.v_out : a.k_out) + row * HEAD_DIM + 2 * lane;
    *(uint32_t*)o = (uint32_t)float_to_bf16_bits(x0) | ((uint32_t)float_to_bf16_bits(x1) << 16);
  }
}

hipError_t launch_dequant(int kb, int vb, const DequantArgs& a, hipStream_t stream) {
  const int64_t rows = (int64_t)a.B * a.Hkv * a.T;
  const dim3 grid(row_grid(rows), 2), block(256);
  if (kb == 8 && vb == 8) hipLaunchKernelGGL((dequant_kernel<8, 8>), grid, block, 0, stream, a);
  else if (kb == 8 && vb == 4) hipLaunchKernelGGL((dequant_kernel<8, 4>), grid, block, 0, stream, a);
  else if (kb == 4 && vb == 8) hipLaunchKernelGGL((dequant_kernel<4, 8>), grid, block, 0, stream, a);
  else if (kb == FMT_A8 && vb == FMT_A4) hipLaunchKernelGGL((dequant_kernel<FMT_A8, FMT_A4>), grid, block, 0, stream, a);
  else if (kb == FMT_A8H && vb == FMT_A4H)
    hipLaunchKernelGGL((dequant_kernel<FMT_A8H, FMT_A4H>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((dequant_kernel<4, 4>), grid, block, 0, stream, a);
  return hipGetLastError();
}

// Zero a word range (graph-safe replacement for hipMemsetAsync).
__global__ void fill_zero_kernel(uint32_t* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

hipError_t launch_append(int kb, int vb, const AppendArgs& a, hipStream_t stream) {
  // Whole blocks from 192 per tensor on, where the rows load as 16-byte runs.
  // One row per wavefront stores a V row as 128 single bytes 16 apart and
  // spends 80 instructions on a row's two divisions per lane; a block's stores
  // are 64-byte runs, its divisions two or four multiply-adds.  4 KV heads,
  // bf16, µs, rows → blocks: int8 32,768 tokens 86.7 → 26.1 (101 MB, 3.9 TB/s),
  // 2,048 (256 blocks) 9.1 → 6.6; uint4 84.2 → 26.2, 8.2 → 7.0; affine 93.3 →
  // 31.5, 8.9 → 7.8.  Fewer blocks leave SIMDs idle behind one block's 6 µs
  // chain: 1,000 tokens (124 blocks) 5.4 in rows, 6.5 in blocks, affine 5.3, 7.8.
  const BlockRange r = whole_blocks(a);
  int64_t nblk = (r.end - r.first) / BLOCK_T;
  if (!a.k.vec || !a.v.vec || (int64_t)a.B * a.Hkv * nblk < 192) nblk = 0;
  const int64_t k_units = a.L - (BLOCK_T - 1) * nblk;
  const int64_t v_units = a.v_units - (vb == 8 ? BLOCK_T - 1 : BLOCK_T / 2 - 1) * nblk;
  const int64_t rows = (int64_t)a.B * a.Hkv * (k_units > v_units ? k_units : v_units);
  const dim3 grid(row_grid(rows), 2), block(256);
  const auto go = [&](auto blocks) {
    constexpr int BL = decltype(blocks)::value;
    if (kb == 8 && vb == 8) hipLaunchKernelGGL((append_kernel<8, 8, BL>), grid, block, 0, stream, a);
    else if (kb == 8 && vb == 4) hipLaunchKernelGGL((append_kernel<8, 4, BL>), grid, block, 0, stream, a);
    else if (kb == 4 && vb == 8) hipLaunchKernelGGL((append_kernel<4, 8, BL>), grid, block, 0, stream, a);
    else if (kb == FMT_A8 && vb == FMT_A4)
      hipLaunchKernelGGL((append_kernel<FMT_A8, FMT_A4, BL>), grid, block, 0, stream, a);
    else if (kb == FMT_A8H && vb == FMT_A4H)
      hipLaunchKernelGGL((append_kernel<FMT_A8H, FMT_A4H, BL>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((append_kernel<4, 4, BL>), grid, block, 0, stream, a);
  };
  if (nblk == 0) go(std::integral_constant<int, 0>{});
  else if (a.k.dtype == DT_F32) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 1>{});
  return hipGetLastError();
}

// A plain streaming read of n16 16-byte chunks: consecutive lanes read
// consecutive chunks (1 KB per wavefront and load), four loads in flight per
// lane, grid-stride.  The XOR of everything read is stored only when it hits a
// fixed value, so the loads stay live without a store per lane.  The read floor
// the decode kernels are measured against.
__global__ __launch_bounds__(256) void stream_read_kernel(const v4i* p, int64_t n16, uint32_t* out) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  v4i acc = {0, 0, 0, 0};
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const v4i a = __builtin_nontemporal_load(p + i), b = __builtin_nontemporal_load(p + i + stride);
    const v4i c = __builtin_nontemporal_load(p + i + 2 * stride), d = __builtin_nontemporal_load(p + i + 3 * stride);
    acc ^= a ^ b ^ c ^ d;
  }
  for (; i < n16; i += stride) acc ^= __builtin_nontemporal_load(p + i);
  const uint32_t x = (uint32_t)(acc[0] ^ acc[1] ^ acc[2] ^ acc[3]);
  if (x == 0x9e3779b9u) out[blockIdx.x] = x;
}

hipError_t launch_stream_read(const void* p, int64_t n16, int workgroups, uint32_t* out, hipStream_t stream) {
  hipLaunchKernelGGL(stream_read_kernel, dim3(workgroups), dim3(256), 0, stream, (const v4i*)p, n16, out);
  return hipGetLastError();
}

hipError_t launch_fill_zero(uint32_t* p, int64_t words, hipStream_t stream) {
  if (words <= 0) return hipSuccess;
  const int64_t wgs = (words + 255) / 256;
  hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)(wgs < ROW_GRID_MAX ? wgs : ROW_GRID_MAX)), dim3(256), 0, stream,
                     p, words);
  return hipGetLastError();
}

}  // namespace rec
