// int4 group-64 GEMV of the decoder's projections on bf16 MFMA.
//
// Restates q4 / dot16 of engine/src/rec_mlx/kernels/megakernel.py:161-232:
// y[m][r] = Σ_g ( s[r][g] · Σ_{k∈g} q[r][k] x[m][k] + b[r][g] · Σ_{k∈g} x[m][k] )
// for an MLX affine 4-bit matrix (group 64: uint32 words of 8 codes, code e
// at bits 4e; bf16 scales and biases per (row, group)), bf16 x and a bf16 (or
// fp32) result.  The weights are repacked once (q4_pack_kernel) into records
// that one wavefront streams linearly.
//
// Packed layout: per 16-row tile and 128-element span, one 1152-byte record
//   [64 lanes][16 B]  codes: lane (r, kq) holds row r, elements 32kq .. 32kq+31
//                     of the span (four MLX words, unchanged)
//   [4 rg][2 gs][16 B] row group rg, group 2·span+gs: scales of rows 4rg..4rg+3
//                     (4 x bf16), then their biases (4 x bf16)
// Records are ordered [tile][span]; rows past N are zero.
//
// Arithmetic: the codes enter a bf16 MFMA 16x16x32 as 128 + q (exact: the
// nibble under the bf16 exponent of 128), x as bf16, products exact in fp32.
// The B operand's 16 columns are (vector m, group half gs): a column only
// holds x for the elements of its group, so one MFMA yields separate sums
// D = Σ (128 + q) x for the two groups of a span, and
// y += s·D + (b − 128 s)·X with X = Σ x over the group.
#include "q4.h"

namespace rec {

namespace {

constexpr int GV_WAVES = 4;   // waves per workgroup (more for matrices of few tiles)
constexpr int GV_ZERO = 256;  // zero bytes read by B lanes without data

// bf16 round-to-nearest-even of a finite or infinite float (NaN stays NaN).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  const uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

}  // namespace

// One workgroup of 64 threads per (tile, span) record.
__global__ __launch_bounds__(64) void q4_pack_kernel(const Q4PackArgs a) {
  const int l = threadIdx.x;
  const int64_t tile = blockIdx.y, span = blockIdx.x;
  const int64_t S = a.K / GV_SPAN, words = a.K / 8, groups = a.K / 64;
  uint8_t* rec = a.packed + (tile * S + span) * GV_REC;
  {
    const int64_t row = tile * 16 + (l & 15);
    v4i w = {0, 0, 0, 0};
    if (row < a.N) {
      const uint32_t* src = a.w + row * words + span * 16 + 4 * (l >> 4);
      w = (v4i){(int)src[0], (int)src[1], (int)src[2], (int)src[3]};
    }
    *(v4i*)(rec + 16 * l) = w;
  }
  if (l < 8) {
    const int rg = l >> 1, gs = l & 1;
    const int64_t g = 2 * span + gs;
    uint16_t v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t row = tile * 16 + 4 * rg + i;
      v[i] = row < a.N ? a.scales[row * groups + g] : 0;
      v[4 + i] = row < a.N ? a.biases[row * groups + g] : 0;
    }
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (int)(v[2 * i] | ((uint32_t)v[2 * i + 1] << 16));
    *(v4i*)(rec + 1024 + 16 * l) = o;
  }
}

// LDS: [M][S][4 slabs][4 kq][8 bf16] permuted x, a zero block, [M][K/64]
// group sums, and the waves' partial results ([4 waves][64 lanes][4 floats]).
__host__ __device__ size_t q4_gemv_red_offset(int M, int64_t K) {
  return ((size_t)M * K * 2 + GV_ZERO + (size_t)M * (K / 64) * 4 + 15) & ~(size_t)15;
}

static size_t lds_bytes_nw(int M, int64_t K, int nw) { return q4_gemv_red_offset(M, K) + (size_t)nw * 64 * 16; }

size_t q4_gemv_lds_bytes(int M, int64_t K) { return lds_bytes_nw(M, K, GV_WAVES); }

// WPT waves share one 16-row tile, wave p taking spans p, p + WPT, ...: small
// matrices (the attention projections, the experts) then still spread over
// every SIMD.  A workgroup of NW waves covers NW / WPT tiles.
template <int WPT, int NW>
__global__ __launch_bounds__(64 * NW) void q4_gemv_kernel(const Q4GemvArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = (int)(a.K / GV_SPAN), G = (int)(a.K / 64), M = a.M;
  char* xp = smem;
  char* zero = smem + (size_t)M * a.K * 2;
  float* xs = (float*)(zero + GV_ZERO);
  v4f* red = (v4f*)(smem + q4_gemv_red_offset(M, a.K));

  const int tile = blockIdx.x * (NW / WPT) + wave / WPT, part = wave % WPT;
  const bool live = tile * 16 < a.N;  // wave-uniform
  const int n_w = live && part < S ? (S - part + WPT - 1) / WPT : 0;  // spans of this wave

  const int c = lane & 15, q4 = lane >> 4;  // output column / row group, A-operand row / k quarter
  const int m = c >> 1, gs = c & 1;
  // B lanes of absent vectors, or of the other group of a span, read zeros
  const bool bval = m < M && (q4 >> 1) == gs;
  const char* bbase = bval ? xp + (((size_t)m * S) * 16 + q4) * 16 : zero + 16 * q4;
  const int bstride = bval ? 256 : 0;
  const bool xval = m < M;
  const float* xsum = xs + (xval ? m : 0) * G + gs;

  // Every span slot of the ring loads; slots past the last span load through
  // an empty resource (zeros, no memory access), so no load sits under a branch.
  const __amdgpu_buffer_rsrc_t R =
      make_rsrc(a.packed + (live ? (int64_t)tile * S * GV_REC : 0), live ? (int64_t)S * GV_REC : 0);
  const __amdgpu_buffer_rsrc_t R0 = make_rsrc(a.packed, 0);
  const uint32_t wl = 16 * lane, sl = 1024 + 16 * (2 * q4 + gs);

  constexpr int NB = 4;  // spans in flight
  v4i wbuf[NB], sbuf[NB];
#pragma unroll
  for (int i = 0; i < NB - 1; ++i) {
    const __amdgpu_buffer_rsrc_t r = i < n_w ? R : R0;
    wbuf[i] = ld128(r, wl, (part + WPT * i) * GV_REC);
    sbuf[i] = ld128(r, sl, (part + WPT * i) * GV_REC);
  }
  // (the first spans' loads above are in flight while x is staged)

  // ---- stage x: records of 8 elements in the MFMA's k order, and group sums ----
  // Thread order (m, span, gs, slab, kq & 1) puts the 8 records of one group
  // on 8 consecutive lanes.
  for (int t = tid; t < GV_ZERO / 4; t += 64 * NW) ((uint32_t*)zero)[t] = 0;
  const int nrec = M * S * 16;
  for (int t0 = 0; t0 < nrec; t0 += 64 * NW) {
    const int t = t0 + tid;
    float sum = 0.f;
    if (t < nrec) {
      const int k1 = t & 1, slab = (t >> 1) & 3, gs = (t >> 3) & 1, rest = t >> 4;
      const int span = rest % S, m = rest / S;
      const int kq = 2 * gs + k1;
      const int64_t e0 = (int64_t)span * GV_SPAN + 32 * kq + 8 * slab;
      const v4i in = *(const v4i*)(a.x + (int64_t)m * a.x_stride + e0);
      const uint32_t d0 = in[0], d1 = in[1], d2 = in[2], d3 = in[3];
      // element order of the A operand's unpack: 0, 4, 1, 5, 2, 6, 3, 7
      v4i o;
      o[0] = (int)__builtin_amdgcn_perm(d2, d0, 0x05040100u);
      o[1] = (int)__builtin_amdgcn_perm(d2, d0, 0x07060302u);
      o[2] = (int)__builtin_amdgcn_perm(d3, d1, 0x05040100u);
      o[3] = (int)__builtin_amdgcn_perm(d3, d1, 0x07060302u);
      *(v4i*)(xp + ((((size_t)m * S + span) * 4 + slab) * 4 + kq) * 16) = o;
      sum = ((bf16_lo(d0) + bf16_hi(d0)) + (bf16_lo(d1) + bf16_hi(d1))) +
            ((bf16_lo(d2) + bf16_hi(d2)) + (bf16_lo(d3) + bf16_hi(d3)));
    }
    sum = group8_sum(sum);
    if (t < nrec && (t & 7) == 0) {
      const int gs = (t >> 3) & 1, rest = t >> 4;
      xs[(rest / S) * G + 2 * (rest % S) + gs] = sum;
    }
  }
  __syncthreads();

  v4f y = {0.f, 0.f, 0.f, 0.f};
  const int n_pad = (n_w + NB - 1) / NB * NB;
  for (int i0 = 0; i0 < n_pad; i0 += NB) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int i = i0 + j, span = part + WPT * i;
      const __amdgpu_buffer_rsrc_t r = i + NB - 1 < n_w ? R : R0;
      wbuf[(j + NB - 1) % NB] = ld128(r, wl, (span + WPT * (NB - 1)) * GV_REC);
      sbuf[(j + NB - 1) % NB] = ld128(r, sl, (span + WPT * (NB - 1)) * GV_REC);
      if (i < n_w) {
        const v4i w4 = wbuf[j], sb = sbuf[j];
        const char* bp = bbase + span * bstride;
        v4f d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int slab = 0; slab < 4; ++slab) {
          const uint32_t w = (uint32_t)w4[slab];
          v4i av;
          av[0] = (int)and_or(w, 0x000f000fu, 0x43004300u);
          av[1] = (int)and_or(w >> 4, 0x000f000fu, 0x43004300u);
          av[2] = (int)and_or(w >> 8, 0x000f000fu, 0x43004300u);
          av[3] = (int)and_or(w >> 12, 0x000f000fu, 0x43004300u);
          const v4i bv = *(const v4i*)(bp + 64 * slab);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, av), __builtin_bit_cast(v8bf, bv), d,
                                                      0, 0, 0);
        }
        const float X = xval ? xsum[2 * span] : 0.f;
        const uint32_t s01 = (uint32_t)sb[0], s23 = (uint32_t)sb[1], b01 = (uint32_t)sb[2], b23 = (uint32_t)sb[3];
        const float sc[4] = {bf16_lo(s01), bf16_hi(s01), bf16_lo(s23), bf16_hi(s23)};
        const float bi[4] = {bf16_lo(b01), bf16_hi(b01), bf16_lo(b23), bf16_hi(b23)};
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = fmaf(fmaf(-128.f, sc[r], bi[r]), X, fmaf(sc[r], d[r], y[r]));
      }
    }
  }

  if constexpr (WPT > 1) {  // sum the partial results of the tile's waves
    red[wave * 64 + lane] = y;
    __syncthreads();
    if (part != 0) return;  // no barrier follows
#pragma unroll
    for (int p = 1; p < WPT; ++p) y += red[(wave + p) * 64 + lane];
  }
  if (!live) return;

  // the two group halves of a vector sit in lanes c, c ^ 1
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float mine = y[i];  // a copy: a bit_cast of a vector subscript reads element 0
    const int other = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, mine), 0xb1, 0xf, 0xf, false);  // quad_perm 1,0,3,2
    y[i] = mine + __builtin_bit_cast(float, other);
  }
  if (gs == 0 && m < M) {
    const int64_t r0 = (int64_t)tile * 16 + 4 * q4;
    if (a.out_dtype == DT_F32) {
      float* o = (float*)a.out + (int64_t)m * a.out_stride + r0;
      if (r0 + 3 < a.N) {
        *(v4f*)o = y;
      } else {
        for (int i = 0; i < 4; ++i)
          if (r0 + i < a.N) o[i] = y[i];
      }
    } else {
      uint16_t* o = (uint16_t*)a.out + (int64_t)m * a.out_stride + r0;
      const uint16_t h[4] = {f32_to_bf16(y[0]), f32_to_bf16(y[1]), f32_to_bf16(y[2]), f32_to_bf16(y[3])};
      if (r0 + 3 < a.N) {
        *(v2i*)o = (v2i){(int)(h[0] | ((uint32_t)h[1] << 16)), (int)(h[2] | ((uint32_t)h[3] << 16))};
      } else {
        for (int i = 0; i < 4; ++i)
          if (r0 + i < a.N) o[i] = h[i];
      }
    }
  }
}

hipError_t launch_q4_pack(const Q4PackArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)(a.K / GV_SPAN), (unsigned)((a.N + 15) / 16));
  hipLaunchKernelGGL(q4_pack_kernel, grid, dim3(64), 0, stream, a);
  return hipGetLastError();
}

template <int WPT, int NW = GV_WAVES>
hipError_t launch_q4_gemv_wpt(const Q4GemvArgs& a, int64_t tiles, hipStream_t stream) {
  constexpr int TPG = NW / WPT;  // tiles per workgroup
  const size_t lds = lds_bytes_nw(a.M, a.K, NW);
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)q4_gemv_kernel<WPT, NW>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((q4_gemv_kernel<WPT, NW>), dim3((unsigned)((tiles + TPG - 1) / TPG)), dim3(64 * NW), lds,
                     stream, a);
  return hipGetLastError();
}

hipError_t launch_q4_gemv(const Q4GemvArgs& a, hipStream_t stream) {
  const int64_t tiles = (a.N + 15) / 16, S = a.K / GV_SPAN;
  // fewest waves per tile that still give every SIMD (1024) two waves
  if (tiles >= 2048) return launch_q4_gemv_wpt<1>(a, tiles, stream);
  if (tiles >= 1024) return launch_q4_gemv_wpt<2>(a, tiles, stream);
  // Fewer tiles than CUs (o_proj 2048 x 4096, down_proj 2048 x 6144: 128
  // tiles): one tile per workgroup of 8 or 16 waves, so that each wave's
  // spans fit its ring of NB and are all in flight at once
  if (tiles < 256 && S > 4 * 4) {
    if (S <= 8 * 4 && lds_bytes_nw(a.M, a.K, 8) <= 160 * 1024) return launch_q4_gemv_wpt<8, 8>(a, tiles, stream);
    if (lds_bytes_nw(a.M, a.K, 16) <= 160 * 1024) return launch_q4_gemv_wpt<16, 16>(a, tiles, stream);
  }
  return launch_q4_gemv_wpt<4>(a, tiles, stream);
}

}  // namespace rec
