// Many vectors: the int4 projections of a prefill chunk, a short turn or a
// batch of sequences (M rows of x), over the records of gemv.hip.
//
// A GEMM on bf16 MFMA 16x16x32 with exact products: codes enter as 128 + q, x
// as bf16, sums run in fp32 over one 64-element group at a time.  A k-step
// covers 32 consecutive elements of one group -- lane (r, kq) takes word
// 4t + kq of row r, dword kq of record lane r + 16t -- so the two groups of a
// span accumulate apart.
#include "dma.h"
#include "q4.h"

namespace rec {

// Z[g][m] = −128 Σ x[m][64g .. 64g+63] in fp32, 32 vectors of one span per
// workgroup and turn: 16 lanes per vector's 256 bytes, eight of them per
// group; the sums leave through LDS as two 128-byte rows.
constexpr int64_t XSUM_GRID_MAX = 1 << 20;  // keeps the launch's thread count in 32 bits
__global__ __launch_bounds__(256) void q4_xsum_kernel(const Q4GemmArgs a) {
  __shared__ float z[2][2][32];
  const int t = threadIdx.x;
  const int64_t S = a.K / GV_SPAN, n = (((int64_t)a.M + 31) / 32) * S;
  int buf = 0;
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x, buf ^= 1) {
    const int64_t span = i % S, m0 = i / S * 32;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int v = 16 * j + (t >> 4);
      const int64_t m = min(m0 + v, (int64_t)a.M - 1);
      const v4i w = *(const v4i*)(a.x + m * a.x_stride + span * GV_SPAN + 8 * (t & 15));  // 16-byte aligned rows
      const uint32_t d0 = w[0], d1 = w[1], d2 = w[2], d3 = w[3];
      const float s = group8_sum(((bf16_lo(d0) + bf16_hi(d0)) + (bf16_lo(d1) + bf16_hi(d1))) +
                                 ((bf16_lo(d2) + bf16_hi(d2)) + (bf16_lo(d3) + bf16_hi(d3))));
      if ((t & 7) == 0) z[buf][(t >> 3) & 1][v] = -128.f * s;
    }
    __syncthreads();  // (two buffers: the next turn's writes need no barrier of their own)
    if (t < 64 && m0 + (t & 31) < a.M) a.xsum[(2 * span + (t >> 5)) * a.M + m0 + (t & 31)] = z[buf][t >> 5][t & 31];
  }
}

constexpr int GM_VECS = 64;   // vectors per workgroup: four 16-column tiles
constexpr int GM_TILES = 16;  // 16-row tiles per workgroup (256 rows): four per wave
// One group's LDS: x, the waves' codes and scale blocks, Z.
constexpr int GM_X = GM_VECS * 128;
constexpr int GM_W = 4 * 512;  // per wave: four tiles' codes
constexpr int GM_SC = 256;     // per wave: four tiles' scale blocks
constexpr int GM_STAGE = GM_X + 4 * (GM_W + GM_SC) + GM_VECS * 4;

// Workgroup: 256 rows against 64 vectors, KS groups of four waves.  A wave
// owns 64 rows (four row tiles) against all 64 vectors, so an x operand read
// from LDS feeds four row tiles; set h of the waves takes the 64-element groups
// h, h + KS, ...  A group's x, codes, scales and Z come into LDS by direct
// loads issued a whole step ahead (two buffers, one barrier per step); the
// 16-byte pieces of vector v lie at piece ^ (v / 2 & 7), so that the 16 rows of
// an operand read fall on distinct banks.
//
// The SIMD's vector instructions hardly overlap its matrix products here, so
// there are as few as possible: x is the A operand, which leaves lane (r, kq)
// with row r's products with the vectors 4kq .. 4kq+3, one scale per lane; the
// products' accumulators start at Z = −128 Σx, so that they end as D = Σ q x
// without a correction; y += s·D is one multiply-add per value; and the terms
// b·Σx of all groups are matrix products of their own before the loop, eight
// groups each: [b' b' b' 0] of row r, b' = −b/128 (exact in bf16), against
// [h m l 0] of a vector, Z = h + m + l cut into three bf16 values (its 24 bits).
//
// At the end the two sets exchange half of their sums through LDS, and the
// waves turn their tiles there into runs of consecutive rows.
//
// Bound by the SIMD's issue: per wave and group 32 matrix products (512 cycles)
// and 153 vector instructions (612 cycles), which overlap little (counters:
// matrix cores busy 36% of the cycles).  2,000 vectors, with the group sums:
// 5,120 x 2,048 92 → 67 µs, 2,048 x 4,096 66 → 49, 12,288 x 2,048 181 → 129 (779
// TFLOP/s), 2,048 x 6,144 94 → 71.  Its error against float64 is half the one
// before (5e-7 against 1e-6), as the codes' offset of 128 is taken off inside
// each group.  Not faster: the next span's operands through registers (a
// round trip to memory exposed per half span, 197 µs at 12,288 x 2,048), a
// whole span per step (two workgroups per CU instead of three, 136), the
// b·Σx and offset terms as vector instructions (134 with 507 of them per
// span for 289).
template <int KS>
__global__ __launch_bounds__(256 * KS, KS == 1 ? 3 : 2) void q4_gemm_kernel(const Q4GemmArgs a) {
  // (the epilogue's exchange and row images need more than the stages)
  constexpr int NRT = 4 / KS;          // row tiles a wave stores
  constexpr int PITCH = 16 * NRT + 4;  // floats per vector of its LDS image
  constexpr int XCHG = KS == 1 ? 0 : 65536, EPI = XCHG + 4 * KS * 16 * PITCH * 4;
  __shared__ __attribute__((aligned(1024))) char sm[EPI > KS * 2 * GM_STAGE ? EPI : KS * 2 * GM_STAGE];
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int64_t tiles = (a.N + 15) / 16;
  const int S = (int)(a.K / GV_SPAN);
  const int r = lane & 15, kq = lane >> 4;

  // Workgroup i runs on XCD i % 8: each XCD takes a run of consecutive blocks,
  // ordered in bands of four row blocks, vectors next, so that the 32 blocks
  // an XCD computes at a time share four row blocks and eight vector blocks in
  // its L2.
  int bx, by;
  {
    const uint32_t nbx = (uint32_t)((tiles + GM_TILES - 1) / GM_TILES);
    const uint32_t nby = (uint32_t)((a.M + GM_VECS - 1) / GM_VECS), n = nbx * nby;
    const uint32_t xcd = blockIdx.x % 8, q = n / 8, rem = n % 8;
    const uint32_t l = xcd * q + min(xcd, rem) + blockIdx.x / 8;
    const uint32_t band = l / (4 * nby), in = l - band * 4 * nby, w = min(4u, nbx - 4 * band);
    bx = (int)(4 * band + in % w);
    by = (int)(in / w);
  }
  const int m0 = by * GM_VECS;
  const int rows = min(GM_VECS, a.M - m0);  // vectors of this workgroup (>= 1)
  const int64_t tile0 = (int64_t)bx * GM_TILES + 4 * wave;

  // Direct loads: vectors past M and tiles past the matrix load the last one
  // again (their sums are not stored).
  const char* xg = uniform_ptr(a.x + (int64_t)m0 * a.x_stride);
  uint32_t xv[2];  // the wave's vectors 16 wave + 8 j + lane / 8
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int v = 16 * wave + 8 * j + (lane >> 3);
    xv[j] = (uint32_t)((int64_t)min(v, rows - 1) * a.x_stride * 2) + 16 * ((lane & 7) ^ (v >> 1 & 7));
  }
  const char* zg = uniform_ptr(a.xsum + m0);
  const uint32_t zv = 4 * (uint32_t)min(lane, rows - 1);
  const uint8_t* wg[2];  // tiles 2 j + lane / 32
#pragma unroll
  for (int j = 0; j < 2; ++j)
    wg[j] = a.packed + min(tile0 + 2 * j + (lane >> 5), tiles - 1) * S * GV_REC + 16 * (lane & 31);
  // lanes 0-15: row group lane % 4 of tile lane / 4
  const uint8_t* cg = a.packed + min(tile0 + (lane >> 2 & 3), tiles - 1) * S * GV_REC + 1024 + 32 * (lane & 3);
  const uint32_t sm0 = lds_address(sm) + half * 2 * GM_STAGE;
  const auto load = [&](int buf, int g) {
    const uint32_t l0 = sm0 + buf * GM_STAGE;
    const int64_t rec = (int64_t)(g >> 1) * GV_REC;
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(l0 + (2 * wave + j) * 1024, xg + 128 * (int64_t)g, xv[j]);
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(l0 + GM_X + wave * GM_W + j * 1024, wg[j] + rec + 512 * (g & 1));
    if (lane < 16) dma16(l0 + GM_X + 4 * GM_W + wave * GM_SC, cg + rec + 16 * (g & 1));
    if (wave == 0) dma4(l0 + GM_X + 4 * (GM_W + GM_SC), zg + (int64_t)g * a.M * 4, zv);
  };

  const uint32_t base = code_base();
  v4f y[4][4];  // [row tile][vector tile]
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int vt = 0; vt < 4; ++vt) y[rt][vt] = (v4f){0.f, 0.f, 0.f, 0.f};

  const int G = 2 * S, steps = (G + KS - 1) / KS;
  if (half < G) load(0, half);

  {  // the b·Σx terms, groups 8j .. 8j + 7 (lane kq: 8j + 2kq, + 1), j = half, half + KS, ...
    __amdgpu_buffer_rsrc_t R[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const bool live = tile0 + rt < tiles;
      R[rt] = make_rsrc(a.packed + (live ? (tile0 + rt) * S * GV_REC : 0), live ? (int64_t)S * GV_REC : 0);
    }
    const uint32_t bl = GV_REC * kq + 1024 + 32 * (r >> 2) + 8 + 2 * (r & 3);
    const uint32_t zl = 4 * ((uint32_t)(2 * kq) * (uint32_t)a.M + (uint32_t)r), zM = 4 * (uint32_t)a.M;
    const int octs = (S + 3) / 4;
#pragma unroll 2
    for (int j = half; j < octs; j += KS) {
      // groups and vectors past the last read zeros or other vectors' sums
      const __amdgpu_buffer_rsrc_t RZ =
          make_rsrc(a.xsum + (int64_t)8 * j * a.M + m0, ((int64_t)min(8, 2 * S - 8 * j) * a.M - m0) * 4);
      uint32_t bb[4][2];
      float z[4][2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
          bb[rt][e] = __builtin_amdgcn_raw_buffer_load_b16(R[rt], bl + 16 * e, (uint32_t)(4 * j) * GV_REC, 0);
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) z[vt][e] = __builtin_bit_cast(float, ld32<0>(RZ, zl + zM * e + 64 * vt, 0));
      }
      v8bf av[4];
#pragma unroll
      for (int vt = 0; vt < 4; ++vt) {
        v4i o;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const uint32_t h = __builtin_bit_cast(uint32_t, z[vt][e]) & 0xffff0000u;
          const float t = z[vt][e] - __builtin_bit_cast(float, h);
          const uint32_t m = __builtin_bit_cast(uint32_t, t) & 0xffff0000u;
          const uint32_t l = __builtin_bit_cast(uint32_t, t - __builtin_bit_cast(float, m));
          o[2 * e] = (int)(m | (h >> 16));
          o[2 * e + 1] = (int)(l >> 16);
        }
        av[vt] = __builtin_bit_cast(v8bf, o);
      }
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        v4i o;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const uint32_t u = __builtin_bit_cast(uint32_t, -0.0078125f * bf16_lo(bb[rt][e]));
          o[2 * e] = (int)(u | (u >> 16));
          o[2 * e + 1] = (int)(u >> 16);
        }
        const v8bf bv = __builtin_bit_cast(v8bf, o);
#pragma unroll
        for (int vt = 0; vt < 4; ++vt)
          y[rt][vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[vt], bv, y[rt][vt], 0, 0, 0);
      }
    }
  }

#pragma unroll 1
  for (int st = 0; st < steps; ++st) {
    const int g = st * KS + half;
    dma_wait();
    __syncthreads();
    if (g + KS < G) load((st & 1) ^ 1, g + KS);
    if (g < G) {  // wave-uniform
      const char* l0 = sm + half * 2 * GM_STAGE + (st & 1) * GM_STAGE;
      const char* wp = l0 + GM_X + wave * GM_W + 16 * r + 4 * kq;
      const char* cp = l0 + GM_X + 4 * GM_W + wave * GM_SC + 16 * (r >> 2) + 2 * (r & 3);
      const char* zp = l0 + GM_X + 4 * (GM_W + GM_SC) + 16 * kq;
      const char* xp = l0 + r * 128;
      const int p0 = 16 * (kq ^ (r >> 1)), p1 = 16 * ((4 + kq) ^ (r >> 1));
      v8bf wv[4][2];
      float sc[4];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        wv[rt][0] = unpack_codes_in_order(*(const uint32_t*)(wp + 512 * rt), base);
        wv[rt][1] = unpack_codes_in_order(*(const uint32_t*)(wp + 512 * rt + 256), base);
        sc[rt] = bf16_lo(*(const uint16_t*)(cp + 64 * rt));
      }
#pragma unroll
      for (int vt = 0; vt < 4; ++vt) {
        const v8bf x0 = *(const v8bf*)(xp + 2048 * vt + p0);
        const v8bf x1 = *(const v8bf*)(xp + 2048 * vt + p1);
        const v4f z = *(const v4f*)(zp + 64 * vt);
        v4f d[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) d[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, wv[rt][0], z, 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) d[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1, wv[rt][1], d[rt], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int i = 0; i < 4; ++i) y[rt][vt][i] = fmaf(sc[rt], d[rt][i], y[rt][vt][i]);
      }
    }
  }
  __syncthreads();

  // (the exchange of two sets, then one vector tile's image at a time)
  float* img = (float*)(sm + XCHG) + (half * 4 + wave) * 16 * PITCH;
  if constexpr (KS == 2) {
    // each set hands over the half of its sums that the other one stores; the
    // tiles a wave stores end in y[0], y[1]
    v4f* mine = (v4f*)sm + (half * 4 + wave) * 512 + lane;
    const v4f* theirs = (const v4f*)sm + ((half ^ 1) * 4 + wave) * 512 + lane;
    if (half == 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) mine[64 * i] = y[2 + (i >> 2)][i & 3];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        mine[64 * i] = y[i >> 2][i & 3];
        y[i >> 2][i & 3] = y[2 + (i >> 2)][i & 3];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i >> 2][i & 3] += theirs[64 * i];
  }
  // eight consecutive rows of one vector per lane
  const int64_t nb = (tile0 + (KS == 1 ? 0 : 2 * half)) * 16;
#pragma unroll
  for (int vt = 0; vt < 4; ++vt) {
#pragma unroll
    for (int t = 0; t < NRT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) img[(4 * kq + i) * PITCH + 16 * t + r] = y[t][vt][i];
    wave_lds_sync();
#pragma unroll
    for (int c0 = 0; c0 < 32 * NRT; c0 += 64) {
      const int c = c0 + lane, v = c / (2 * NRT), n8 = 8 * (c % (2 * NRT)), m = 16 * vt + v;
      if (m < rows && nb + n8 < a.N) {
        const v4f lo = *(const v4f*)(img + v * PITCH + n8), hi = *(const v4f*)(img + v * PITCH + n8 + 4);
        q4_store8(a, m0 + m, nb + n8, lo, hi);
      }
    }
    wave_lds_sync();
  }
}

// Few vectors: the weights streamed once for up to 16·VT vectors.  Workgroup
// (x, y): row tiles Rx .. Rx + R - 1 against vectors 16·VT·y ...; its NW waves
// split K (wave w takes spans w, w + NW, ...) and sum their partial tiles
// through LDS.  Operands come straight from memory, weights as records, x (a
// few hundred KB, held by the L2) as 16-byte runs in its own order; X is a
// matrix product with ones, whose result lies in the lanes that need it.
template <int R, int VT>
__global__ __launch_bounds__(512) void q4_few_kernel(const Q4GemmArgs a) {
  constexpr int NW = 8;
  __shared__ v4f red[NW * R * VT * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t tiles = (a.N + 15) / 16, tile0 = (int64_t)blockIdx.x * R;
  const int S = (int)(a.K / GV_SPAN);
  const int r = lane & 15, kq = lane >> 4;
  const int m0 = (int)blockIdx.y * 16 * VT;
  const int rows = min(16 * VT, a.M - m0);
  const int n_w = wave < S ? (S - wave + NW - 1) / NW : 0;  // spans of this wave

  __amdgpu_buffer_rsrc_t RW[R];
#pragma unroll
  for (int rt = 0; rt < R; ++rt) {
    const bool live = tile0 + rt < tiles;
    RW[rt] = make_rsrc(a.packed + (live ? (tile0 + rt) * S * GV_REC : 0), live ? (int64_t)S * GV_REC : 0);
  }
  // vectors past M lie past the resource's end and read zero
  const __amdgpu_buffer_rsrc_t RX =
      make_rsrc(a.x + (int64_t)m0 * a.x_stride, ((int64_t)(rows - 1) * a.x_stride + a.K) * 2);
  uint32_t xoff[VT];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) xoff[vt] = (uint32_t)(((int64_t)(16 * vt + r) * a.x_stride + 8 * kq) * 2);
  const uint32_t wl = 16 * r + 4 * kq, sl = 1024 + 32 * kq;

  const uint32_t base = code_base();

  constexpr int NB = 2;  // spans in flight
  uint32_t wr[NB][R][4];
  v4i sbr[NB][R][2];
  v4i xr[NB][VT][4];
  const auto fetch = [&](int b, int sp) {
    const uint32_t rec = (uint32_t)sp * GV_REC;
#pragma unroll
    for (int rt = 0; rt < R; ++rt) {
#pragma unroll
      for (int t = 0; t < 4; ++t) wr[b][rt][t] = ld32(RW[rt], wl + 256 * t, rec);
      sbr[b][rt][0] = ld128(RW[rt], sl, rec);
      sbr[b][rt][1] = ld128(RW[rt], sl + 16, rec);
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int t = 0; t < 4; ++t) xr[b][vt][t] = ld128<0>(RX, xoff[vt] + 64 * t, (uint32_t)(256 * sp));
  };

  v4f y[R][VT];
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) y[rt][vt] = (v4f){0.f, 0.f, 0.f, 0.f};
  const v8bf ones = __builtin_bit_cast(v8bf, (v4i){0x3f803f80, 0x3f803f80, 0x3f803f80, 0x3f803f80});

  const auto compute = [&](int b) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      v8bf bx[VT][2];
      v4f X[VT];  // the sums of column r, four times
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        bx[vt][0] = __builtin_bit_cast(v8bf, xr[b][vt][2 * g]);
        bx[vt][1] = __builtin_bit_cast(v8bf, xr[b][vt][2 * g + 1]);
        v4f x4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bx[vt][0], (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        x4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bx[vt][1], x4, 0, 0, 0);
        X[vt] = x4;
      }
#pragma unroll
      for (int rt = 0; rt < R; ++rt) {
        const v8bf a0 = unpack_codes_in_order(wr[b][rt][2 * g], base);
        const v8bf a1 = unpack_codes_in_order(wr[b][rt][2 * g + 1], base);
        const v4i sb = sbr[b][rt][g];
        const uint32_t s01 = (uint32_t)sb[0], s23 = (uint32_t)sb[1], b01 = (uint32_t)sb[2], b23 = (uint32_t)sb[3];
        const float sc[4] = {bf16_lo(s01), bf16_hi(s01), bf16_lo(s23), bf16_hi(s23)};
        const float cb[4] = {fmaf(-128.f, sc[0], bf16_lo(b01)), fmaf(-128.f, sc[1], bf16_hi(b01)),
                             fmaf(-128.f, sc[2], bf16_lo(b23)), fmaf(-128.f, sc[3], bf16_hi(b23))};
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          v4f d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, bx[vt][0], (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, bx[vt][1], d, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) y[rt][vt][i] = fmaf(cb[i], X[vt][i], fmaf(sc[i], d[i], y[rt][vt][i]));
        }
      }
    }
  };

  if (n_w > 0) fetch(0, wave);
  for (int i = 0; i < n_w; i += 2) {
    if (i + 1 < n_w) fetch(1, wave + NW * (i + 1));
    compute(0);
    if (i + 1 < n_w) {
      if (i + 2 < n_w) fetch(0, wave + NW * (i + 2));
      compute(1);
    }
  }

  // sum the waves' partial tiles, tile p by wave p % NW
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) red[(wave * R * VT + rt * VT + vt) * 64 + lane] = y[rt][vt];
  __syncthreads();
  for (int p = wave; p < R * VT; p += NW) {
    const int64_t tile = tile0 + p / VT;
    const int m = m0 + 16 * (p % VT) + r;
    if (tile >= tiles || m >= a.M) continue;
    v4f s = red[p * 64 + lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[(w * R * VT + p) * 64 + lane];
    q4_store(a, m, tile * 16 + 4 * kq, s);
  }
}

// Few vectors, many rows, K ≤ 2,048: 256 workgroups stream the row tiles b,
// b + grid, ...  A wave keeps the x of its spans (w, w + 8) in registers, and
// their group sums, and has the records of the next two tiles in flight; the
// eight partial tiles of a row tile are summed through LDS, one value per lane.
template <int VT>
__global__ __launch_bounds__(512, 2) void q4_stream_kernel(const Q4GemmArgs a) {
  constexpr int NSP = 2;  // spans per wave
  __shared__ v4f red[2][8 * VT * 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = (int)((a.N + 15) / 16), S = (int)(a.K / GV_SPAN);
  const int r = lane & 15, kq = lane >> 4;
  const int rows = a.M;  // at most 16 VT
  const int grid = (int)gridDim.x, n_t = (tiles - (int)blockIdx.x + grid - 1) / grid;
  const int64_t bytes = (int64_t)tiles * S * GV_REC;  // below 2^31
  const __amdgpu_buffer_rsrc_t RW = make_rsrc(a.packed, bytes);
  const uint32_t base = code_base();

  constexpr int NB = 3;
  uint32_t wr[NB][NSP][4], sb[NB][NSP][4];
  const uint32_t wl = 16 * r + 4 * kq, sl = 1024 + 32 * (r >> 2) + 2 * (r & 3);
  const auto fetch = [&](int b, int it) {
    const int tile = (int)blockIdx.x + it * grid;
#pragma unroll
    for (int j = 0; j < NSP; ++j) {
      const int sp = wave + 8 * j;  // absent spans and tiles past the last read zeros
      const uint32_t rec = it < n_t && sp < S ? (uint32_t)(tile * S + sp) * GV_REC : 0x7fffffffu;
#pragma unroll
      for (int t = 0; t < 4; ++t) wr[b][j][t] = ld32(RW, wl + 256 * t, rec);
#pragma unroll
      for (int t = 0; t < 4; ++t)  // group t / 2: scale, then bias
        sb[b][j][t] = __builtin_amdgcn_raw_buffer_load_b16(RW, sl + 16 * (t >> 1) + 8 * (t & 1), rec, BUF_NT);
    }
  };
#pragma unroll
  for (int b = 0; b < NB - 1; ++b) fetch(b, b);

  // x, and X = Σx of each group by a matrix product with ones: lane (r, kq)
  // gets the sums of the vectors 4kq .. 4kq+3
  const __amdgpu_buffer_rsrc_t RX = make_rsrc(a.x, ((int64_t)(rows - 1) * a.x_stride + a.K) * 2);
  const v8bf ones = __builtin_bit_cast(v8bf, (v4i){0x3f803f80, 0x3f803f80, 0x3f803f80, 0x3f803f80});
  v8bf x[NSP][VT][4];
  v4f X[NSP][VT][2];
#pragma unroll
  for (int j = 0; j < NSP; ++j)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      const uint32_t off = (uint32_t)(((int64_t)(16 * vt + r) * a.x_stride + 8 * kq) * 2);
      const uint32_t so = wave + 8 * j < S ? (uint32_t)(256 * (wave + 8 * j)) : 0x7fffffffu;
#pragma unroll
      for (int t = 0; t < 4; ++t) x[j][vt][t] = __builtin_bit_cast(v8bf, ld128<0>(RX, off + 64 * t, so));
    }
#pragma unroll
  for (int j = 0; j < NSP; ++j)
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        v4f d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j][vt][2 * g], ones, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        X[j][vt][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j][vt][2 * g + 1], ones, d, 0, 0, 0);
      }

  // the value this lane stores: component i of vector tile vs's lane
  const int vs = wave % VT, i = wave / VT;
  const int m = 16 * vs + 4 * kq + i;
  const bool mine = i < 4 && m < a.M;
  for (int it0 = 0; it0 < n_t; it0 += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int it = it0 + b;
      if (it < n_t) {  // the same for the workgroup
        fetch((b + NB - 1) % NB, it + NB - 1);
        v4f y[VT];
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) y[vt] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NSP; ++j)
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            const v8bf w0 = unpack_codes_in_order(wr[b][j][2 * g], base);
            const v8bf w1 = unpack_codes_in_order(wr[b][j][2 * g + 1], base);
            const float sc = bf16_lo(sb[b][j][2 * g]), cb = fmaf(-128.f, sc, bf16_lo(sb[b][j][2 * g + 1]));
#pragma unroll
            for (int vt = 0; vt < VT; ++vt) {
              v4f d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j][vt][2 * g], w0, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j][vt][2 * g + 1], w1, d, 0, 0, 0);
#pragma unroll
              for (int e = 0; e < 4; ++e) y[vt][e] = fmaf(cb, X[j][vt][g][e], fmaf(sc, d[e], y[vt][e]));
            }
          }
        v4f* rd = red[it & 1];
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) rd[(wave * VT + vt) * 64 + lane] = y[vt];
        __syncthreads();  // (two buffers: the next tile's writes need no barrier of their own)
        if (mine) {
          float s = 0.f;
#pragma unroll
          for (int w = 0; w < 8; ++w) s += ((const float*)(rd + (w * VT + vs) * 64 + lane))[i];
          const int64_t n = (int64_t)((int)blockIdx.x + it * grid) * 16 + r;
          if (n < a.N) {
            if (a.out_dtype == DT_F32) ((float*)a.out)[(int64_t)m * a.out_stride + n] = s;
            else ((__bf16*)a.out)[(int64_t)m * a.out_stride + n] = (__bf16)s;
          }
        }
      }
    }
  }
}

template <int VT>
static hipError_t launch_stream(const Q4GemmArgs& a, hipStream_t stream) {
  const int64_t tiles = (a.N + 15) / 16;
  hipLaunchKernelGGL(q4_stream_kernel<VT>, dim3((unsigned)(tiles < 256 ? tiles : 256)), dim3(512), 0, stream, a);
  return hipGetLastError();
}

template <int R, int VT>
static hipError_t launch_few(const Q4GemmArgs& a, hipStream_t stream) {
  const int64_t tiles = (a.N + 15) / 16;
  const dim3 grid((unsigned)((tiles + R - 1) / R), (unsigned)((a.M + 16 * VT - 1) / (16 * VT)));
  hipLaunchKernelGGL((q4_few_kernel<R, VT>), grid, dim3(512), 0, stream, a);
  return hipGetLastError();
}

template <int KS>
static hipError_t launch_wide(const Q4GemmArgs& a, int64_t n, hipStream_t stream) {
  const int64_t sums = ((int64_t)a.M + 31) / 32 * (a.K / GV_SPAN);
  hipLaunchKernelGGL(q4_xsum_kernel, dim3((unsigned)(sums < XSUM_GRID_MAX ? sums : XSUM_GRID_MAX)), dim3(256), 0,
                     stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(q4_gemm_kernel<KS>, dim3((unsigned)n), dim3(256 * KS), 0, stream, a);
  return hipGetLastError();
}

// Which kernel, by sizes (MI355X, µs, x·Wᵀ with bf16 results; before these
// kernels: GEMV launches of 8 vectors, and from 24 + 8·⌊K/1024⌋ vectors on one
// GEMM that read each x operand for two row tiles, its LDS reads the bound):
//  * q4_stream_kernel up to 32 vectors, from 512 row tiles (two per workgroup)
//    and K ≤ 2,048 (a wave's x in registers).  24 vectors: 12,288 rows 23.2 →
//    10.8 (q4_few_kernel 15.5), 150,144 rows 121 → 61 (173 MB in 61 µs, the
//    rest the start and end of the stream); 5,120 rows are 320 tiles, 9.6
//    against 8.5 in q4_few_kernel.
//  * q4_few_kernel while its 32-vector grid has at most 704 workgroups: 2,048 x
//    4,096 at 24 / 100 / 350 vectors 21.8 / 50.5 / 53 → 8.6 / 15.2 / 40.5 (the
//    wide kernel 43-44, 450 vectors 55.5); 5,120 x 2,048 at 24 / 100 vectors 19.5 /
//    29 → 8.5 / 22.2 (wide 25.2; 130 vectors 27.3 against 25.4).  Bound by one
//    round trip to memory per two spans.  The smallest tile whose grid still
//    gives a CU at most one workgroup: 2,048 x 4,096 at 24 vectors 8.6 / 11.1 /
//    13.6 with one tile and 16 vectors / two and 16 / two and 32, at 64 vectors
//    14.5 / 11.4 / 14.8, at 100 24.2 / 20.7 / 15.2.
//  * else q4_gemm_kernel: up to one workgroup per CU with two wave sets (2,048
//    x 4,096 at 2,000 vectors 49 against 68 with one), beyond with one (12,288
//    x 2,048: 129 against 145).
hipError_t launch_q4_gemm(const Q4GemmArgs& a, hipStream_t stream) {
  const int64_t tiles = (a.N + 15) / 16, M = a.M;
  if (M <= 32 && tiles >= 512 && a.K <= 2048) {
    return M <= 16 ? launch_stream<1>(a, stream) : launch_stream<2>(a, stream);
  }
  const int64_t pairs = (tiles + 1) / 2, cols = (M + 15) / 16;
  if (pairs * ((M + 31) / 32) <= 704) {
    if (tiles * cols <= 256) return launch_few<1, 1>(a, stream);
    if (pairs * cols <= 256) return launch_few<2, 1>(a, stream);
    return launch_few<2, 2>(a, stream);
  }
  const int64_t n = (tiles + GM_TILES - 1) / GM_TILES * ((M + GM_VECS - 1) / GM_VECS);
  return n <= 256 ? launch_wide<2>(a, n, stream) : launch_wide<1>(a, n, stream);
}

}  // namespace rec
