// NVFP4 block quantization for gfx950: e2m1 values in blocks of 16 with an e4m3 scale per
// block under a per-tensor fp32 scale, and the exact dequantization of such blocks to bf16.
//
// Replaces TE's NVFP4BlockScaling quantizer behind te.Linear under the 'nvfp4' recipe
// (bongard/te_linear.py:17,38; bongard/fused_mlp.py:9,32) for the part its arithmetic
// fixes without TE at hand (round to nearest even everywhere; no random Hadamard
// transform, no stochastic rounding, 1-D blocks along the GEMM's reduction dimension):
//
//   S_enc = fp32(2688 / max(f64(amax), 1e-12))       2688 = e4m3 max (448) x e2m1 max (6)
//   S_dec = fp32(1 / S_enc)
//   per block of 16 (b = max |x| over the block):
//     s    = e4m3_rne_sat(fp32(fp32(b / 6) * S_enc))  the stored block scale
//     mult = s == 0 ? 0 : fp32(S_enc / s)
//     q_i  = e2m1_rne(fp32(x_i * mult))               saturating at +-6
//   x_i ~ e2m1(q_i) * s * S_dec
//
// gfx950's block-scaled MFMA takes FP4 only with power-of-two scales per 32 values, so the
// GEMM runs on the bf16 MFMA instead: e2m1(q) * s has at most 6 significant bits and is
// exact in bf16 (bf8_dequant_nvfp4 writes it), and the GEMM epilogue applies S_dec of both
// operands. Codes: bit 3 the sign (copied from the product, so -0 is 0x8), bits 0-2 the
// magnitude index into {0, 0.5, 1, 1.5, 2, 3, 4, 6}; two codes per byte, the even element
// in the low nibble. A NaN product gives code 0 with its sign bit (unpinned: no reference
// result exists for non-finite blocks).
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace bf8 {
namespace {

constexpr int kNT = 256;
constexpr float kNvfp4Max = 6.0f;
constexpr float kNvfp4Global = 448.0f * 6.0f;
constexpr int64_t kMaxNvfp4Blocks = 2048;

// Round-to-nearest-even onto the e2m1 grid by threshold counting: each midpoint between
// neighbours rounds to the neighbour whose code is even (0.25 -> 0, 0.75 -> 1, 1.25 -> 1,
// 1.75 -> 2, 2.5 -> 2, 3.5 -> 4, 5 -> 4); beyond 5 everything (inf included) is 6.
__device__ __forceinline__ uint32_t e2m1_code(float p) {
  const float a = fabsf(p);
  const uint32_t m = (uint32_t)(a > 0.25f) + (uint32_t)(a >= 0.75f) + (uint32_t)(a > 1.25f) +
                     (uint32_t)(a >= 1.75f) + (uint32_t)(a > 2.5f) + (uint32_t)(a >= 3.5f) +
                     (uint32_t)(a > 5.0f);
  return m | ((__float_as_uint(p) >> 31) << 3);
}

// e4m3 byte of v (RNE, saturating at 448; NaN as 0x7F | sign), and the fp32 value of a byte.
__device__ __forceinline__ uint32_t e4m3_byte(float v) {
  return quant4<BF8_E4M3>(v, 0.f, 0.f, 0.f, v, 0.f, 0.f, 0.f, 1.0f) & 0xFFu;
}
__device__ __forceinline__ float e4m3_value(uint32_t byte) {
  return __builtin_amdgcn_cvt_f32_fp8((int)byte, 0);
}

// The block scale byte and the multiplier of a block whose max |x| is the bf16 key k.
__device__ __forceinline__ void block_scale(uint32_t key, float s_enc, uint32_t& sbyte,
                                            float& mult) {
  const float bmax = __uint_as_float(key);
  sbyte = e4m3_byte((bmax / kNvfp4Max) * s_enc);
  const float s = e4m3_value(sbyte);
  mult = s == 0.0f ? 0.0f : s_enc / s;
}

// 16 bf16 values (two uint4) -> 8 packed code bytes.
__device__ __forceinline__ uint2 pack16(const uint32_t (&w)[8], float mult) {
  uint32_t r[2] = {0u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t lo = e2m1_code(bf16_lo(w[i]) * mult);
    const uint32_t hi = e2m1_code(bf16_hi(w[i]) * mult);
    r[i >> 2] |= (lo | (hi << 4)) << (8 * (i & 3));
  }
  return make_uint2(r[0], r[1]);
}

// The two codes of byte B of c times s, as packed bf16. e2m1 x e4m3 has at most 6 significant
// bits: the fp32 product is exact, and so is its bf16 (upper half).
template <int B>
__device__ __forceinline__ uint32_t dequant_pair(uint32_t c, float s) {
  const auto v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, B);
  return __builtin_amdgcn_perm(__float_as_uint(v[1] * s), __float_as_uint(v[0] * s), 0x07060302u);
}
__device__ __forceinline__ uint4 dequant8(uint32_t c, float s) {
  return make_uint4(dequant_pair<0>(c, s), dequant_pair<1>(c, s), dequant_pair<2>(c, s),
                    dequant_pair<3>(c, s));
}

// Packed codes of 8 bf16 values times their multipliers (element j in nibble j).
// FAST: v_cvt_scalef32_pk_fp4_f32 with scale 1, which rounds and saturates as e2m1_code does
// for every fp32 but NaN (compared over all 2^32 values); no product is NaN there.
template <bool FAST>
__device__ __forceinline__ uint32_t codes8(uint4 v, const float* m) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t c = 0;
  if constexpr (FAST) {
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, bf16_lo(w[0]) * m[0], bf16_hi(w[0]) * m[1], 1.0f, 0);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, bf16_lo(w[1]) * m[2], bf16_hi(w[1]) * m[3], 1.0f, 1);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, bf16_lo(w[2]) * m[4], bf16_hi(w[2]) * m[5], 1.0f, 2);
    c = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(c, bf16_lo(w[3]) * m[6], bf16_hi(w[3]) * m[7], 1.0f, 3);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      c |= (e2m1_code(bf16_lo(w[i]) * m[2 * i]) | (e2m1_code(bf16_hi(w[i]) * m[2 * i + 1]) << 4))
           << (8 * i);
  }
  return c;
}

// block_scale for a finite block under a finite S_enc (key16: bf16 bits of max |x|): b / 6 from a
// reciprocal and one correction (equal to the division for every finite bf16 b), S_enc / s from
// the block's table of the 127 scale values.
__device__ __forceinline__ void block_scale_fast(uint32_t key16, float s_enc,
                                                 const float* __restrict__ mult_of,
                                                 uint32_t& sbyte, float& mult) {
  constexpr float kSixth = 1.0f / kNvfp4Max;
  const float b = __uint_as_float(key16 << 16);
  float q = b * kSixth;
  q = __builtin_fmaf(__builtin_fmaf(-kNvfp4Max, q, b), kSixth, q);
  const float v = __builtin_fminf(q * s_enc, 448.0f);
  sbyte = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v, 0.0f, 0, false) & 0xFFu;
  mult = mult_of[sbyte];
}

// Rowwise and / or columnwise quantization. Rowwise: blocks of 16
// consecutive elements of a row, out [rows, cols / 2] with scales [rows, cols / 16], or their
// exact bf16 dequantization deq [rows, cols]. Columnwise: the rowwise quantization of x^T,
// out_t [cols, rows / 2] with scales_t [cols, rows / 16], or its dequantization deq_t
// [cols, rows].
struct NvTile {
  int64_t rows, cols;
  uint8_t* out;
  uint8_t* scales;
  uint16_t* deq;
  uint8_t* out_t;
  uint8_t* scales_t;
  uint16_t* deq_t;
};

constexpr int kNT4 = 128;            // tile (rows x cols) of a block
constexpr int kNvPitch = kNT4 / 8 + 1;  // staged dwords per row (8 codes each; odd)
constexpr int kMaxNvTileBlocks = 1024;

template <bool FAST>
__device__ __forceinline__ void nv_tile_body(const NvTile& p, int64_t r0, int64_t c0,
                                             const uint4 (&v)[8], const uint32_t (&rk)[8],
                                             const uint32_t (&cm)[2][4], float s_enc,
                                             const float* __restrict__ mult_of, uint32_t* stage,
                                             uint8_t (*scol)[kNT4], int wid, int lane) {
  const int cl = lane & 15, lr = lane >> 4;
  const int64_t c = c0 + 8 * cl;
  auto scale_of = [&](uint32_t key16, uint32_t& sbyte, float& mult) {
    if constexpr (FAST)
      block_scale_fast(key16, s_enc, mult_of, sbyte, mult);
    else
      block_scale(key16 << 16, s_enc, sbyte, mult);
  };
  if (p.out || p.deq) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t r = r0 + 32 * wid + 4 * k + lr;
      uint32_t sbyte;
      float mult;
      scale_of(rk[k], sbyte, mult);
      const float m[8] = {mult, mult, mult, mult, mult, mult, mult, mult};
      const uint32_t code = codes8<FAST>(v[k], m);
      if (r < p.rows && c < p.cols) {
        if (p.deq) {
          *reinterpret_cast<uint4*>(p.deq + r * p.cols + c) = dequant8(code, e4m3_value(sbyte));
        } else {
          *reinterpret_cast<uint32_t*>(p.out + ((r * p.cols + c) >> 1)) = code;
          if ((cl & 1) == 0) p.scales[(r * p.cols + c) >> 4] = (uint8_t)sbyte;
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {  // the wave's 16-row blocks
    float m[8];
    uint32_t sb[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint32_t sbyte;
      scale_of((cm[b][e >> 1] >> (16 * (e & 1))) & 0xFFFFu, sbyte, m[e]);
      sb[e >> 2] |= sbyte << (8 * (e & 3));
    }
    if (lr == 0) {
      uint32_t* d = reinterpret_cast<uint32_t*>(&scol[2 * wid + b][8 * cl]);
      d[0] = sb[0];
      d[1] = sb[1];
    }
#pragma unroll
    for (int k = 4 * b; k < 4 * b + 4; ++k)
      stage[(32 * wid + 4 * k + lr) * kNvPitch + cl] = codes8<FAST>(v[k], m);
  }
}

// The columnwise copy, with or without the rowwise one, in one pass over x. A block walks
// 128 x 128 tiles, each wave 32 rows of all 128 columns: lane l holds columns
// 8 (l & 15) .. +7 of the rows 4 k + l / 16, k < 8. A row block of 16 is two neighbouring
// lanes, a column block of 16 four pieces and the four lanes of a column group. The columnwise
// codes meet in LDS as 8-column dwords; each thread then turns 8 rows x 8 columns of nibbles.
// Loads, and every store of the bf16 outputs, are whole 128-byte lines; the next tile's loads
// are issued before the columnwise stores.
// HBM-bound (2 B read, 0.5625 or 2 B written per element and copy) once the rounding is one
// hardware conversion per two values and the two divisions per block are a multiply-add
// pair and a table: before, seven comparisons per value and the divisions made it VALU-bound,
// and the columnwise kernel's 8-byte stores each had a line of their own. Rowwise bf16 and
// columnwise codes, inputs rotated past the MALL: [4096, 20480] 253.3 -> 101.1 us (3.8 TB/s),
// [20480, 2560] 169.9 -> 60.8, [2048, 20480] 105.2 -> 47.1; both copies as bf16 [4096, 10240]
// 49.6 us (5.1 TB/s).
__global__ __launch_bounds__(kNT) void nvfp4_tile_kernel(const uint16_t* __restrict__ x,
                                                         NvTile p,
                                                         const uint32_t* __restrict__ partials,
                                                         int64_t np, float* __restrict__ meta) {
  __shared__ uint32_t stage[kNT4 * kNvPitch];
  __shared__ __attribute__((aligned(16))) uint8_t scol[kNT4 / 16][kNT4];  // [row block][column]
  __shared__ float mult_of[128];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t tiles_c = (p.cols + kNT4 - 1) / kNT4, tiles_r = (p.rows + kNT4 - 1) / kNT4;
  const int64_t ntiles = tiles_c * tiles_r;
  const int cl = lane & 15, lr = lane >> 4;
  uint4 v[8];
  auto load = [&](int64_t t) {
    const int64_t r0 = (t / tiles_c) * kNT4, c = (t % tiles_c) * kNT4 + 8 * cl;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t r = r0 + 32 * wid + 4 * k + lr;
      v[k] = make_uint4(0u, 0u, 0u, 0u);
      if (t < ntiles && r < p.rows && c < p.cols)
        v[k] = *reinterpret_cast<const uint4*>(x + r * p.cols + c);
    }
  };
  load(blockIdx.x);
  const float s_enc = scale_from_partials_block<kNT>(partials, np, kNvfp4Global, meta, false,
                                                     blockIdx.x == 0);
  if (threadIdx.x < 128) {
    const float s = e4m3_value(threadIdx.x);
    mult_of[threadIdx.x] = s == 0.0f ? 0.0f : s_enc / s;
  }
  __syncthreads();
  const bool s_finite = fabsf(s_enc) < INFINITY;
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int64_t r0 = (t / tiles_c) * kNT4, c0 = (t % tiles_c) * kNT4;
    uint32_t rk[8], cm[2][4] = {};
    uint32_t top = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t a[4] = {v[k].x & 0x7FFF7FFFu, v[k].y & 0x7FFF7FFFu, v[k].z & 0x7FFF7FFFu,
                             v[k].w & 0x7FFF7FFFu};
#pragma unroll
      for (int i = 0; i < 4; ++i) cm[k >> 2][i] = pk_max_u16(cm[k >> 2][i], a[i]);
      uint32_t m = pk_max_u16(pk_max_u16(a[0], a[1]), pk_max_u16(a[2], a[3]));
      m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, true));
      rk[k] = max(m & 0xFFFFu, m >> 16);
      top = max(top, rk[k]);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        cm[b][i] = pk_max_u16(cm[b][i], (uint32_t)__shfl_xor((int)cm[b][i], 16, 64));
        cm[b][i] = pk_max_u16(cm[b][i], (uint32_t)__shfl_xor((int)cm[b][i], 32, 64));
      }
    if (__builtin_expect(__any(top >= 0x7F80u) || !s_finite, 0))
      nv_tile_body<false>(p, r0, c0, v, rk, cm, s_enc, mult_of, stage, scol, wid, lane);
    else
      nv_tile_body<true>(p, r0, c0, v, rk, cm, s_enc, mult_of, stage, scol, wid, lane);
    load(t + gridDim.x);
    __syncthreads();
    // thread: rows 8 rg .. +7 of columns 8 cg .. +7; nibble j of d[i] is column j of row i
    const int rg = threadIdx.x & 15, cg = threadIdx.x >> 4;
    const int64_t tc = r0 + 8 * rg;  // column of the transposed outputs (a row of x)
    uint32_t d[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) d[i] = stage[(8 * rg + i) * kNvPitch + cg];
    uint32_t ev[4], od[4];  // rows 2i, 2i + 1: the even / odd columns' code pairs, one byte each
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ev[i] = (d[2 * i] & 0x0F0F0F0Fu) | ((d[2 * i + 1] & 0x0F0F0F0Fu) << 4);
      od[i] = ((d[2 * i] >> 4) & 0x0F0F0F0Fu) | (d[2 * i + 1] & 0xF0F0F0F0u);
    }
    uint32_t q[8];  // the 8 rows' codes of each column
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t* w = h == 0 ? ev : od;
      const uint32_t t0 = __byte_perm(w[0], w[1], 0x5140), t1 = __byte_perm(w[0], w[1], 0x7362);
      const uint32_t t2 = __byte_perm(w[2], w[3], 0x5140), t3 = __byte_perm(w[2], w[3], 0x7362);
      q[h] = __byte_perm(t0, t2, 0x5410);
      q[2 + h] = __byte_perm(t0, t2, 0x7632);
      q[4 + h] = __byte_perm(t1, t3, 0x5410);
      q[6 + h] = __byte_perm(t1, t3, 0x7632);
    }
    const uint2 sb = *reinterpret_cast<const uint2*>(&scol[rg >> 1][8 * cg]);
    if (tc < p.rows && c0 + 8 * cg < p.cols) {  // cols % 8 == 0: eight columns in or out
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t tr = c0 + 8 * cg + j;
        const uint32_t sbyte = ((j < 4 ? sb.x : sb.y) >> (8 * (j & 3))) & 0xFFu;
        if (p.deq_t) {
          *reinterpret_cast<uint4*>(p.deq_t + tr * p.rows + tc) = dequant8(q[j], e4m3_value(sbyte));
        } else {
          *reinterpret_cast<uint32_t*>(p.out_t + ((tr * p.rows + tc) >> 1)) = q[j];
          if ((rg & 1) == 0) p.scales_t[(tr * p.rows + tc) >> 4] = (uint8_t)sbyte;
        }
      }
    }
    __syncthreads();
  }
}

// The rowwise copy by blocks 0 .. nblk - 1: one 16-block per thread (grid-stride).
__device__ __forceinline__ void nv_rows_body(const uint16_t* __restrict__ x, const NvTile& p,
                                             float s_enc, float* mult_of, int64_t blk,
                                             int64_t nblk) {
  if (threadIdx.x < 128) {
    const float s = e4m3_value(threadIdx.x);
    mult_of[threadIdx.x] = s == 0.0f ? 0.0f : s_enc / s;
  }
  __syncthreads();
  const bool s_finite = fabsf(s_enc) < INFINITY;
  const int64_t items = p.rows * (p.cols / 16);
  for (int64_t b = blk * kNT + threadIdx.x; b < items; b += nblk * kNT) {
    const uint4* src = reinterpret_cast<const uint4*>(x + b * 16);
    const uint4 v0 = src[0], v1 = src[1];
    const uint32_t key = max(absmax_key8(v0), absmax_key8(v1));
    uint32_t sbyte, c0, c1;
    float mult;
    if (__builtin_expect(!s_finite || key >= 0x7F800000u, 0)) {
      block_scale(key, s_enc, sbyte, mult);
      const float m[8] = {mult, mult, mult, mult, mult, mult, mult, mult};
      c0 = codes8<false>(v0, m);
      c1 = codes8<false>(v1, m);
    } else {
      block_scale_fast(key >> 16, s_enc, mult_of, sbyte, mult);
      const float m[8] = {mult, mult, mult, mult, mult, mult, mult, mult};
      c0 = codes8<true>(v0, m);
      c1 = codes8<true>(v1, m);
    }
    if (p.deq) {
      const float s = e4m3_value(sbyte);
      uint4* dst = reinterpret_cast<uint4*>(p.deq + b * 16);
      dst[0] = dequant8(c0, s);
      dst[1] = dequant8(c1, s);
    } else {
      *reinterpret_cast<uint2*>(p.out + b * 8) = make_uint2(c0, c1);
      p.scales[b] = (uint8_t)sbyte;
    }
  }
}

// The rowwise copy alone: codes and scale bytes leave in whole lines, where the tile kernel's
// 128-column rows would write the codes in half lines. Codes of [4096, 20480]: 40.5 us (5.3 TB/s;
// 56.3 us on the tile kernel, 54.6 us with the rounding by comparisons).
__global__ __launch_bounds__(kNT) void nvfp4_rows_kernel(const uint16_t* __restrict__ x, NvTile p,
                                                         const uint32_t* __restrict__ partials,
                                                         int64_t np, float* __restrict__ meta) {
  __shared__ float mult_of[128];
  const float s_enc = scale_from_partials_block<kNT>(partials, np, kNvfp4Global, meta, false,
                                                     blockIdx.x == 0);
  nv_rows_body(x, p, s_enc, mult_of, blockIdx.x, gridDim.x);
}

// The columnwise copy by blocks 0 .. nblk - 1: one (column, 16-row block) per thread, consecutive
// threads on consecutive columns. out_t [cols, rows / 2], scales_t [cols, rows / 16].
__device__ __forceinline__ void nv_cols_body(const uint16_t* __restrict__ x, int64_t rows,
                                             int64_t cols, float s_enc,
                                             uint8_t* __restrict__ out_t,
                                             uint8_t* __restrict__ scales_t, int64_t blk,
                                             int64_t nblk) {
  const int64_t rblocks = rows / 16;
  const int64_t nitems = cols * rblocks;
  for (int64_t it = blk * kNT + threadIdx.x; it < nitems; it += nblk * kNT) {
    const int64_t rb = it / cols, c = it - rb * cols;
    uint32_t w[8];
    uint32_t key = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t lo = x[(rb * 16 + 2 * i) * cols + c];
      const uint32_t hi = x[(rb * 16 + 2 * i + 1) * cols + c];
      w[i] = lo | (hi << 16);
      key = max(key, max((lo & 0x7FFFu) << 16, (hi & 0x7FFFu) << 16));
    }
    uint32_t sbyte;
    float mult;
    block_scale(key, s_enc, sbyte, mult);
    *reinterpret_cast<uint2*>(out_t + c * (rows / 2) + rb * 8) = pack16(w, mult);
    scales_t[c * rblocks + rb] = (uint8_t)sbyte;
  }
}

// Columnwise quantization of a small tensor, or of one whose rows are not whole 16-byte vectors
// (cols % 8 != 0), which the tile kernel's loads need.
__global__ __launch_bounds__(kNT) void nvfp4_cols_kernel(const uint16_t* __restrict__ x,
                                                         int64_t rows, int64_t cols,
                                                         const uint32_t* __restrict__ partials,
                                                         int64_t np, float* __restrict__ meta,
                                                         uint8_t* __restrict__ out_t,
                                                         uint8_t* __restrict__ scales_t) {
  const float s_enc = scale_from_partials_block<kNT>(partials, np, kNvfp4Global, meta, false,
                                                     blockIdx.x == 0);
  nv_cols_body(x, rows, cols, s_enc, out_t, scales_t, blockIdx.x, gridDim.x);
}

// Both copies of a small tensor: the first row_blocks blocks take the rowwise copy, the others the
// columnwise codes, each reading x for itself (the second time from a cache).
__global__ __launch_bounds__(kNT) void nvfp4_pair_kernel(const uint16_t* __restrict__ x, NvTile p,
                                                         const uint32_t* __restrict__ partials,
                                                         int64_t np, float* __restrict__ meta,
                                                         int row_blocks) {
  __shared__ float mult_of[128];
  const float s_enc = scale_from_partials_block<kNT>(partials, np, kNvfp4Global, meta, false,
                                                     blockIdx.x == 0);
  if ((int)blockIdx.x < row_blocks)
    nv_rows_body(x, p, s_enc, mult_of, blockIdx.x, row_blocks);
  else
    nv_cols_body(x, p.rows, p.cols, s_enc, p.out_t, p.scales_t, blockIdx.x - row_blocks,
                 gridDim.x - row_blocks);
}

// bf16 [rows, cols] = e2m1(q) * s for every block (exact); S_dec is left to the GEMM.
__global__ __launch_bounds__(kNT) void nvfp4_dequant_kernel(const uint8_t* __restrict__ q,
                                                            const uint8_t* __restrict__ scales,
                                                            int64_t nblk,
                                                            uint16_t* __restrict__ out) {
  for (int64_t b = (int64_t)blockIdx.x * kNT + threadIdx.x; b < nblk;
       b += (int64_t)gridDim.x * kNT) {
    const uint2 c = *reinterpret_cast<const uint2*>(q + b * 8);
    const float s = e4m3_value(scales[b]);
    uint4* dst = reinterpret_cast<uint4*>(out + b * 16);
    dst[0] = dequant8(c.x, s);
    dst[1] = dequant8(c.y, s);
  }
}

unsigned stream_grid(int64_t items) {
  int64_t g = (items + kNT - 1) / kNT;
  if (g < 1) g = 1;
  return (unsigned)(g < kMaxNvfp4Blocks ? g : kMaxNvfp4Blocks);
}

}  // namespace
}  // namespace bf8

using namespace bf8;

// Argument checks shared by the NVFP4 quantize entry points (before anything launches).
static int nvfp4_args(const char* who, const void* x, int64_t rows, int64_t cols,
                      const uint8_t* out, const uint8_t* out_scales, const uint8_t* out_t,
                      const uint8_t* out_t_scales, const float* meta) {
  BF8_CHECK(rows >= 0 && cols >= 0, "%s: negative shape", who);
  BF8_CHECK(out || out_t, "%s: out and out_t are both NULL", who);
  BF8_CHECK(!out || (out_scales && cols % 16 == 0),
            "%s: rowwise blocks need cols %% 16 == 0 (got %lld) and scales", who,
            (long long)cols);
  BF8_CHECK(!out_t || (out_t_scales && rows % 16 == 0),
            "%s: columnwise blocks need rows %% 16 == 0 (got %lld) and scales", who,
            (long long)rows);
  BF8_CHECK(meta != nullptr, "%s: meta is NULL", who);
  BF8_CHECK(((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 7) == 0 && ((uintptr_t)out_t & 7) == 0,
            "%s: x must be 16-byte and out, out_t 8-byte aligned", who);
  BF8_CHECK(rows * cols == 0 || x != nullptr, "%s: x is NULL", who);
  return BF8_OK;
}

// Columnwise codes alone of at most this many elements take the columns kernel, one block of 16
// values per thread: the tile kernel's 128 x 128 tiles leave most CUs idle and its code is long.
// Tile / columns kernel, us, inputs not seen before: 64 x 640 5.3 / 3.4, 320 x 2048 5.9 / 4.0,
// 1216 x 2048 6.7 / 5.9, 3584 x 2048 9.3 / 10.4, 2304 x 2560 9.1 / 11.1.
constexpr int64_t kMaxColsKernel = 4 << 20;
// Both copies, the columnwise one as codes: the same with the rows kernel's work beside it, where
// the second read of x costs less than the idle CUs. Tile / pair kernel, us, likewise: 32 x 2560
// 7.2 / 3.6, 736 x 1024 7.5 / 4.4, 800 x 2560 8.0 / 6.2, 1792 x 2048 8.9 / 8.2, 256 x 16384 9.2 /
// 8.2, 1312 x 3584 11.2 / 12.6, 1664 x 3584 11.5 / 14.4. (One launch a copy at 32 x 2560: 6.7.)
constexpr int64_t kMaxPairKernel = kMaxColsKernel;

// The rowwise and/or columnwise casts, the per-tensor amax reduced from np partials (maxima
// of |x| as fp32 bits) that are already written.
static int nvfp4_casts(const void* x, const NvTile& p, const uint32_t* partials, int64_t np,
                       float* meta, hipStream_t s) {
  if (!p.out_t && !p.deq_t) {
    hipLaunchKernelGGL(nvfp4_rows_kernel, dim3(stream_grid(p.rows * p.cols / 16)), dim3(kNT), 0, s,
                       (const uint16_t*)x, p, partials, np, meta);
    return launch_status("nvfp4_rows_kernel");
  }
  if (p.cols % 8 != 0)  // rows of broken vectors: only columnwise codes take these shapes
    BF8_CHECK(!p.deq_t, "nvfp4: a columnwise dequantization needs cols %% 8 == 0 (got %lld)",
              (long long)p.cols);
  if (p.cols % 8 != 0 || (!p.out && !p.deq && !p.deq_t && p.rows * p.cols <= kMaxColsKernel)) {
    hipLaunchKernelGGL(nvfp4_cols_kernel, dim3(stream_grid(p.rows * p.cols / 16)), dim3(kNT), 0, s,
                       (const uint16_t*)x, p.rows, p.cols, partials, np, meta, p.out_t,
                       p.scales_t);
    return launch_status("nvfp4_cols_kernel");
  }
  if ((p.out || p.deq) && !p.deq_t && p.rows * p.cols <= kMaxPairKernel) {
    const unsigned half = stream_grid(p.rows * p.cols / 16);
    hipLaunchKernelGGL(nvfp4_pair_kernel, dim3(2 * half), dim3(kNT), 0, s, (const uint16_t*)x, p,
                       partials, np, meta, (int)half);
    return launch_status("nvfp4_pair_kernel");
  }
  const int64_t tiles = ((p.rows + kNT4 - 1) / kNT4) * ((p.cols + kNT4 - 1) / kNT4);
  const unsigned grid = (unsigned)(tiles < kMaxNvTileBlocks ? tiles : kMaxNvTileBlocks);
  hipLaunchKernelGGL(nvfp4_tile_kernel, dim3(grid), dim3(kNT), 0, s, (const uint16_t*)x, p,
                     partials, np, meta);
  return launch_status("nvfp4_tile_kernel");
}

extern "C" {

int bf8_quantize_nvfp4_partials_bf16(const void* x, int64_t rows, int64_t cols,
                                     const uint32_t* partials, int64_t n_partials, uint8_t* out,
                                     uint8_t* out_scales, uint8_t* out_t, uint8_t* out_t_scales,
                                     float* meta, void* stream) {
  const char* who = "bf8_quantize_nvfp4_partials_bf16";
  int rc = nvfp4_args(who, x, rows, cols, out, out_scales, out_t, out_t_scales, meta);
  if (rc != BF8_OK) return rc;
  BF8_CHECK(partials && n_partials >= 1, "%s: partials is NULL or empty", who);
  if (rows * cols == 0) return BF8_OK;
  return nvfp4_casts(x, NvTile{rows, cols, out, out_scales, nullptr, out_t, out_t_scales, nullptr},
                     partials, n_partials, meta, as_stream(stream));
}

int bf8_quantize_nvfp4_bf16(const void* x, int64_t rows, int64_t cols, uint8_t* out,
                            uint8_t* out_scales, uint8_t* out_t, uint8_t* out_t_scales,
                            float* meta, uint32_t* partials, void* stream) {
  const char* who = "bf8_quantize_nvfp4_bf16";
  int rc = nvfp4_args(who, x, rows, cols, out, out_scales, out_t, out_t_scales, meta);
  if (rc != BF8_OK) return rc;
  BF8_CHECK(partials, "%s: partials is NULL", who);
  const int64_t n = rows * cols;
  if (n == 0) return BF8_OK;
  rc = bf8_amax_bf16(x, n, partials, stream);
  if (rc != BF8_OK) return rc;
  return nvfp4_casts(x, NvTile{rows, cols, out, out_scales, nullptr, out_t, out_t_scales, nullptr},
                     partials, bf8_amax_partials(n), meta, as_stream(stream));
}

static int nvfp4_dequant_entry(const char* who, const void* x, int64_t rows, int64_t cols,
                               uint32_t* partials, int64_t n_partials, void* deq, void* deq_t,
                               uint8_t* out_t, uint8_t* out_t_scales, float* meta, void* stream) {
  BF8_CHECK(rows >= 0 && cols >= 0, "%s: negative shape", who);
  BF8_CHECK(deq != nullptr || deq_t != nullptr, "%s: deq and deq_t are both NULL", who);
  BF8_CHECK(!deq || cols % 16 == 0, "%s: needs cols %% 16 == 0 (got %lld)", who, (long long)cols);
  BF8_CHECK(!out_t || !deq_t, "%s: give out_t or deq_t", who);
  BF8_CHECK(!out_t || (out_t_scales && rows % 16 == 0),
            "%s: columnwise blocks need rows %% 16 == 0 (got %lld) and scales", who,
            (long long)rows);
  BF8_CHECK(!deq_t || (rows % 16 == 0 && cols % 8 == 0),
            "%s: deq_t needs rows %% 16 == 0 and cols %% 8 == 0 (got %lld x %lld)", who,
            (long long)rows, (long long)cols);
  BF8_CHECK(meta != nullptr && partials != nullptr && n_partials >= 0,
            "%s: meta or partials is NULL", who);
  BF8_CHECK((((uintptr_t)x | (uintptr_t)deq | (uintptr_t)deq_t) & 15) == 0 &&
                ((uintptr_t)out_t & 7) == 0,
            "%s: x and deq must be 16-byte and out_t 8-byte aligned", who);
  BF8_CHECK(rows * cols == 0 || x != nullptr, "%s: x is NULL", who);
  int rc = BF8_OK;
  const int64_t n = rows * cols;
  if (n == 0) return BF8_OK;
  if (n_partials == 0) {
    rc = bf8_amax_bf16(x, n, partials, stream);
    if (rc != BF8_OK) return rc;
    n_partials = bf8_amax_partials(n);
  }
  return nvfp4_casts(x,
                     NvTile{rows, cols, nullptr, nullptr, (uint16_t*)deq, out_t, out_t_scales,
                            (uint16_t*)deq_t},
                     partials, n_partials, meta, as_stream(stream));
}

int bf8_quantize_nvfp4_dequant_bf16(const void* x, int64_t rows, int64_t cols,
                                    uint32_t* partials, int64_t n_partials, void* deq,
                                    uint8_t* out_t, uint8_t* out_t_scales, float* meta,
                                    void* stream) {
  const char* who = "bf8_quantize_nvfp4_dequant_bf16";
  BF8_CHECK(deq != nullptr && cols % 16 == 0, "%s: needs deq and cols %% 16 == 0 (got %lld)", who,
            (long long)cols);
  return nvfp4_dequant_entry(who, x, rows, cols, partials, n_partials, deq, nullptr, out_t,
                             out_t_scales, meta, stream);
}

int bf8_quantize_nvfp4_dequant2_bf16(const void* x, int64_t rows, int64_t cols,
                                     uint32_t* partials, int64_t n_partials, void* deq,
                                     void* deq_t, uint8_t* out_t, uint8_t* out_t_scales,
                                     float* meta, void* stream) {
  return nvfp4_dequant_entry("bf8_quantize_nvfp4_dequant2_bf16", x, rows, cols, partials,
                             n_partials, deq, deq_t, out_t, out_t_scales, meta, stream);
}

int bf8_dequant_nvfp4(const uint8_t* q, const uint8_t* scales, int64_t rows, int64_t cols,
                      void* out, void* stream) {
  BF8_CHECK(rows >= 0 && cols >= 0 && cols % 16 == 0,
            "bf8_dequant_nvfp4: need cols %% 16 == 0 (got %lld)", (long long)cols);
  BF8_CHECK(((uintptr_t)q & 7) == 0 && ((uintptr_t)out & 15) == 0,
            "bf8_dequant_nvfp4: q must be 8-byte and out 16-byte aligned");
  const int64_t nblk = rows * (cols / 16);
  if (nblk == 0) return BF8_OK;
  BF8_CHECK(q && scales && out, "bf8_dequant_nvfp4: NULL pointer");
  hipLaunchKernelGGL(nvfp4_dequant_kernel, dim3(stream_grid(nblk)), dim3(kNT), 0,
                     as_stream(stream), q, scales, nblk, (uint16_t*)out);
  return launch_status("nvfp4_dequant_kernel");
}

}  // extern "C"
