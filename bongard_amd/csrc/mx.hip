// MXFP8 quantization (OCP microscaling: blocks of 32 elements sharing one E8M0 scale) for
// gfx950, the arithmetic of TransformerEngine's MXFP8BlockScaling recipe (TE 2.19.0, the
// recipe named at bongard/te_linear.py:17,38-39 and bongard/fused_mlp.py:9,31-33).
//
// Per block of 32 bf16 values (along a row for the rowwise copy, along a column for the
// columnwise copy):
//   amax = max |x| (NaN-propagating), val = fp32(amax * fp32(1 / fp8_max)),
//   e    = E8M0 of val rounded up to a power of two (ceil; 0xFE at most; NaN -> 0xFF),
//   q    = fp8(clamp(f32(x) * 2^(127 - e), +-fp8_max)),
// so that the block's largest magnitude lands in (fp8_max / 2, fp8_max] and x ~ q * 2^(e-127).
// Scales are stored one byte per block, rows of bf8_mx_scale_ld(K) bytes (a multiple of 4;
// the bytes past the last block hold 127 = 1.0 so that the GEMM can read whole dwords).
// The columnwise copy is stored transposed ([cols, rows], blocks along rows of x), the
// K-contiguous operand layout of the TN GEMM.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "gelu.hpp"

namespace bf8 {
namespace {

constexpr int kMxNT = 256;
constexpr int kMT = 128;               // tile of the two-copy kernel (rows x cols)
constexpr int kMaxMxTileBlocks = 2048;
constexpr int kMaxMxRowBlocks = 8192;
// Exponents (mx_exponent) of two packed |x| maxima given as finite bf16 keys: fp8_max is
// 1.75 x 2^S, so amax / fp8_max rounds up to a power of two with exponent E - S where the
// mantissa is at most 1.75 (96 / 128 above 1) and E - S + 1 past it, i.e. ((key + 31) >> 7) - S,
// at least 0 (equal to mx_exponent on every finite key).
template <int FMT>
__device__ __forceinline__ uint32_t mx_exponent_finite_pk(uint32_t keys) {
  constexpr unsigned short S = FMT == BF8_E4M3 ? 8 : 15;
  const u16x2 lim = {S, S};
  u16x2 k = __builtin_bit_cast(u16x2, keys);
  k = (u16x2)((u16x2)(k + (u16x2){31, 31}) >> 7);
  k = (u16x2)(__builtin_elementwise_max(k, lim) - lim);
  return __builtin_bit_cast(uint32_t, k);
}

// Quantizes 8 bf16 values with their own multipliers. FINITE: none of the values is inf or
// NaN, so no product leaves +-fp8_max.
template <int FMT, bool FINITE>
__device__ __forceinline__ uint2 mx_quant8_vs(uint4 v, const float* s) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t q[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float x0 = bf16_lo(w[2 * k]), x1 = bf16_hi(w[2 * k]);
    const float x2 = bf16_lo(w[2 * k + 1]), x3 = bf16_hi(w[2 * k + 1]);
    const float* t = s + 4 * k;
    if constexpr (FINITE) {
      q[k] = quant4_finite<FMT, false>(x0 * t[0], x1 * t[1], x2 * t[2], x3 * t[3]);
    } else {
      q[k] = quant4<FMT>(x0 * t[0], x1 * t[1], x2 * t[2], x3 * t[3], x0, x1, x2, x3, t[0]);
      // quant4 signs a NaN product by one scale: redo those by their own column's
      const float xs[4] = {x0, x1, x2, x3};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float pr = xs[e] * t[e];
        if (__builtin_expect(pr != pr, 0))
          q[k] = (q[k] & ~(0xFFu << (8 * e))) | (nan_byte(xs[e], t[e]) << (8 * e));
      }
    }
  }
  return make_uint2(q[0], q[1]);
}

// Both copies of x in one pass, or the columnwise one. A block takes 128 x 128 tiles, each wave 32 rows of
// all 128 columns: lane l holds columns 8 (l & 15) .. +7 of the rows 4 k + l / 16, k < 8, so a
// row block of 32 is four neighbouring lanes (two DPP exchanges) and a column block of 32 rows is
// the wave's eight pieces and the four lanes of a column group (two lane exchanges of packed
// 16-bit maxima). The columnwise bytes meet in LDS; each wave then turns 32 columns of all 128
// rows. Every store instruction of either output writes whole 128-byte lines, and a scale dword
// holds the four blocks of 128 K-values: rows of bytes (sc) and / or planes, one dword per row
// and group of 128 (the layout the GEMM loads in whole lines).
// HBM-bound: 2 B read, 1 B (+ 1/32) written per element and copy; x is read once for the two
// copies, where a rowwise and a columnwise pass read it twice. Both copies, inputs rotated past
// the MALL: [4096, 20480] 133.1 us in two passes, 78.4 us in one (4.3 TB/s); [20480, 2560]
// 72.9 -> 45.4 us (4.7 TB/s); one pass over 64 x 64 tiles per wave, whose stores are half
// lines, 99.7 and 56.3 us. With planes in place of the scale rows' scattered dwords 75.2 and
// 43.0 us. The rowwise copy alone is mx_rows_kernel's, a small tensor's copies mx_wave_kernel's.
struct MxTile {
  const uint16_t* x;
  int64_t rows, cols;
  uint8_t* out;
  uint8_t* sc;
  uint32_t* planes;
  int64_t ld_sc;
  uint8_t* out_t;
  uint8_t* sc_t;
  uint32_t* planes_t;
  int64_t ld_sc_t;
  int fmt;
};

constexpr int kMPitch = kMT / 4 + 1;  // dwords per staged row (odd)

template <int FMT, bool FINITE>
__device__ __forceinline__ void mx_tile_body(const MxTile& p, int64_t r0, int64_t c0,
                                             const uint4 (&v)[8], const uint32_t (&rk)[8],
                                             const uint32_t (&cm)[4], uint32_t* stage,
                                             uint32_t* erow, uint8_t* ecol, int wid, int lane) {
  const int cl = lane & 15, lr = lane >> 4;
  const int64_t c = c0 + 8 * cl;
  const int64_t wr0 = r0 + 32 * wid;
  if (p.out) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t r = wr0 + 4 * k + lr;
      uint32_t e;
      if constexpr (FINITE)
        e = mx_exponent_finite_pk<FMT>(rk[k]) & 0xFFFFu;
      else
        e = mx_exponent<FMT>(rk[k] << 16);
      if (r < p.rows && c < p.cols) {
        const float mult = mx_multiplier(e);
        *reinterpret_cast<uint2*>(p.out + r * p.cols + c) =
            FINITE ? quant8_bf16_finite<FMT, false>(v[k], mult) : quant8_bf16<FMT>(v[k], mult);
      }
      if (c >= p.cols) e = kMxPadScale;  // blocks past the row pad its last dword of scales
      // lanes 0, 4, 8, 12 of the 16 hold the four blocks: gather into lane 0
      e |= (uint32_t)__shfl_down((int)e, 4, 64) << 8;
      e |= (uint32_t)__shfl_down((int)e, 8, 64) << 16;
      if (cl == 0) {
        erow[32 * wid + 4 * k + lr] = e;
        if (p.sc && r < p.rows)
          *reinterpret_cast<uint32_t*>(p.sc + r * p.ld_sc + (c0 >> 5)) = e;
      }
    }
    // the wave's own 32 dwords as one line of the plane (a wave's LDS accesses are in order)
    if (p.planes && lane < 32 && wr0 + lane < p.rows)
      p.planes[(c0 >> 7) * p.rows + wr0 + lane] = erow[32 * wid + lane];
  }
  if (!p.out_t) return;
  float s[8];
  uint32_t ex[4];  // packed pairs of the lane's column exponents
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (FINITE)
      ex[i] = mx_exponent_finite_pk<FMT>(cm[i]);
    else
      ex[i] = mx_exponent<FMT>(cm[i] << 16) | (mx_exponent<FMT>(cm[i] & 0xFFFF0000u) << 16);
    s[2 * i] = mx_multiplier(ex[i] & 0xFFFFu);
    s[2 * i + 1] = mx_multiplier(ex[i] >> 16);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint2 q = mx_quant8_vs<FMT, FINITE>(v[k], s);
    uint32_t* d = stage + (32 * wid + 4 * k + lr) * kMPitch + 2 * cl;
    d[0] = q.x;
    d[1] = q.y;
  }
  if (lr == 0) {
    const bool valid = wr0 < p.rows;  // rows % 32 == 0: the wave's block is whole or absent
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ecol[(8 * cl + 2 * i) * 4 + wid] = valid ? (uint8_t)ex[i] : (uint8_t)kMxPadScale;
      ecol[(8 * cl + 2 * i + 1) * 4 + wid] = valid ? (uint8_t)(ex[i] >> 16) : (uint8_t)kMxPadScale;
    }
  }
}

// The loaded tile at (r0, c0), by four waves (wid 0 .. 3) that share stage, erow and ecol; every
// wave of the block calls it alike. A tile with r0 >= p.rows writes nothing.
template <int FMT>
__device__ __forceinline__ void mx_tile_finish(const MxTile& p, int64_t r0, int64_t c0,
                                               const uint4 (&v)[8], uint32_t* stage,
                                               uint32_t* erow, uint32_t* ecol, int wid, int lane) {
  uint32_t rk[8], cm[4] = {};
  uint32_t top = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t a[4] = {v[k].x & 0x7FFF7FFFu, v[k].y & 0x7FFF7FFFu, v[k].z & 0x7FFF7FFFu,
                           v[k].w & 0x7FFF7FFFu};
#pragma unroll
    for (int i = 0; i < 4; ++i) cm[i] = pk_max_u16(cm[i], a[i]);
    uint32_t m = pk_max_u16(pk_max_u16(a[0], a[1]), pk_max_u16(a[2], a[3]));
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, true));
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4E, 0xF, 0xF, true));
    rk[k] = max(m & 0xFFFFu, m >> 16);
    top = max(top, rk[k]);
  }
  if (p.out_t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cm[i] = pk_max_u16(cm[i], (uint32_t)__shfl_xor((int)cm[i], 16, 64));
      cm[i] = pk_max_u16(cm[i], (uint32_t)__shfl_xor((int)cm[i], 32, 64));
    }
  }
  uint8_t* ecolb = reinterpret_cast<uint8_t*>(ecol);
  if (__builtin_expect(__any(top >= 0x7F80u), 0))
    mx_tile_body<FMT, false>(p, r0, c0, v, rk, cm, stage, erow, ecolb, wid, lane);
  else
    mx_tile_body<FMT, true>(p, r0, c0, v, rk, cm, stage, erow, ecolb, wid, lane);
  if (!p.out_t) return;
  __syncthreads();
  {
    // lane: 16 rows (lane & 7) x 4 columns (lane >> 3) of the wave's 32 columns
    const int rg = (lane & 7) * 16, cg = 8 * wid + (lane >> 3);
    uint32_t d[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = stage[(rg + i) * kMPitch + cg];
    uint4 tq[4];
    transpose_4x16(d, tq);
    const int64_t tc = r0 + rg;  // column of out_t (a row of x)
    if (tc < p.rows) {
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        const int64_t tr = c0 + 4 * cg + cc;  // row of out_t (a column of x)
        if (tr < p.cols) *reinterpret_cast<uint4*>(p.out_t + tr * p.rows + tc) = tq[cc];
      }
    }
    const int tid = 64 * wid + lane;
    if (tid < kMT && c0 + tid < p.cols && r0 < p.rows) {
      // four blocks of one column; the last tile row's absent blocks pad the last dword
      const uint32_t e4 = ecol[tid];
      if (p.planes_t) p.planes_t[(r0 >> 7) * p.cols + c0 + tid] = e4;
      if (p.sc_t) {
        uint8_t* dst = p.sc_t + (c0 + tid) * p.ld_sc_t + (r0 >> 5);
        if (((uintptr_t)p.sc_t & 3) == 0) {
          *reinterpret_cast<uint32_t*>(dst) = e4;
        } else {
#pragma unroll
          for (int b = 0; b < 4; ++b) dst[b] = (uint8_t)(e4 >> (8 * b));
        }
      }
    }
  }
  __syncthreads();
}

// The tiles blk, blk + nblk, .. of p (every thread of the block calls it alike).
template <int FMT>
__device__ __forceinline__ void mx_tiles(const MxTile& p, int64_t blk, int64_t nblk,
                                         uint32_t* stage, uint32_t* erow, uint32_t* ecol) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t tiles_c = (p.cols + kMT - 1) / kMT, tiles_r = (p.rows + kMT - 1) / kMT;
  const int64_t ntiles = tiles_c * tiles_r;
  const int cl = lane & 15, lr = lane >> 4;
  for (int64_t t = blk; t < ntiles; t += nblk) {
    const int64_t r0 = (t / tiles_c) * kMT, c0 = (t % tiles_c) * kMT;
    const int64_t c = c0 + 8 * cl;
    uint4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t r = r0 + 32 * wid + 4 * k + lr;
      v[k] = make_uint4(0u, 0u, 0u, 0u);
      if (r < p.rows && c < p.cols)
        v[k] = *reinterpret_cast<const uint4*>(p.x + r * p.cols + c);
    }
    mx_tile_finish<FMT>(p, r0, c0, v, stage, erow, ecol, wid, lane);
  }
}

// d_g (G) or d_u of 8 elements: the chain of geglu_bwd8, one half of it.
template <bool G>
__device__ __forceinline__ uint4 geglu_bwd8_half(uint4 dh, uint4 g, uint4 u, const uint16_t* ta,
                                                 const uint32_t* tf) {
  const uint32_t dw[4] = {dh.x, dh.y, dh.z, dh.w}, gw[4] = {g.x, g.y, g.z, g.w};
  const uint32_t uw[4] = {u.x, u.y, u.z, u.w};
  uint32_t outside = 0, ix[4], t[8], o[4];
#pragma unroll
  for (int w = 0; w < 4; ++w)
    ix[w] = G ? gelu_factor_index2(gw[w], outside) : gelu_index2(gw[w], outside);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    t[2 * w] = G ? tf[ix[w] & 0xFFFFu] : ta[ix[w] & 0xFFFFu];
    t[2 * w + 1] = G ? tf[ix[w] >> 16] : ta[ix[w] >> 16];
  }
  if (__builtin_expect(__any(outside != 0), 0)) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      t[2 * w] = G ? gelu_factor_finish(gw[w], t[2 * w]) : gelu_finish(gw[w], t[2 * w]);
      t[2 * w + 1] = G ? gelu_factor_finish(gw[w] >> 16, t[2 * w + 1])
                       : gelu_finish(gw[w] >> 16, t[2 * w + 1]);
    }
  }
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float d0 = bf16_lo(dw[w]), d1 = bf16_hi(dw[w]);
    if constexpr (G) {
      const uint32_t da = pack_bf16x2(d0 * bf16_lo(uw[w]), d1 * bf16_hi(uw[w]));
      o[w] = pack_bf16x2(bf16_lo(da) * __uint_as_float(t[2 * w]),
                         bf16_hi(da) * __uint_as_float(t[2 * w + 1]));
    } else {
      const uint32_t a = t[2 * w] | (t[2 * w + 1] << 16);
      o[w] = pack_bf16x2(d0 * bf16_lo(a), d1 * bf16_hi(a));
    }
    o[w] = nan_ffff_bf16x2(o[w]);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// d_g or d_u of the lane's eight rows 4 k of a tile, in two batches of loads.
template <bool G>
__device__ __forceinline__ void geglu_bwd_rows(const uint16_t* dp, const uint16_t* gp, int64_t I,
                                               int64_t rows_left, const uint16_t* ta,
                                               const uint32_t* tf, uint4 (&v)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    uint4 d[4], g[4], u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int row = 4 * (4 * q + k);
      d[k] = g[k] = u[k] = make_uint4(0u, 0u, 0u, 0u);
      if (row < rows_left) {
        d[k] = *reinterpret_cast<const uint4*>(dp + row * I);
        g[k] = *reinterpret_cast<const uint4*>(gp + row * 2 * I);
        if (G) u[k] = *reinterpret_cast<const uint4*>(gp + row * 2 * I + I);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) v[4 * q + k] = geglu_bwd8_half<G>(d[k], g[k], u[k], ta, tf);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The gated-GELU backward fused with the quantization of its output: dGU [M, 2I] of dH [M, I]
// and GU [M, 2I] goes from registers to its MX copies (p: rows M, cols 2I; I % 128 == 0), the
// bf16 dGU itself is never written. The first four waves of a block take the d_g tile of a
// 128 x 128 tile of I, the others its d_u tile: neither holds both (one wave holding d_g and d_u
// spilled 140 registers), and dH and g come from the CU's own cache the second time. The gelu
// tables (39 KB of LDS) and two stages let two blocks, 16 waves, run on a CU.
// HBM-bound: 6 B read, 4 B (+ 1/8) written per element of H, where the two passes read 10 B and
// wrote 8. [4096, 10240]: 73 + 72 us in two passes, 126 in one (3.4 TB/s: at 16 waves a CU the
// table lookups and the turning are not all hidden; loading the next tile during them spilled).
constexpr int kBwdNT = 512;
constexpr int kMaxBwdBlocks = 512;
template <int FMT>
__global__ __launch_bounds__(kBwdNT, 4) void geglu_bwd_mx_kernel(
    const uint16_t* __restrict__ dH, const uint16_t* __restrict__ GU, int64_t I, MxTile p) {
  __shared__ __attribute__((aligned(16))) uint16_t ta[kGeluABytes / 2];
  __shared__ __attribute__((aligned(16))) uint32_t tf[kGeluFBytes / 4];
  __shared__ uint32_t stage[2][kMT * kMPitch];
  __shared__ uint32_t erow[2][kMT], ecol[2][kMT];
  load_gelu_tables<kBwdNT>(ta, tf);
  __syncthreads();
  const int lane = threadIdx.x & 63, wid = (threadIdx.x >> 6) & 3;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int64_t tiles_c = I / kMT, tiles_r = (p.rows + kMT - 1) / kMT;
  const int64_t ntiles = tiles_c * tiles_r;
  const int cl = lane & 15, lr = lane >> 4;
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int64_t r0 = (t / tiles_c) * kMT, c0 = (t % tiles_c) * kMT;
    const int64_t rw = r0 + 32 * wid + lr;
    const uint16_t* dp = dH + rw * I + c0 + 8 * cl;
    const uint16_t* gp = GU + rw * 2 * I + c0 + 8 * cl;
    uint4 v[8];
    if (half == 0)
      geglu_bwd_rows<true>(dp, gp, I, p.rows - rw, ta, tf, v);
    else
      geglu_bwd_rows<false>(dp, gp, I, p.rows - rw, ta, tf, v);
    mx_tile_finish<FMT>(p, r0, half * I + c0, v, stage[half], erow[half], ecol[half], wid, lane);
  }
}

template <int FMT>
__global__ __launch_bounds__(kMxNT) void mx_tile_kernel(MxTile p) {
  __shared__ uint32_t stage[kMT * kMPitch];
  __shared__ uint32_t erow[kMT], ecol[kMT];  // scale dwords of the tile's rows and columns
  mx_tiles<FMT>(p, blockIdx.x, gridDim.x, stage, erow, ecol);
}

// Rowwise quantization of a wave's 4 LR rows x 128 columns: lane l holds columns 8 (l & 15) .. +7
// of the rows LR (l / 16) + k, k < LR (rk: the maximum of its block of 32, a bf16 key).
template <int FMT, bool FINITE, int LR>
__device__ __forceinline__ void mx_rows_body(const MxTile& p, int64_t r0, int64_t c0,
                                             const uint4 (&v)[LR], const uint32_t (&rk)[LR],
                                             int lane) {
  const int cl = lane & 15;
  const int64_t c = c0 + 8 * cl, rl = r0 + LR * (lane >> 4);
  uint32_t mine = 0;  // the scale dword of row rl + cl, in the lanes cl < LR
#pragma unroll
  for (int k = 0; k < LR; ++k) {
    uint32_t e;
    if constexpr (FINITE)
      e = mx_exponent_finite_pk<FMT>(rk[k]) & 0xFFFFu;
    else
      e = mx_exponent<FMT>(rk[k] << 16);
    if (rl + k < p.rows && c < p.cols) {
      const float mult = mx_multiplier(e);
      *reinterpret_cast<uint2*>(p.out + (rl + k) * p.cols + c) =
          FINITE ? quant8_bf16_finite<FMT, false>(v[k], mult) : quant8_bf16<FMT>(v[k], mult);
    }
    if (c >= p.cols) e = kMxPadScale;  // blocks past the row pad its last dword of scales
    e <<= 8 * (cl >> 2);
    e |= (uint32_t)__shfl_xor((int)e, 4, 64);
    e |= (uint32_t)__shfl_xor((int)e, 8, 64);
    if (cl == k) mine = e;
  }
  const int64_t r = rl + cl;
  if (cl < LR && r < p.rows) {
    if (p.planes) p.planes[(c0 >> 7) * p.rows + r] = mine;
    if (p.sc) *reinterpret_cast<uint32_t*>(p.sc + r * p.ld_sc + (c0 >> 5)) = mine;
  }
}

template <int FMT, int LR>
__device__ __forceinline__ void mx_rows(const MxTile& p, int64_t blk, int64_t nblk) {
  const int lane = threadIdx.x & 63;
  // wave-uniform 32-bit tile arithmetic (a tile is 512 LR elements)
  const uint32_t groups = (uint32_t)((p.cols + kMT - 1) / kMT);
  const uint32_t ntiles = groups * (uint32_t)((p.rows + LR * 4 - 1) / (LR * 4));
  const uint32_t wid = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (uint32_t t = (uint32_t)blk * (kMxNT / 64) + wid; t < ntiles;
       t += (uint32_t)nblk * (kMxNT / 64)) {
    const int64_t r0 = (int64_t)(t / groups) * (LR * 4), c0 = (int64_t)(t % groups) * kMT;
    const int64_t c = c0 + 8 * (lane & 15), rl = r0 + LR * (lane >> 4);
    uint4 v[LR];
#pragma unroll
    for (int k = 0; k < LR; ++k) {
      v[k] = make_uint4(0u, 0u, 0u, 0u);
      if (rl + k < p.rows && c < p.cols)
        v[k] = *reinterpret_cast<const uint4*>(p.x + (rl + k) * p.cols + c);
    }
    uint32_t rk[LR], top = 0;
#pragma unroll
    for (int k = 0; k < LR; ++k) {
      uint32_t m = pk_max_u16(pk_max_u16(v[k].x & 0x7FFF7FFFu, v[k].y & 0x7FFF7FFFu),
                              pk_max_u16(v[k].z & 0x7FFF7FFFu, v[k].w & 0x7FFF7FFFu));
      m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, true));
      m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4E, 0xF, 0xF, true));
      rk[k] = max(m & 0xFFFFu, m >> 16);
      top = max(top, rk[k]);
    }
    if (__builtin_expect(__any(top >= 0x7F80u), 0))
      mx_rows_body<FMT, false, LR>(p, r0, c0, v, rk, lane);
    else
      mx_rows_body<FMT, true, LR>(p, r0, c0, v, rk, lane);
  }
}

// The rowwise copy alone. Memory-bound like the tile kernel, whose registers and LDS for the
// columnwise copy hold it to 4 waves per SIMD; this one runs 8 (59 VGPRs, no LDS). Planes only,
// inputs repeated / rotated past the MALL, tile kernel -> this one: [4096, 10240] 24.4 / 26.5 ->
// 20.8 / 22.3 us (5.7 TB/s), [20480, 2560] 27.9 / 29.7 -> 24.9 / 26.5, [8192, 2560] 15.0 / 16.7 ->
// 11.5 / 13.1; with scale rows as well 27.9 / 29.4 -> 22.0 / 23.4. Eight rows per lane (94 VGPRs)
// 22.8 / 24.7 us at [4096, 10240], two 20.1 / 23.0.
// Small tensors take one row per lane, four times the waves (kMxSmallRows).
constexpr int kLR = 4;
template <int FMT, int LR>
__global__ __launch_bounds__(kMxNT) void mx_rows_kernel(MxTile p) {
  mx_rows<FMT, LR>(p, blockIdx.x, gridDim.x);
}

// Both copies, or the columnwise one, of a small tensor: one wave per block takes 32 rows x 64
// columns, so that the waves outnumber the CUs from 0.5M elements on, where the 128 x 128 tiles of
// four waves leave most CUs idle. Lane l holds columns 8 (l & 7) .. +7 of the rows 8 k + l / 8,
// k < 4; the wave holds whole blocks in both directions, and turns its bytes in its own LDS.
// Latency-bound: scales leave as bytes and the columnwise copy in 32-byte pieces, which the L2
// gathers while the tensor fits there.
template <int FMT, bool FINITE>
__device__ __forceinline__ void mx_wave_body(const MxTile& p, int64_t r0, int64_t c0,
                                             const uint4 (&v)[4], const uint32_t (&rk)[4],
                                             const uint32_t (&cm)[4], uint32_t* stage, int lane) {
  const int cl = lane & 7, lr = lane >> 3;
  const int64_t c = c0 + 8 * cl;
  if (p.out && c < p.cols) {
    const int64_t blk = c >> 5, nblk = p.cols >> 5;
    // the block that ends a row also pads its last dword of scales
    const int64_t end = blk == nblk - 1 ? (nblk + 3) & ~3LL : blk + 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t r = r0 + 8 * k + lr;
      if (r >= p.rows) break;
      uint32_t e;
      if constexpr (FINITE)
        e = mx_exponent_finite_pk<FMT>(rk[k]) & 0xFFFFu;
      else
        e = mx_exponent<FMT>(rk[k] << 16);
      const float mult = mx_multiplier(e);
      *reinterpret_cast<uint2*>(p.out + r * p.cols + c) =
          FINITE ? quant8_bf16_finite<FMT, false>(v[k], mult) : quant8_bf16<FMT>(v[k], mult);
      if ((cl & 3) == 0) {
        for (int64_t b = blk; b < end; ++b) {
          const uint8_t byte = b == blk ? (uint8_t)e : (uint8_t)kMxPadScale;
          if (p.sc) p.sc[r * p.ld_sc + b] = byte;
          if (p.planes) reinterpret_cast<uint8_t*>(p.planes + (b >> 2) * p.rows + r)[b & 3] = byte;
        }
      }
    }
  }
  if (!p.out_t) return;
  float s[8];
  uint32_t ex[4];  // packed pairs of the lane's column exponents
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (FINITE)
      ex[i] = mx_exponent_finite_pk<FMT>(cm[i]);
    else
      ex[i] = mx_exponent<FMT>(cm[i] << 16) | (mx_exponent<FMT>(cm[i] & 0xFFFF0000u) << 16);
    s[2 * i] = mx_multiplier(ex[i] & 0xFFFFu);
    s[2 * i + 1] = mx_multiplier(ex[i] >> 16);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint2 q = mx_quant8_vs<FMT, FINITE>(v[k], s);
    uint32_t* d = stage + (8 * k + lr) * kWaveTilePitch + 2 * cl;
    d[0] = q.x;
    d[1] = q.y;
  }
  // lane (cl, lr) stores the scale of column c + lr, which its eight columns' lanes all hold
  if (c + lr < p.cols) {
    const uint32_t pair = lr < 4 ? (lr < 2 ? ex[0] : ex[1]) : (lr < 6 ? ex[2] : ex[3]);
    const int64_t blk = r0 >> 5, nblk = p.rows >> 5;
    const int64_t end = blk == nblk - 1 ? (nblk + 3) & ~3LL : blk + 1;
    for (int64_t b = blk; b < end; ++b) {
      const uint8_t byte = b == blk ? (uint8_t)(pair >> (16 * (lr & 1))) : (uint8_t)kMxPadScale;
      if (p.sc_t) p.sc_t[(c + lr) * p.ld_sc_t + b] = byte;
      if (p.planes_t)
        reinterpret_cast<uint8_t*>(p.planes_t + (b >> 2) * p.cols + c + lr)[b & 3] = byte;
    }
  }
}

// The wave's loaded 32 x 64 tile at (r0, c0), v[k] the lane's vector of row 8 k + l / 8 (zeros past
// p.rows or p.cols). Every wave of the block calls it alike, each with its own stage.
template <int FMT>
__device__ __forceinline__ void mx_wave_finish(const MxTile& p, int64_t r0, int64_t c0,
                                               const uint4 (&v)[4], uint32_t* stage, int lane) {
  uint32_t rk[4], cm[4] = {}, top = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t a[4] = {v[k].x & 0x7FFF7FFFu, v[k].y & 0x7FFF7FFFu, v[k].z & 0x7FFF7FFFu,
                           v[k].w & 0x7FFF7FFFu};
#pragma unroll
    for (int i = 0; i < 4; ++i) cm[i] = pk_max_u16(cm[i], a[i]);
    uint32_t m = pk_max_u16(pk_max_u16(a[0], a[1]), pk_max_u16(a[2], a[3]));
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xF, 0xF, true));
    m = pk_max_u16(m, (uint32_t)__builtin_amdgcn_mov_dpp((int)m, 0x4E, 0xF, 0xF, true));
    rk[k] = max(m & 0xFFFFu, m >> 16);
    top = max(top, rk[k]);
  }
  if (p.out_t) {
#pragma unroll
    for (int off = 8; off < 64; off <<= 1)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        cm[i] = pk_max_u16(cm[i], (uint32_t)__shfl_xor((int)cm[i], off, 64));
  }
  if (__builtin_expect(__any(top >= 0x7F80u), 0))
    mx_wave_body<FMT, false>(p, r0, c0, v, rk, cm, stage, lane);
  else
    mx_wave_body<FMT, true>(p, r0, c0, v, rk, cm, stage, lane);
  if (!p.out_t) return;
  __syncthreads();
  // lane: 8 rows (lane & 3) x 4 columns (lane >> 2)
  const int rg = (lane & 3) * 8, cg = lane >> 2;
  uint32_t t[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = stage[(rg + 4 * h + i) * kWaveTilePitch + cg];
    transpose_4x4(d, t[h]);
  }
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) {
    const int64_t tr = c0 + 4 * cg + cc;  // row of out_t (a column of x)
    if (tr < p.cols)
      *reinterpret_cast<uint2*>(p.out_t + tr * p.rows + r0 + rg) = make_uint2(t[0][cc], t[1][cc]);
  }
}

template <int FMT>
__global__ __launch_bounds__(64) void mx_wave_kernel(MxTile p) {
  __shared__ uint32_t stage[32 * kWaveTilePitch];
  const int lane = threadIdx.x, cl = lane & 7, lr = lane >> 3;
  const uint32_t tiles_c = (uint32_t)((p.cols + 63) / 64);
  const int64_t r0 = (int64_t)(blockIdx.x / tiles_c) * 32, c0 = (int64_t)(blockIdx.x % tiles_c) * 64;
  const int64_t c = c0 + 8 * cl;
  uint4 v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)  // rows % 32 == 0: whole blocks of rows
    v[k] = c < p.cols ? *reinterpret_cast<const uint4*>(p.x + (r0 + 8 * k + lr) * p.cols + c)
                      : make_uint4(0u, 0u, 0u, 0u);
  mx_wave_finish<FMT>(p, r0, c0, v, stage, lane);
}

// d_g (G) or d_u of the lane's four rows 8 k of a wave tile.
template <bool G>
__device__ __forceinline__ void geglu_bwd_wave_rows(const uint16_t* dp, const uint16_t* gp,
                                                    int64_t I, int64_t rows_left,
                                                    const uint16_t* ta, const uint32_t* tf,
                                                    uint4 (&v)[4]) {
  uint4 d[4], g[4], u[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    d[k] = g[k] = u[k] = make_uint4(0u, 0u, 0u, 0u);
    if (8 * k < rows_left) {
      d[k] = *reinterpret_cast<const uint4*>(dp + 8 * k * I);
      g[k] = *reinterpret_cast<const uint4*>(gp + 16 * k * I);
      if (G) u[k] = *reinterpret_cast<const uint4*>(gp + 16 * k * I + I);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = geglu_bwd8_half<G>(d[k], g[k], u[k], ta, tf);
}

// geglu_bwd_mx_kernel for small outputs: a block takes 32 rows x 128 columns of I, two waves their
// d_g tiles and two their d_u tiles (as mx_wave_kernel), where a tile of 128 rows keeps one CU
// busy for 12 us and leaves the others idle.
template <int FMT>
__global__ __launch_bounds__(kMxNT) void geglu_bwd_mx_wave_kernel(const uint16_t* __restrict__ dH,
                                                                  const uint16_t* __restrict__ GU,
                                                                  int64_t I, MxTile p) {
  __shared__ __attribute__((aligned(16))) uint16_t ta[kGeluABytes / 2];
  __shared__ __attribute__((aligned(16))) uint32_t tf[kGeluFBytes / 4];
  __shared__ uint32_t stage[4][32 * kWaveTilePitch];
  load_gelu_tables<kMxNT>(ta, tf);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wid >> 1;
  const uint32_t tiles_c = (uint32_t)(I / kMT);
  const int64_t r0 = (int64_t)(blockIdx.x / tiles_c) * 32;
  const int64_t c0 = (int64_t)(blockIdx.x % tiles_c) * kMT + 64 * (wid & 1);
  const int64_t rw = r0 + (lane >> 3);
  const uint16_t* dp = dH + rw * I + c0 + 8 * (lane & 7);
  const uint16_t* gp = GU + rw * 2 * I + c0 + 8 * (lane & 7);
  uint4 v[4];
  if (half == 0)
    geglu_bwd_wave_rows<true>(dp, gp, I, p.rows - rw, ta, tf, v);
  else
    geglu_bwd_wave_rows<false>(dp, gp, I, p.rows - rw, ta, tf, v);
  mx_wave_finish<FMT>(p, r0, half * I + c0, v, stage[wid], lane);
}

// Up to kMxMany tensors in one launch: tensor t owns blocks [first, next tensor's first), so
// that a forward's small tensors fill the chip together and save launches. A single tensor runs
// mx_rows_kernel: finding a tensor in the list is a chain of loads of the arguments, 1.1 us of the
// 3.3 us that 32 x 2560 took in a list of one (2.2 us without).
constexpr int kMxMany = 8;

struct MxManyArgs {
  MxTile t[kMxMany];
  int64_t first[kMxMany + 1];
  int count;
};

template <int LR>
__global__ __launch_bounds__(kMxNT) void mx_rows_many_kernel(MxManyArgs a) {
  int i = 0;
  for (int k = 1; k < a.count; ++k)
    if ((int64_t)blockIdx.x >= a.first[k]) i = k;
  const int64_t blk = (int64_t)blockIdx.x - a.first[i], nblk = a.first[i + 1] - a.first[i];
  if (a.t[i].fmt == BF8_E4M3)
    mx_rows<BF8_E4M3, LR>(a.t[i], blk, nblk);
  else
    mx_rows<BF8_E5M2, LR>(a.t[i], blk, nblk);
}

// Blocks of the rowwise kernel: four waves take a tile of 4 lr rows x 128 columns each.
int64_t mx_row_blocks(const MxTile& t, int lr) {
  const int64_t tiles = (t.rows + 4 * lr - 1) / (4 * lr) * ((t.cols + kMT - 1) / kMT);
  return std::min<int64_t>((tiles + 3) / 4, kMaxMxRowBlocks);
}

// Elements up to which a tensor takes the small kernels. Large / small kernel, us, input not seen
// before (repeated): rowwise 2.5M 5.1 / 4.1 (3.6 / 3.1), 5.6M 6.5 / 6.3 (4.8 / 4.9), 8.1M 7.9 / 7.8
// (6.1 / 6.3), 10.4M 9.0 / 9.2; both copies 0.9M 7.8 / 5.0, 4.4M 10.8 / 8.5 (9.3 / 7.2), 8.1M 14.1 /
// 11.2, 10.0M 14.5 / 13.7, 11.1M 15.2 / 16.3 (14.0 / 12.6), 30M 30.6 / 38.5 (29.2 / 26.6).
constexpr int64_t kMxSmallRows = 6 << 20, kMxSmallTile = 8 << 20;
// The same for the fused gated-GELU backward's dGU, us on gradients not seen before: both copies
// 0.2M 15.0 / 7.4, 2.5M 16.0 / 9.8, 5.6M 17.5 / 13.3, 6.6M 18.1 / 19.1; rowwise alone 2.5M 13.1 /
// 7.4, 8.8M 19.0 / 14.2, 12.8M 19.9 / 19.4.
constexpr int64_t kBwdSmallRows = 12 << 20, kBwdSmall = 6 << 20;

template <int FMT>
int mx_launch_one(const MxTile& t, hipStream_t s) {
  const int64_t n = t.rows * t.cols;
  if (!t.out_t) {
    if (n <= kMxSmallRows)
      hipLaunchKernelGGL((mx_rows_kernel<FMT, 1>), dim3((unsigned)mx_row_blocks(t, 1)), dim3(kMxNT),
                         0, s, t);
    else
      hipLaunchKernelGGL((mx_rows_kernel<FMT, kLR>), dim3((unsigned)mx_row_blocks(t, kLR)),
                         dim3(kMxNT), 0, s, t);
    return launch_status("mx_rows_kernel");
  }
  if (n <= kMxSmallTile) {
    hipLaunchKernelGGL(mx_wave_kernel<FMT>, dim3((unsigned)(t.rows / 32 * ((t.cols + 63) / 64))),
                       dim3(64), 0, s, t);
    return launch_status("mx_wave_kernel");
  }
  const int64_t tiles = (t.rows + kMT - 1) / kMT * ((t.cols + kMT - 1) / kMT);
  hipLaunchKernelGGL(mx_tile_kernel<FMT>,
                     dim3((unsigned)std::min<int64_t>(tiles, kMaxMxTileBlocks)), dim3(kMxNT), 0, s,
                     t);
  return launch_status("mx_tile_kernel");
}

int mx_launch(const MxTile& t, void* stream) {
  return t.fmt == BF8_E4M3 ? mx_launch_one<BF8_E4M3>(t, as_stream(stream))
                           : mx_launch_one<BF8_E5M2>(t, as_stream(stream));
}

}  // namespace
}  // namespace bf8

using namespace bf8;

extern "C" {

static int quantize_mx_entry(const char* who, const void* x, int64_t rows, int64_t cols, int fmt,
                             uint8_t* out, uint8_t* out_scales, uint32_t* out_planes,
                             uint8_t* out_t, uint8_t* out_t_scales, uint32_t* out_t_planes,
                             void* stream) {
  BF8_CHECK(fmt == BF8_E4M3 || fmt == BF8_E5M2, "%s: bad fmt %d", who, fmt);
  BF8_CHECK(rows >= 0 && cols >= 0, "%s: negative shape", who);
  BF8_CHECK((out == nullptr) == (!out_scales && !out_planes) &&
                (out_t == nullptr) == (!out_t_scales && !out_t_planes) && (out || out_t),
            "%s: give out and / or out_t, each with its scale rows or planes", who);
  BF8_CHECK(!out || cols % 32 == 0, "%s: rowwise blocks need cols %% 32 == 0 (got %lld)", who,
            (long long)cols);
  BF8_CHECK(!out_t || (rows % 32 == 0 && cols % 16 == 0),
            "%s: columnwise blocks need rows %% 32 == 0 and cols %% 16 == 0 (got %lld x %lld)", who,
            (long long)rows, (long long)cols);
  if (rows == 0 || cols == 0) return BF8_OK;
  BF8_CHECK(x != nullptr, "%s: x is NULL", who);
  BF8_CHECK(((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 7) == 0 && ((uintptr_t)out_t & 15) == 0 &&
                (((uintptr_t)out_scales | (uintptr_t)out_planes | (uintptr_t)out_t_planes) & 3) == 0,
            "%s: x, out_t 16-byte, out 8-byte, out_scales and scale planes 4-byte aligned", who);
  return mx_launch(MxTile{(const uint16_t*)x, rows, cols, out, out_scales, out_planes,
                          out ? bf8_mx_scale_ld(cols) : 0, out_t, out_t_scales, out_t_planes,
                          bf8_mx_scale_ld(rows), fmt},
                   stream);
}

int bf8_quantize_mx_planes_bf16(const void* x, int64_t rows, int64_t cols, int fmt, uint8_t* out,
                                uint8_t* out_scales, uint32_t* out_planes, uint8_t* out_t,
                                uint8_t* out_t_scales, uint32_t* out_t_planes, void* stream) {
  return quantize_mx_entry("bf8_quantize_mx_planes_bf16", x, rows, cols, fmt, out, out_scales,
                           out_planes, out_t, out_t_scales, out_t_planes, stream);
}

int bf8_geglu_bwd_mx_planes(const void* dH, const void* GU, int64_t M, int64_t I, int fmt,
                            uint8_t* out, uint32_t* out_planes, uint8_t* out_t,
                            uint32_t* out_t_planes, void* stream) {
  const char* who = "bf8_geglu_bwd_mx_planes";
  BF8_CHECK(fmt == BF8_E4M3 || fmt == BF8_E5M2, "%s: bad fmt %d", who, fmt);
  BF8_CHECK(M >= 0 && I >= 0 && I % kMT == 0, "%s: need I %% 128 == 0 (M=%lld, I=%lld)", who,
            (long long)M, (long long)I);
  BF8_CHECK((out == nullptr) == (out_planes == nullptr) &&
                (out_t == nullptr) == (out_t_planes == nullptr) && (out || out_t),
            "%s: give out with out_planes and/or out_t with out_t_planes", who);
  BF8_CHECK(!out_t || M % 32 == 0, "%s: columnwise blocks need M %% 32 == 0 (got %lld)", who,
            (long long)M);
  if (M == 0 || I == 0) return BF8_OK;
  BF8_CHECK(dH && GU, "%s: NULL pointer", who);
  BF8_CHECK((((uintptr_t)dH | (uintptr_t)GU | (uintptr_t)out_t) & 15) == 0 &&
                ((uintptr_t)out & 7) == 0 &&
                (((uintptr_t)out_planes | (uintptr_t)out_t_planes) & 3) == 0,
            "%s: dH, GU, out_t 16-byte, out 8-byte, planes 4-byte aligned", who);
  const MxTile p{nullptr, M, 2 * I, out, nullptr, out_planes, 0, out_t, nullptr, out_t_planes, 0,
                 fmt};
  const auto* d = (const uint16_t*)dH;
  const auto* g = (const uint16_t*)GU;
  hipStream_t s = as_stream(stream);
  if (2 * M * I <= (out_t ? kBwdSmall : kBwdSmallRows)) {
    const dim3 grid((unsigned)((M + 31) / 32 * (I / kMT)));
    if (fmt == BF8_E4M3)
      hipLaunchKernelGGL(geglu_bwd_mx_wave_kernel<BF8_E4M3>, grid, dim3(kMxNT), 0, s, d, g, I, p);
    else
      hipLaunchKernelGGL(geglu_bwd_mx_wave_kernel<BF8_E5M2>, grid, dim3(kMxNT), 0, s, d, g, I, p);
    return launch_status("geglu_bwd_mx_wave_kernel");
  }
  const int64_t tiles = ((M + kMT - 1) / kMT) * (I / kMT);
  const dim3 grid((unsigned)std::min<int64_t>(tiles, kMaxBwdBlocks));
  if (fmt == BF8_E4M3)
    hipLaunchKernelGGL(geglu_bwd_mx_kernel<BF8_E4M3>, grid, dim3(kBwdNT), 0, s, d, g, I, p);
  else
    hipLaunchKernelGGL(geglu_bwd_mx_kernel<BF8_E5M2>, grid, dim3(kBwdNT), 0, s, d, g, I, p);
  return launch_status("geglu_bwd_mx_kernel");
}

int bf8_quantize_mx_bf16(const void* x, int64_t rows, int64_t cols, int fmt, uint8_t* out,
                         uint8_t* out_scales, uint8_t* out_t, uint8_t* out_t_scales,
                         void* stream) {
  return quantize_mx_entry("bf8_quantize_mx_bf16", x, rows, cols, fmt, out, out_scales, nullptr,
                           out_t, out_t_scales, nullptr, stream);
}

static int quantize_mx_many_entry(const char* who, int count, const void* const* x,
                                  const int64_t* rows, const int64_t* cols, const int* fmt,
                                  uint8_t* const* out, uint8_t* const* out_scales,
                                  uint32_t* const* out_planes, void* stream) {
  BF8_CHECK(count >= 1 && count <= kMxMany, "%s: count %d outside [1, %d]", who, count, kMxMany);
  BF8_CHECK(x && rows && cols && fmt && out && out_scales, "%s: NULL array", who);
  MxManyArgs a{};
  int64_t n = 0;
  for (int t = 0; t < count; ++t) {
    BF8_CHECK(fmt[t] == BF8_E4M3 || fmt[t] == BF8_E5M2, "%s: tensor %d: bad fmt %d", who, t, fmt[t]);
    BF8_CHECK(rows[t] >= 0 && cols[t] >= 0, "%s: tensor %d: negative shape", who, t);
    BF8_CHECK(cols[t] % 32 == 0,
              "%s: tensor %d: rowwise blocks need cols %% 32 == 0 (got %lld)", who, t,
              (long long)cols[t]);
    if (rows[t] == 0 || cols[t] == 0) continue;
    uint32_t* planes = out_planes ? out_planes[t] : nullptr;
    BF8_CHECK(x[t] && out[t] && (out_scales[t] || planes),
              "%s: tensor %d: x, out or the scales (rows and planes alike) is NULL", who, t);
    BF8_CHECK(((uintptr_t)x[t] & 15) == 0 && ((uintptr_t)out[t] & 7) == 0 &&
                  (((uintptr_t)out_scales[t] | (uintptr_t)planes) & 3) == 0,
              "%s: tensor %d: x 16-byte, out 8-byte, out_scales and scale planes 4-byte aligned", who, t);
    a.t[a.count++] = MxTile{(const uint16_t*)x[t], rows[t], cols[t], out[t], out_scales[t], planes,
                            bf8_mx_scale_ld(cols[t]), nullptr, nullptr, nullptr, 0, fmt[t]};
    n += rows[t] * cols[t];
  }
  if (a.count == 0) return BF8_OK;
  if (a.count == 1) return mx_launch(a.t[0], stream);
  const int lr = n <= kMxSmallRows ? 1 : kLR;
  for (int t = 0; t < a.count; ++t) a.first[t + 1] = a.first[t] + mx_row_blocks(a.t[t], lr);
  const dim3 grid((unsigned)a.first[a.count]);
  if (lr == 1)
    hipLaunchKernelGGL(mx_rows_many_kernel<1>, grid, dim3(kMxNT), 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL(mx_rows_many_kernel<kLR>, grid, dim3(kMxNT), 0, as_stream(stream), a);
  return launch_status("mx_rows_many_kernel");
}

int bf8_quantize_mx_many_planes_bf16(int count, const void* const* x, const int64_t* rows,
                                     const int64_t* cols, const int* fmt, uint8_t* const* out,
                                     uint8_t* const* out_scales, uint32_t* const* out_planes,
                                     void* stream) {
  return quantize_mx_many_entry("bf8_quantize_mx_many_planes_bf16", count, x, rows, cols, fmt, out,
                                out_scales, out_planes, stream);
}

int bf8_quantize_mx_many_bf16(int count, const void* const* x, const int64_t* rows,
                              const int64_t* cols, const int* fmt, uint8_t* const* out,
                              uint8_t* const* out_scales, void* stream) {
  return quantize_mx_many_entry("bf8_quantize_mx_many_bf16", count, x, rows, cols, fmt, out,
                                out_scales, nullptr, stream);
}

}  // extern "C"
