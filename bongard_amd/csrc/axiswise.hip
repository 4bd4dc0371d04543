// Axiswise (per-row / per-column) FP8 quantization for gfx950: torchao's AXISWISE scaling
// granularity, used by its `rowwise` and `rowwise_with_gw_hp` recipes.
//
// Replaces torchao hp_tensor_to_float8_dynamic(..., scaling_granularity=AXISWISE,
// axiswise_dim=d, round_scales_to_power_of_2=True) as reached from TrainingLinear.forward
// (bongard/float8_training.py:22, Float8Linear.forward) for recipes named at
// bongard/float8_training.py:9. For a bf16 tensor x [rows, cols]:
//   dim -1 (one scale per row):    amax_r = max_c |x[r, c]|
//   dim 0  (one scale per column): amax_c = max_r |x[r, c]|
//   scale = fp32(fp8_max / max(f64(amax), 1e-12)), rounded down to a power of two when
//   BF8_SCALE_POW2 is set; q = fp8(clamp(f32(x) * scale, +-fp8_max)).
// The per-row quantization is stored as q [rows, cols]; the per-column one is stored
// transposed, q_t [cols, rows] (row c of q_t holds column c of x, the K-contiguous layout
// the GEMM reads), each with its scale_inv vector.
//
// Kernels (bf16 x is read at most twice):
//   axis_row_kernel      one pass over x: per-row amax -> scale -> cast (row output), and
//                        per-block column amax partials (bf16 keys) for the column scales;
//   axis_col_scale_kernel the column partials -> per-column scale and scale_inv;
//   axis_col_cast_kernel  second pass over x: per-column cast, turned in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"

namespace bf8 {
namespace {

constexpr int kAxNT = 512;              // threads of the row kernel (8 waves)
constexpr int kAxMaxCols = 16384;       // widest row the row kernel holds in registers
constexpr int kAxBlocksPartials = 512;  // row-kernel blocks when it writes column partials
constexpr int kAxBlocksPlain = 2048;    // ... when it does not
constexpr int kColNT = 256;
constexpr int kScaleNT = 1024;          // threads of the column-scale kernel
constexpr int kCT = 128;                // column-cast tile (rows x cols)
constexpr int kCPitch = kCT / 4 + 1;    // dwords per staged row (odd)
constexpr int kMaxColCastBlocks = 2048;

// |x| keys of two packed bf16: clearing the sign makes the unsigned order of each half the
// order of |x| (NaN above inf).
__device__ __forceinline__ uint4 abs_keys(uint4 v) {
  return make_uint4(v.x & 0x7FFF7FFFu, v.y & 0x7FFF7FFFu, v.z & 0x7FFF7FFFu, v.w & 0x7FFF7FFFu);
}

// Quantize 8 bf16 values with one scale each. FINITE: no value and no scale is inf or NaN.
template <int FMT, bool FINITE>
__device__ __forceinline__ uint2 quant8_bf16_vs(uint4 v, const float* sc) {
  const float x0 = bf16_lo(v.x), x1 = bf16_hi(v.x), x2 = bf16_lo(v.y), x3 = bf16_hi(v.y);
  const float x4 = bf16_lo(v.z), x5 = bf16_hi(v.z), x6 = bf16_lo(v.w), x7 = bf16_hi(v.w);
  uint2 r;
  if constexpr (FINITE) {
    r.x = quant4_finite<FMT, true>(x0 * sc[0], x1 * sc[1], x2 * sc[2], x3 * sc[3]);
    r.y = quant4_finite<FMT, true>(x4 * sc[4], x5 * sc[5], x6 * sc[6], x7 * sc[7]);
    return r;
  }
  r.x = quant4<FMT>(x0 * sc[0], x1 * sc[1], x2 * sc[2], x3 * sc[3], x0, x1, x2, x3, sc[0]);
  r.y = quant4<FMT>(x4 * sc[4], x5 * sc[5], x6 * sc[6], x7 * sc[7], x4, x5, x6, x7, sc[4]);
  // quant4 takes one scale for the sign of a NaN product; patch lanes whose own scale is
  // the NaN source (a NaN column or row amax) with their own scale's rule.
  const float xs[8] = {x0, x1, x2, x3, x4, x5, x6, x7};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float pr = xs[e] * sc[e];
    if (__builtin_expect(pr != pr, 0)) {
      uint32_t& w = e < 4 ? r.x : r.y;
      const int sh = 8 * (e & 3);
      w = (w & ~(0xFFu << sh)) | (nan_byte(xs[e], sc[e]) << sh);
    }
  }
  return r;
}

// Max of m over the TPR threads of a row group (TPR = 64: one wave; TPR = 256: four waves
// of a kAxNT / 256 group block, through LDS; every thread of the block must call it).
template <int TPR>
__device__ __forceinline__ uint32_t group_max(uint32_t m) {
  m = wave_max_u32(m);
  if constexpr (TPR == 64) {
    return m;
  } else {
    static_assert(TPR == 256, "row groups of 64 or 256 threads");
    __shared__ uint32_t red[kAxNT / 64];
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[w] = m;
    __syncthreads();
    const int base = (w / 4) * 4;
    const uint32_t r = max(max(red[base], red[base + 1]), max(red[base + 2], red[base + 3]));
    __syncthreads();
    return r;
  }
}

// Rows [blockIdx.x * strip, + strip) of x, one row per TPR-thread group at a time (strip is
// a multiple of the kAxNT / TPR groups, so every group runs the same number of steps).
// Thread tl of a group holds the row's 16-byte vectors tl, tl + TPR, ... (V of them).
// The next row's vectors are loaded before the current row's maximum is known, and V is the
// row's exact number of vectors per thread. Memory-bound: rows alone (2 B read, 1 B written per
// element) [4096, 10240] 25.1 us with V rounded up to 8 and no load ahead, 22.5 so (5.6 TB/s);
// [2560, 10240] 17.2 and 15.7.
// out / row_sinv: per-row quantization (NULL: skipped). colpart: per-block max |x| keys
// of each column (bf16 keys, [gridDim.x][cols]), or NULL.
template <int FMT, int TPR, int V>
__global__ __launch_bounds__(kAxNT) void axis_row_kernel(
    const uint16_t* __restrict__ x, int rows, int cols, int strip, int pow2,
    uint8_t* __restrict__ out, float* __restrict__ row_sinv, uint16_t* __restrict__ colpart) {
  constexpr int G = kAxNT / TPR;
  extern __shared__ uint4 cbuf[];  // [G - 1][cols / 8] column keys of groups 1.. (colpart)
  const int g = threadIdx.x / TPR, tl = threadIdx.x % TPR;
  const int nvec = cols >> 3;
  uint4 ck[V];
#pragma unroll
  for (int j = 0; j < V; ++j) ck[j] = make_uint4(0u, 0u, 0u, 0u);
  const int r0 = blockIdx.x * strip;
  // (the widest rows' registers for a second row cost more waves than the loads ahead save:
  // 141 VGPRs, 3 waves per SIMD; [14912, 4096] 37.7 us with, 34.3 without)
  constexpr bool kAhead = V < 8;
  uint4 next[V];
  auto load = [&](int r) {
    const uint4* xr = reinterpret_cast<const uint4*>(x + (int64_t)r * cols);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int v = tl + TPR * j;
      next[j] = (r < rows && v < nvec) ? xr[v] : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  if (kAhead) load(r0 + g);
  for (int rr = g; rr < strip; rr += G) {
    const int r = r0 + rr;
    const bool valid = r < rows;
    if (!kAhead) load(r);
    uint4 xv[V];
#pragma unroll
    for (int j = 0; j < V; ++j) xv[j] = next[j];
    if (kAhead && rr + G < strip) load(r + G);  // in flight during this row's reduction and cast
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < V; ++j) m = max(m, absmax_key8(xv[j]));
    m = group_max<TPR>(m);
    if (colpart) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const uint4 k = abs_keys(xv[j]);
        ck[j] = make_uint4(pk_max_u16(ck[j].x, k.x), pk_max_u16(ck[j].y, k.y),
                           pk_max_u16(ck[j].z, k.z), pk_max_u16(ck[j].w, k.w));
      }
    }
    if (valid && (out || row_sinv)) {
      float scale, sinv;
      scale_from_amax_key(m, Fp8Max<FMT>::value, pow2 != 0, scale, sinv);
      if (row_sinv && tl == 0) row_sinv[r] = sinv;
      if (out) {
        uint2* orow = reinterpret_cast<uint2*>(out + (int64_t)r * cols);
        if (__builtin_expect(m < 0x7F800000u, 1)) {
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const int v = tl + TPR * j;
            if (v < nvec) orow[v] = quant8_bf16_finite<FMT, true>(xv[j], scale);
          }
        } else {
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const int v = tl + TPR * j;
            if (v < nvec) orow[v] = quant8_bf16<FMT>(xv[j], scale);
          }
        }
      }
    }
  }
  if (!colpart) return;
  uint4* dst = reinterpret_cast<uint4*>(colpart + (int64_t)blockIdx.x * cols);
  if constexpr (G == 1) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int v = tl + TPR * j;
      if (v < nvec) dst[v] = ck[j];
    }
  } else {
    // groups 1.. hand their keys to group 0, whose threads hold the same columns
    if (g > 0) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int v = tl + TPR * j;
        if (v < nvec) cbuf[(g - 1) * nvec + v] = ck[j];
      }
    }
    __syncthreads();
    if (g == 0) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const int v = tl + TPR * j;
        if (v >= nvec) continue;
        uint4 k = ck[j];
#pragma unroll
        for (int gg = 1; gg < G; ++gg) {
          const uint4 o = cbuf[(gg - 1) * nvec + v];
          k = make_uint4(pk_max_u16(k.x, o.x), pk_max_u16(k.y, o.y), pk_max_u16(k.z, o.z),
                         pk_max_u16(k.w, o.w));
        }
        dst[v] = k;
      }
    }
  }
}

// Column scales from the row kernel's partials [nblk][cols]: a block covers 64 columns
// (8 threads x 8 columns) and splits the nblk partial rows over 128 thread rows, so that each
// thread's few loads are in flight together; one thread per column computes its scale.
// Latency-bound: at 512 partial rows of 2560 columns 256 threads, whose last 8 computed 8
// scales each (fp64 divisions) one after the other, took 6.0 us, this 4.9.
template <int FMT>
__global__ __launch_bounds__(kScaleNT) void axis_col_scale_kernel(
    const uint16_t* __restrict__ colpart, int nblk, int cols, int pow2,
    float* __restrict__ col_scale, float* __restrict__ col_sinv) {
  constexpr int kTR = kScaleNT / 8, kW = kScaleNT / 64;
  __shared__ uint4 red[kW][8];
  const int cg = threadIdx.x & 7, rg = threadIdx.x >> 3;
  const int nvec = cols >> 3;
  const int v = blockIdx.x * 8 + cg;
  uint32_t k[4] = {0u, 0u, 0u, 0u};
  if (v < nvec) {
    const uint4* src = reinterpret_cast<const uint4*>(colpart);
#pragma unroll 4
    for (int b = rg; b < nblk; b += kTR) {
      const uint4 o = src[(int64_t)b * nvec + v];
      k[0] = pk_max_u16(k[0], o.x);
      k[1] = pk_max_u16(k[1], o.y);
      k[2] = pk_max_u16(k[2], o.z);
      k[3] = pk_max_u16(k[3], o.w);
    }
  }
  // the 8 thread rows of a wave, then the waves
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) k[i] = pk_max_u16(k[i], (uint32_t)__shfl_xor((int)k[i], off, 64));
  }
  if ((threadIdx.x & 63) < 8) red[threadIdx.x >> 6][cg] = make_uint4(k[0], k[1], k[2], k[3]);
  __syncthreads();
  const int c = blockIdx.x * 64 + threadIdx.x;
  if (threadIdx.x >= 64 || c >= cols) return;
  uint32_t m = 0;
#pragma unroll
  for (int w = 0; w < kW; ++w)
    m = max(m, (uint32_t)reinterpret_cast<const uint16_t*>(red[w])[threadIdx.x]);
  float scale, sinv;
  scale_from_amax_key(m << 16, Fp8Max<FMT>::value, pow2 != 0, scale, sinv);
  col_scale[c] = scale;
  col_sinv[c] = sinv;
}

// q_t [cols, rows] = per-column cast of x. A block takes 128 x 128 tiles, each wave 32 rows of
// all 128 columns: lane l holds columns 8 (l & 15) .. +7 of the rows 4 k + l / 16, k < 8, and
// casts them with its 8 column scales; the bytes meet in LDS and each wave turns 32 columns of
// all 128 rows, so that every store instruction writes whole 128-byte lines.
// Memory-bound: 2 B read (x again, from the MALL where it fits), 1 B written per element. On
// 64 x 64 tiles per wave, whose stores were half lines: [10240, 2560] 20.9 us, now 15.6
// (5.0 TB/s); [4096, 10240] 25.9 and 23.7 us (5.3 TB/s).
template <int FMT>
__global__ __launch_bounds__(kColNT) void axis_col_cast_kernel(
    const uint16_t* __restrict__ x, int64_t rows, int64_t cols,
    const float* __restrict__ col_scale, uint8_t* __restrict__ out_t) {
  __shared__ uint32_t stage[kCT * kCPitch];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int64_t tiles_c = (cols + kCT - 1) / kCT;
  const int64_t ntiles = tiles_c * ((rows + kCT - 1) / kCT);
  const bool t16 = (rows & 15) == 0;
  const int cl = lane & 15, lr = lane >> 4;
  for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int64_t r0 = (t / tiles_c) * kCT, c0 = (t % tiles_c) * kCT;
    const int64_t c = c0 + 8 * cl;
    uint4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t r = r0 + 32 * wid + 4 * k + lr;
      v[k] = make_uint4(0u, 0u, 0u, 0u);
      if (r < rows && c < cols) v[k] = *reinterpret_cast<const uint4*>(x + r * cols + c);
    }
    float sc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (c < cols) {
      const float4 s0 = reinterpret_cast<const float4*>(col_scale + c)[0];
      const float4 s1 = reinterpret_cast<const float4*>(col_scale + c)[1];
      sc[0] = s0.x; sc[1] = s0.y; sc[2] = s0.z; sc[3] = s0.w;
      sc[4] = s1.x; sc[5] = s1.y; sc[6] = s1.z; sc[7] = s1.w;
    }
    // a column of finite values has a finite scale above 0; an inf gives 0, a NaN gives NaN
    bool special = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) special |= c < cols && !(sc[e] > 0.f);
    if (__builtin_expect(__any(special), 0)) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint2 q = quant8_bf16_vs<FMT, false>(v[k], sc);
        uint32_t* d = stage + (32 * wid + 4 * k + lr) * kCPitch + 2 * cl;
        d[0] = q.x;
        d[1] = q.y;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint2 q = quant8_bf16_vs<FMT, true>(v[k], sc);
        uint32_t* d = stage + (32 * wid + 4 * k + lr) * kCPitch + 2 * cl;
        d[0] = q.x;
        d[1] = q.y;
      }
    }
    __syncthreads();
    // lane: 16 rows (lane & 7) x 4 columns (lane >> 3) of the wave's 32 columns
    const int rg = (lane & 7) * 16, cg = 8 * wid + (lane >> 3);
    uint32_t d[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = stage[(rg + i) * kCPitch + cg];
    uint4 tq[4];
    transpose_4x16(d, tq);
    const int64_t tc = r0 + rg;  // column of out_t (a row of x)
    if (tc < rows) {
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        const int64_t tr = c0 + 4 * cg + cc;  // row of out_t (a column of x)
        if (tr >= cols) continue;
        uint8_t* dst = out_t + tr * rows + tc;
        if (t16) {
          *reinterpret_cast<uint4*>(dst) = tq[cc];
        } else {
          const uint32_t w[4] = {tq[cc].x, tq[cc].y, tq[cc].z, tq[cc].w};
          for (int j = 0; j < 16 && tc + j < rows; ++j)
            dst[j] = (uint8_t)(w[j >> 2] >> (8 * (j & 3)));
        }
      }
    }
    __syncthreads();
  }
}

struct AxisPlan {
  int tpr, v, groups, strip, blocks;
  size_t part_bytes;  // column partials, 256-byte aligned
};

AxisPlan axis_plan(int64_t rows, int64_t cols, bool colwise) {
  AxisPlan p{};
  const int64_t nvec = cols / 8;
  p.tpr = cols <= 4096 ? 64 : 256;
  const int64_t per = (nvec + p.tpr - 1) / p.tpr;
  p.v = (int)per;  // <= 8: cols <= kAxMaxCols
  p.groups = kAxNT / p.tpr;
  const int64_t cap = colwise ? kAxBlocksPartials : kAxBlocksPlain;
  int64_t strip = (rows + cap - 1) / cap;
  strip = (strip + p.groups - 1) / p.groups * p.groups;
  if (strip < p.groups) strip = p.groups;
  p.strip = (int)strip;
  p.blocks = (int)std::max<int64_t>(1, (rows + strip - 1) / strip);
  p.part_bytes = colwise ? ((size_t)p.blocks * (size_t)cols * 2 + 255) / 256 * 256 : 0;
  return p;
}

template <int FMT, int TPR>
void launch_row(const AxisPlan& p, const uint16_t* x, int rows, int cols, int pow2, uint8_t* out,
                float* row_sinv, uint16_t* colpart, hipStream_t s) {
  const size_t lds = (colpart && p.groups > 1) ? (size_t)(p.groups - 1) * cols * 2 : 0;
  const dim3 grid((unsigned)p.blocks), block(kAxNT);
#define BF8_AXIS_ROW(VV)                                                                      \
  hipLaunchKernelGGL((axis_row_kernel<FMT, TPR, VV>), grid, block, lds, s, x, rows, cols,    \
                     p.strip, pow2, out, row_sinv, colpart)
  switch (p.v) {
    case 1: BF8_AXIS_ROW(1); break;
    case 2: BF8_AXIS_ROW(2); break;
    case 3: BF8_AXIS_ROW(3); break;
    case 4: BF8_AXIS_ROW(4); break;
    case 5: BF8_AXIS_ROW(5); break;
    case 6: BF8_AXIS_ROW(6); break;
    case 7: BF8_AXIS_ROW(7); break;
    default: BF8_AXIS_ROW(8); break;
  }
#undef BF8_AXIS_ROW
}

template <int FMT>
int run_axiswise(const uint16_t* x, int rows, int cols, int pow2, uint8_t* out, float* row_sinv,
                 uint8_t* out_t, float* col_sinv, uint8_t* ws, hipStream_t s) {
  const bool colwise = out_t != nullptr;
  const AxisPlan p = axis_plan(rows, cols, colwise);
  uint16_t* colpart = colwise ? reinterpret_cast<uint16_t*>(ws) : nullptr;
  if (p.tpr == 64)
    launch_row<FMT, 64>(p, x, rows, cols, pow2, out, row_sinv, colpart, s);
  else
    launch_row<FMT, 256>(p, x, rows, cols, pow2, out, row_sinv, colpart, s);
  int rc = launch_status("axis_row_kernel");
  if (rc != BF8_OK || !colwise) return rc;
  float* col_scale = reinterpret_cast<float*>(ws + p.part_bytes);
  hipLaunchKernelGGL(axis_col_scale_kernel<FMT>, dim3((unsigned)((cols / 8 + 7) / 8)),
                     dim3(kScaleNT), 0, s, colpart, p.blocks, cols, pow2, col_scale, col_sinv);
  rc = launch_status("axis_col_scale_kernel");
  if (rc != BF8_OK) return rc;
  const int64_t tiles = ((int64_t)(rows + kCT - 1) / kCT) * ((cols + kCT - 1) / kCT);
  const unsigned grid = (unsigned)std::min<int64_t>(tiles, kMaxColCastBlocks);
  hipLaunchKernelGGL(axis_col_cast_kernel<FMT>, dim3(grid), dim3(kColNT), 0, s, x,
                     (int64_t)rows, (int64_t)cols, col_scale, out_t);
  return launch_status("axis_col_cast_kernel");
}

}  // namespace
}  // namespace bf8

using namespace bf8;

extern "C" {

size_t bf8_axiswise_workspace(int64_t rows, int64_t cols) {
  if (rows <= 0 || cols <= 0) return 0;
  const AxisPlan p = axis_plan(rows, cols, true);
  return p.part_bytes + (size_t)cols * 4;
}

int bf8_quantize_axiswise_bf16(const void* x, int64_t rows, int64_t cols, int fmt, uint8_t* out,
                               float* row_scale_inv, uint8_t* out_t, float* col_scale_inv,
                               void* ws, size_t ws_bytes, void* stream) {
  const int pow2 = (fmt & BF8_SCALE_POW2) ? 1 : 0;
  fmt &= ~BF8_SCALE_POW2;
  BF8_CHECK(fmt == BF8_E4M3 || fmt == BF8_E5M2, "bf8_quantize_axiswise_bf16: bad fmt %d", fmt);
  BF8_CHECK(rows >= 0 && cols >= 0 && rows < (1LL << 31),
            "bf8_quantize_axiswise_bf16: bad shape");
  BF8_CHECK(cols % 16 == 0 && cols <= kAxMaxCols,
            "bf8_quantize_axiswise_bf16: need cols %% 16 == 0 and cols <= %d (got %lld)",
            kAxMaxCols, (long long)cols);
  BF8_CHECK((out == nullptr) == (row_scale_inv == nullptr) &&
                (out_t == nullptr) == (col_scale_inv == nullptr) && (out || out_t),
            "bf8_quantize_axiswise_bf16: give out with row_scale_inv and/or out_t with "
            "col_scale_inv");
  if (rows == 0 || cols == 0) return BF8_OK;
  BF8_CHECK(x != nullptr, "bf8_quantize_axiswise_bf16: x is NULL");
  BF8_CHECK(((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)out_t & 15) == 0,
            "bf8_quantize_axiswise_bf16: x, out, out_t must be 16-byte aligned");
  if (out_t) {
    const size_t need = bf8_axiswise_workspace(rows, cols);
    BF8_CHECK(ws && ws_bytes >= need && ((uintptr_t)ws & 255) == 0,
              "bf8_quantize_axiswise_bf16: workspace needs %zu bytes, 256-byte aligned (got %zu)",
              need, ws_bytes);
    BF8_CHECK(((uintptr_t)col_scale_inv & 15) == 0,
              "bf8_quantize_axiswise_bf16: col_scale_inv must be 16-byte aligned");
  }
  const uint16_t* xs = (const uint16_t*)x;
  hipStream_t s = as_stream(stream);
  if (fmt == BF8_E4M3)
    return run_axiswise<BF8_E4M3>(xs, (int)rows, (int)cols, pow2, out, row_scale_inv, out_t,
                                  col_scale_inv, (uint8_t*)ws, s);
  return run_axiswise<BF8_E5M2>(xs, (int)rows, (int)cols, pow2, out, row_scale_inv, out_t,
                                col_scale_inv, (uint8_t*)ws, s);
}

}  // extern "C"
