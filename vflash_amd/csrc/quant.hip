// Per-token (per-row) E4M3 activation quantization for gfx950.
//
// Arithmetic (reference: src/vflash/native/h3_fp8_activation.py:12-28 and its
// portable twin src/vflash/native/h3_fp8_linear.py:18-31):
//   amax  = max_k |x[row, k]|, NaN if any x is NaN  (binary32, torch's amax)
//   scale = amax > 0 ? max(amax / 448, FLT_MIN) : 1 (IEEE division)
//   code  = E4M3(clamp(x / scale, -448, 448))       (IEEE division, RNE)
// Rows in [m, m_pad) are the GEMM padding rows: codes 0, scale 1.
//
// Layout: one 64-lane wave owns one row and a 256-thread workgroup 4 rows, or,
// with few or wide rows, the workgroup's four waves share one row (WPR = 4).
// The aligned kernel keeps the whole row in VGPRs (16-byte loads, one HBM
// read per element), reduces the maximum across the wave with XOR shuffles and
// writes 8 codes per 16-byte input vector.
#include "quant_ops.h"

#include <type_traits>

namespace vfa {

// Aligned path: k % 8 == 0, ldx % 8 == 0, x 16-byte aligned, k <= 512 * VPL * WPR.
template <int VPL, int WPR>
__global__ void __launch_bounds__(256) quant_rows_vec(const uint16_t* __restrict__ x,
                                                      int64_t m, int64_t k, int64_t ldx,
                                                      uint8_t* __restrict__ codes,
                                                      float* __restrict__ scales,
                                                      int64_t m_pad) {
  const int lane = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;  // in the row
  const int64_t row = WPR == 1 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : grid_row();
  if (row >= m_pad) return;
  if (row >= m) {
    if (lane < 64) pad_row(codes, scales, row, k, lane);
    return;
  }
  // Widen the row index before the multiply: row * ldx may exceed 2^31.
  const v4i* xr = reinterpret_cast<const v4i*>(x + row * ldx);
  const int nvec = (int)(k >> 3);
  v4i v[VPL];
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    int j = lane + 64 * WPR * i;
    if (j < nvec) {
      v[i] = __builtin_nontemporal_load(xr + j);
      amax = nan_max(amax, absmax8(v[i]));
    }
  }
  amax = wave_nan_max(amax);
  if constexpr (WPR > 1) {
    __shared__ float part[WPR];
    if ((lane & 63) == 0) part[lane >> 6] = amax;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WPR; ++w) amax = nan_max(amax, part[w]);
  }
  const float scale = row_scale(amax);
  quant_row_regs<VPL, 64 * WPR>(reinterpret_cast<uint2*>(codes + row * k), v, lane, nvec, scale, amax);
  if (lane == 0) scales[row] = scale;
}

// Any k, any row stride: two passes over the row with scalar bf16 loads.
__global__ void __launch_bounds__(256) quant_rows_generic(const uint16_t* __restrict__ x,
                                                          int64_t m, int64_t k, int64_t ldx,
                                                          uint8_t* __restrict__ codes,
                                                          float* __restrict__ scales,
                                                          int64_t m_pad) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= m_pad) return;
  if (row >= m) {
    pad_row(codes, scales, row, k, lane);
    return;
  }
  const uint16_t* xr = x + row * ldx;
  float amax = 0.0f;
  for (int64_t j = lane; j < k; j += 64) amax = nan_max(amax, bf16_to_f32(xr[j] & 0x7fffu));
  amax = wave_nan_max(amax);
  const float scale = row_scale(amax);
  uint8_t* cr = codes + row * k;
  for (int64_t j = lane; j < k; j += 64) cr[j] = (uint8_t)quant1(bf16_to_f32(xr[j]), scale);
  if (lane == 0) scales[row] = scale;
}

// Requantization of a GEMM output whose epilogue already reduced |g| per row
// over each of its `parts` column tiles (amax_part[row * parts + p]).  The
// arithmetic is exactly quant_rows_*: the maximum of the partial maxima is the
// row maximum.  Streaming: no row is held in registers.  gridDim.y splits each
// row's vectors (few rows would leave the GPU idle otherwise); a lane has four
// vectors in flight.
__global__ void __launch_bounds__(256) requant_rows(const uint16_t* __restrict__ g, int64_t m,
                                                    int64_t k, int64_t ldg,
                                                    const float* __restrict__ amax_part,
                                                    int parts, uint8_t* __restrict__ codes,
                                                    float* __restrict__ scales, int64_t m_pad) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= m_pad) return;
  if (row >= m) {
    if (blockIdx.y == 0) pad_row(codes, scales, row, k, lane);
    return;
  }
  float amax = 0.0f;
  for (int p = lane; p < parts; p += 64) amax = nan_max(amax, amax_part[row * parts + p]);
  amax = wave_nan_max(amax);
  const float scale = row_scale(amax);
  const v4i* gr = reinterpret_cast<const v4i*>(g + row * ldg);
  uint2* cr = reinterpret_cast<uint2*>(codes + row * k);
  const int nvec = (int)(k >> 3), segs = (int)gridDim.y, seg = (int)blockIdx.y;
  const int v0 = (int)((int64_t)nvec * seg / segs), v1 = (int)((int64_t)nvec * (seg + 1) / segs);
  const RowDivisor d = row_divisor(scale, amax);
  auto codes_of = [&](auto fast) {
    for (int j = v0 + lane; j < v1; j += 256) {
      v4i in[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j + 64 * i < v1) in[i] = __builtin_nontemporal_load(gr + j + 64 * i);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (j + 64 * i < v1) cr[j + 64 * i] = quant8<fast>(in[i], d);
    }
  };
  if (d.fast)
    codes_of(std::true_type{});
  else
    codes_of(std::false_type{});
  if (seg == 0 && lane == 0) scales[row] = scale;
}

}  // namespace vfa

// ---------------------------------------------------------------------------
// Host launchers (called from capi.hip)
// ---------------------------------------------------------------------------
namespace vfa {

// Segments of a row for the kernels that split rows over gridDim.y: enough for
// about four waves per SIMD, none below 256 vectors of 8 elements (four per lane).
unsigned row_segments(int64_t rows, int64_t k) {
  const int64_t want = 4096 / (rows > 0 ? rows : 1), most = (k / 8 + 255) / 256;
  const int64_t segs = want < most ? want : most;
  return (unsigned)(segs > 1 ? segs : 1);
}

// Rows up to which the four waves of a workgroup share one row at any width.
// Microseconds unshared -> shared: 300 x 5376 9.5 -> 4.8, 2048 x 5120 11.9 -> 9.1,
// 32760 x 5120 90 -> 79, 32760 x 14336 387 -> 262, 4095 x 13824 50 -> 33; narrow rows
// of long calls lose: 4095 x 1536 6.8 -> 7.3, 4096 x 3072 10.1 -> 10.4, 8192 x 2304
// 13.6 -> 15.6, 32760 x 1536 27 -> 38, x 3072 57 -> 57.  Close to either line the
// shared form is still ahead: 2064 x 3072 7.8 -> 6.9, 4096 x 4096 12.6 -> 11.7, 32760 x
// 4096 69 -> 65.
constexpr int64_t QUANT_SHARED_ROWS = 2048;

hipError_t launch_quant_rows(const uint16_t* x, int64_t m, int64_t k, int64_t ldx,
                             uint8_t* codes, float* scales, int64_t m_pad, hipStream_t s) {
  const dim3 block(256), grid((unsigned)((m_pad + 3) / 4));
  const bool aligned = (k % 8 == 0) && (ldx % 8 == 0) &&
                       ((reinterpret_cast<uintptr_t>(x) & 15) == 0) &&
                       ((reinterpret_cast<uintptr_t>(codes) & 7) == 0);
  const int64_t nvec = k / 8;
  if (aligned && nvec <= 64 * 32) {
    // Four waves share a row when rows are few, and always above 4096 columns,
    // where one wave's registers for the whole row leave too few waves in flight.
    if (nvec > 64 && (m_pad <= QUANT_SHARED_ROWS || nvec > 512)) {
      const dim3 rows = row_grid(m_pad);
      if (nvec <= 256) quant_rows_vec<1, 4><<<rows, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
      else if (nvec <= 512) quant_rows_vec<2, 4><<<rows, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
      else if (nvec <= 1024) quant_rows_vec<4, 4><<<rows, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
      else quant_rows_vec<8, 4><<<rows, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
    } else if (nvec <= 64) quant_rows_vec<1, 1><<<grid, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
    else if (nvec <= 128) quant_rows_vec<2, 1><<<grid, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
    else if (nvec <= 256) quant_rows_vec<4, 1><<<grid, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
    else quant_rows_vec<8, 1><<<grid, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
  } else {
    quant_rows_generic<<<grid, block, 0, s>>>(x, m, k, ldx, codes, scales, m_pad);
  }
  return hipGetLastError();
}

hipError_t launch_requant_rows(const uint16_t* g, int64_t m, int64_t k, int64_t ldg,
                               const float* amax_part, int parts, uint8_t* codes,
                               float* scales, int64_t m_pad, hipStream_t s) {
  const dim3 block(256), grid((unsigned)((m_pad + 3) / 4), row_segments(m_pad, k));
  requant_rows<<<grid, block, 0, s>>>(g, m, k, ldg, amax_part, parts, codes, scales, m_pad);
  return hipGetLastError();
}

}  // namespace vfa
