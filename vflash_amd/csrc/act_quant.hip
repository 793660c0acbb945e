// GELU-tanh of the FFN hidden rows fused with their per-token E4M3
// quantization, for gfx950.
//
// Replaces the activation between the FFN's two linears and the second
// linear's own activation quantization (the GELU-tanh form of
// src/vflash/native/h3_native_denoiser.py:369-382; quantization
// src/vflash/native/h3_fp8_activation.py:12-28):
//   g     = bf16(gelu_tanh(y))                    (per element)
//   amax  = max_k |g[row, k]|, NaN if any g is NaN
//   scale = amax > 0 ? max(amax / 448, FLT_MIN) : 1
//   code  = E4M3(clamp(g / scale, -448, 448))
//
// The input y is the bf16 output of the up projection, so GELU is a function of
// 16 bits: kGeluTanhTable (generated at build time, activation_tables.h) holds
// its value for every bf16 pattern, the real function rounded to binary32 and
// then to bf16.  Each workgroup copies the 128 KB table into LDS once (all of its
// DMA and the first rows' loads in flight together) and looks every element up
// with one LDS read; the kernel's work is then HBM-bound.
//
// Layout: one workgroup per CU (the table takes 128 KB of the 160 KB LDS), 12
// waves (three per SIMD), one row per WPR waves at a time with the whole row in
// VGPRs (one HBM read per element); rows are dealt round-robin to the waves of
// the grid.  Row loads and stores go through buffer resources spanning exactly
// the row, so no lane needs a bounds branch and the loads issue back to back.
#include "_gen/activation_tables.h"
#include "quant_ops.h"

#include <type_traits>

namespace vfa {

constexpr int GQ_WAVES = 12;
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// Byte offset of vector i (lanes 64 apart) of `bytes` bytes for this lane, as a
// lane base per group of 4096 bytes plus a constant below 4096 that the buffer
// instruction's immediate field carries (and its range check covers).
// The group base is made opaque so that the compiler cannot merge the two
// constants into one offset register per vector.
// sub: vectors of 64 further lanes that the whole run is moved by.
__device__ __forceinline__ uint32_t vec_off(int lane, int i, int bytes, int sub = 0) {
  const int per_group = 4096 / (64 * bytes);
  uint32_t base = (uint32_t)(lane + 64 * sub) * bytes + (uint32_t)(i / per_group) * 4096u;
  asm volatile("" : "+v"(base));
  return base + (uint32_t)(i % per_group) * 64u * bytes;
}

// y: bf16 [m, k] (row stride ldy); g (optional): bf16 [m, k] (row stride ldg);
// codes: [m_pad, k]; scales: [m_pad].  k % 8 == 0, k <= 512 * VPL * WPR.
template <int VPL, int WPR>
__global__ void __launch_bounds__(64 * GQ_WAVES) gelu_quant_rows(
    const uint16_t* __restrict__ y, int64_t m, int64_t k, int64_t ldy, uint16_t* __restrict__ g,
    int64_t ldg, uint8_t* __restrict__ codes, float* __restrict__ scales, int64_t m_pad) {
  __shared__ __attribute__((aligned(1024))) uint16_t table[65536];
  const int lane = threadIdx.x & 63;
  // The wave index as a scalar: rows, and the buffer resources built from them,
  // are then wave-uniform in the compiler's analysis.
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  {
    // 128 blocks of 1 KB, all in flight at once and beside the first row's loads.
    const __amdgpu_buffer_rsrc_t rt = make_rsrc(kGeluTanhTable, (uint32_t)sizeof(table));
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_addr(table));
    for (int b = wave; b < 128; b += GQ_WAVES)
      lds_dma16(rt, dst + (uint32_t)b * 1024u, (uint32_t)b * 1024u + (uint32_t)lane * 16u);
  }
  // Wave `sub` of the WPR that share a row holds its vectors lane + 64 (WPR i + sub).
  constexpr int ROWS = GQ_WAVES / WPR;  // rows of a workgroup at a time
  const int sub = wave % WPR;
  const int64_t stride = (int64_t)gridDim.x * ROWS;
  // Branch-free row access: buffer resources over exactly this row, so lanes
  // past the end read zeros (T[0] = 0 leaves the maximum alone) and their
  // stores are dropped, and the loads issue back to back.
  auto row_rsrc = [&](int64_t row) {
    return make_rsrc(y + (row < m ? row * ldy : 0), row < m ? (uint32_t)(k * 2) : 0u);
  };
  auto voff = [&](int i, int bytes) { return vec_off(lane, i * WPR, bytes, sub); };
  v4i v[VPL];
  auto load_row = [&](int64_t row) {
    const __amdgpu_buffer_rsrc_t ry = row_rsrc(row);
#pragma unroll
    for (int i = 0; i < VPL; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(ry, voff(i, 16), 0, 0);
  };
  // Every wave of the workgroup makes the same number of rounds (they meet at
  // the barrier below); a wave past the last row works on zeros.
  int64_t row = (int64_t)blockIdx.x * ROWS + wave / WPR;
  const int64_t first = (int64_t)blockIdx.x * ROWS;
  const int rounds = first < m_pad ? (int)((m_pad - first + stride - 1) / stride) : 0;
  load_row(row);
  wait_vmcnt<0, true>();  // this wave's share of the table (and its first row)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  for (int round = 0; round < rounds; ++round, row += stride, load_row(row)) {
    if (WPR == 1 && row >= m) {
      if (row < m_pad) pad_row(codes, scales, row, k, lane);
      continue;
    }
    const __amdgpu_buffer_rsrc_t ry = row_rsrc(row);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t yw = (uint32_t)v[i][w];
        uint32_t gw = (uint32_t)table[yw & 0xffffu] | ((uint32_t)table[yw >> 16] << 16);
        // Only the packed pair stays live: left visible, the compiler keeps the
        // two looked-up halves apart for the later unpacking and runs out of
        // registers.
        asm volatile("" : "+v"(gw));
        v[i][w] = (int)gw;
      }
      amax = nan_max(amax, absmax8(v[i]));
      // At most two vectors' lookups (16 LDS reads) in flight: the compiler
      // would otherwise issue every lookup of the row first, holding one
      // register per half-word.
      if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    if (g && row < m) {
      const __amdgpu_buffer_rsrc_t rg = make_rsrc(g + row * ldg, (uint32_t)(k * 2));
#pragma unroll
      for (int i = 0; i < VPL; ++i)
        __builtin_amdgcn_raw_buffer_store_b128(v[i], rg, voff(i, 16), 0, 0);
    }
    amax = wave_nan_max(amax);
    if constexpr (WPR > 1) {
      // Two sets of maxima in turn: a wave reads one while the next round's are written.
      __shared__ float part[2][GQ_WAVES];
      if (lane == 0) part[round & 1][wave] = amax;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < WPR; ++w) amax = nan_max(amax, part[round & 1][wave - sub + w]);
      if (row >= m) {
        if (row < m_pad && sub == 0) pad_row(codes, scales, row, k, lane);
        continue;
      }
    }
    const float scale = row_scale(amax);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(codes + row * k, (uint32_t)k);
    const RowDivisor d = row_divisor(scale, amax);
    if (d.fast) {
#pragma unroll
      for (int i = 0; i < VPL; ++i) {
        const uint2 c = quant8<true>(v[i], d);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, c), rc, voff(i, 8), 0, 0);
        if (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // bounded live temporaries
      }
    } else {
      // Rows with a NaN or infinite activation (or a scale out of the fast
      // range): the exact path, one vector at a time from a second read of y.
#pragma unroll 1
      for (int i = 0; i < VPL; ++i) {
        v4i yv = __builtin_amdgcn_raw_buffer_load_b128(ry, voff(i, 16), 0, 0);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t yw = (uint32_t)yv[w];
          yv[w] = (int)((uint32_t)table[yw & 0xffffu] | ((uint32_t)table[yw >> 16] << 16));
        }
        const uint2 c = quant8<false>(yv, d);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, c), rc, voff(i, 8), 0, 0);
      }
    }
    if (lane == 0 && sub == 0) scales[row] = scale;
  }
}

int compute_units();

template <int VPL, int WPR>
static void launch_gq(dim3 grid, hipStream_t s, const uint16_t* y, int64_t m, int64_t k,
                      int64_t ldy, uint16_t* g, int64_t ldg, uint8_t* codes, float* scales,
                      int64_t m_pad) {
  gelu_quant_rows<VPL, WPR><<<grid, dim3(64 * GQ_WAVES), 0, s>>>(y, m, k, ldy, g, ldg, codes, scales,
                                                            m_pad);
}

// Requires k % 8 == 0, 8 <= k <= 16384, ldy and ldg multiples of 8, y and g
// 16-byte aligned, codes 8-byte aligned (checked by the caller).
hipError_t launch_gelu_quant_rows(const uint16_t* y, int64_t m, int64_t k, int64_t ldy,
                                  uint16_t* g, int64_t ldg, uint8_t* codes, float* scales,
                                  int64_t m_pad, hipStream_t s) {
  const int64_t cus = compute_units(), nvec = k / 8;
  // Waves per row.  A wave takes its row's lookups and conversions one after the
  // other, so the time is the rounds of rows a wave makes times its share of a
  // row: four waves while one round of them holds every row, two where their
  // rounds come to at most 0.8 of the rounds of whole rows, and on long calls of
  // wide rows.  Microseconds with 1, 2 and 4 waves: 17 x 13824 20.2, 15.9, 12.8;
  // 768 x 5376 13.3, 9.0, 7.3; 1024 x 13824 23.1, 15.7, 16.2; 4095 x 13824 47.4,
  // 41.8, 43.6; 5000 x 13824 46.6, 52.5, 51.6; 16384 x 5120 60.1, 62.9, 72.3;
  // 32760 x 13824 289.9, 260.9, 263.8.
  const int64_t waves = cus * GQ_WAVES;
  const int64_t one = (m_pad + waves - 1) / waves, two = (2 * m_pad + waves - 1) / waves;
  const int wpr = 4 * m_pad <= waves ? 4 : 5 * two <= 8 * one || (one >= 4 && nvec > 1024) ? 2 : 1;
  const int64_t groups = (m_pad + GQ_WAVES / wpr - 1) / (GQ_WAVES / wpr);
  const dim3 grid((unsigned)(groups < cus ? groups : cus));
  auto launch = [&](auto vpl, auto w) {
    launch_gq<vpl, w>(grid, s, y, m, k, ldy, g, ldg, codes, scales, m_pad);
  };
  auto pick = [&](auto w, int64_t nv) {
    if (nv <= 64) launch(std::integral_constant<int, 1>{}, w);
    else if (nv <= 128) launch(std::integral_constant<int, 2>{}, w);
    else if (nv <= 256) launch(std::integral_constant<int, 4>{}, w);
    else if (nv <= 512) launch(std::integral_constant<int, 8>{}, w);
    else if constexpr (w < 4) {
      if (w == 2 && nv <= 896) launch(std::integral_constant<int, 14>{}, w);
      else if (nv <= 1024) launch(std::integral_constant<int, 16>{}, w);
      else if constexpr (w < 2) {
        if (nv <= 1536) launch(std::integral_constant<int, 24>{}, w);
        else if (nv <= 1792) launch(std::integral_constant<int, 28>{}, w);
        else launch(std::integral_constant<int, 32>{}, w);
      }
    }
  };
  // Vectors of a row per wave, rounded up to whole runs of 64.
  if (wpr == 4) pick(std::integral_constant<int, 4>{}, (nvec + 255) / 256 * 64);
  else if (wpr == 2) pick(std::integral_constant<int, 2>{}, (nvec + 127) / 128 * 64);
  else pick(std::integral_constant<int, 1>{}, nvec);
  return hipGetLastError();
}

}  // namespace vfa
