// W8A8 E4M3 GEMM for up to 64 rows on gfx950.
//
// With a few rows the GEMM reads each weight byte once, and its time is the
// chain of K stages of one tile.  In the 64x64 tile every wave issues its share
// of a stage's DMA, reads fragments and multiplies in turn, about 550 cycles a
// stage for two MFMAs of 64 cycles each, on N / 64 workgroups.  Here a workgroup
// owns MB blocks of 32 rows x 32 columns, and the roles are split over waves: MB
// waves read fragments of stage kt + 1 while they multiply stage kt, one wave
// issues the weight rows' DMA and one the activation rows', NS - 1 stages ahead,
// and all meet at one barrier a stage.  The MFMAs, their K order and the epilogue
// are those of fp8_gemm_pipe.h, so the result bits are too.
#pragma once
#include "gemm_epilogue.h"

namespace vfa {

template <int EPI, int MB, int NS>
__global__ void __launch_bounds__(64 * (MB + 2)) fp8_gemm_skinny(const GemmParams p) {
  constexpr int BM = 32 * MB, BN = 32, BK = 128, SLOT = (BM + BN) * BK;
  constexpr int DMA_A = BM / 8, DMA_W = BN / 8;  // 1 KB DMA instructions per stage
  static_assert(NS >= 3 && (NS - 1) * DMA_A < 64 && BM * BN * 2 <= NS * SLOT, "vmcnt range, staging");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * SLOT];
  __shared__ __attribute__((aligned(1024))) uint8_t vec[VEC_LDS];
  int tm, tn;
  tile_coords((int)((p.m + BM - 1) / BM), (int)((p.n + BN - 1) / BN), p.group_m, tm, tn);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  const uint32_t vec_lds = __builtin_amdgcn_readfirstlane(lds_addr(vec));
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int KT = (int)((p.k + BK - 1) / BK);
  auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (wave >= MB) {
    // A DMA wave.  Lane map of pipe_tile: 1 KB block b holds rows 8b .. 8b + 7,
    // lane l fills row 8b + l / 8, slot l % 8, from chunk (l % 8) ^ lds_swizzle(row).
    // Chunks past K, rows past the operand and stages past the end read as zeros.
    const int drow = lane >> 3;
    const int dch0 = (lane & 7) ^ lds_swizzle(drow), dch1 = (lane & 7) ^ lds_swizzle(drow + 8);
    auto produce = [&](const uint8_t* base, int64_t ld, int64_t rows, uint32_t dst, auto count) {
      const __amdgpu_buffer_rsrc_t r = make_rsrc(base, (uint32_t)(rows * ld));
      const uint32_t b0 = (uint32_t)(drow * ld + dch0 * 16), b1 = (uint32_t)((drow + 8) * ld + dch1 * 16);
      const uint32_t step = (uint32_t)(16 * ld);
      auto issue = [&](int j, int s) {
        const int64_t kb = (int64_t)s * BK;
        const uint32_t kill0 = kb + dch0 * 16 < p.k ? 0u : VFA_OOB;
        const uint32_t kill1 = kb + dch1 * 16 < p.k ? 0u : VFA_OOB;
        static_for<count>([&](auto i) {
          const uint32_t off = (i % 2 ? b1 : b0) + (i / 2) * step + (uint32_t)kb;
          lds_dma16(r, dst + (uint32_t)j * SLOT + i * 1024, off | (i % 2 ? kill1 : kill0));
        });
      };
      static_for<NS>([&](auto s) { issue((int)s, (int)s); });
      wait_vmcnt<(NS - 1) * count, true>();  // stage 0 and the vectors, issued before it
      barrier();
      int j = 0;  // slot of stage kt, read by the time of the barrier
      for (int kt = 0; kt < KT; ++kt) {
        wait_vmcnt<(NS - 2) * count, true>();  // stage kt + 1
        barrier();
        issue(j, kt + NS);
        j = j + 1 == NS ? 0 : j + 1;
      }
      wait_vmcnt<0, true>();  // every DMA has landed before the ring becomes the staging tile
      barrier();
    };
    if (wave == MB) {
      static_for<2>([&](auto w) { stage_vectors<BM, BN>(p, m0, n0, 2 * w, lane, vec_lds); });
      produce(p.w + n0 * p.ldw, p.ldw, min((int64_t)BN, p.n - n0), ring_lds + BM * BK,
              std::integral_constant<int, DMA_W>{});
    } else {
      stage_vectors<BM, BN>(p, m0, n0, 1, lane, vec_lds);
      produce(p.a + m0 * p.lda, p.lda, min((int64_t)BM, p.m - m0), ring_lds,
              std::integral_constant<int, DMA_A>{});
    }
    return;  // the barriers left are those of the multiplying waves alone
  }

  const int fr = lane & 31, fh = lane >> 5, fsw = lds_swizzle(fr);
  struct Frags {
    v8i a[2], w[2];  // [K-substep]
  };
  auto read = [&](Frags& q, int j) {
    const uint8_t* src = ring + j * SLOT + fr * BK;
    static_for<2>([&](auto ks) {
      const int cc = ks * 4 + fh * 2;
      const int o0 = (cc ^ fsw) << 4, o1 = ((cc + 1) ^ fsw) << 4;
      auto frag = [&](int row) {
        const v4i lo = *reinterpret_cast<const v4i*>(src + row * BK + o0);
        const v4i hi = *reinterpret_cast<const v4i*>(src + row * BK + o1);
        return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      };
      q.a[ks] = frag(wave * 32);
      q.w[ks] = frag(BM);
    });
  };
  v16f acc[1][1] = {{v16f{}}};
  v16f lora_d[1];
  if constexpr (epi_lora(EPI)) lora_blocks<BM, BN, MB, 1>(p, m0, n0, wave, 0, lane, lora_d);
  barrier();  // stage 0 has landed
  Frags q[2];
  read(q[0], 0);
  int j = 0;
  auto stage = [&](auto par) {
    // Stage kt is in registers (its slot may be refilled), stage kt + 1 has landed.
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    barrier();
    j = j + 1 == NS ? 0 : j + 1;
    read(q[1 - par], j);  // zeros past the last stage, never multiplied
    static_for<2>([&](auto ks) {
      acc[0][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(q[par].w[ks], q[par].a[ks], acc[0][0],
                                                                  0, 0, 0, 0, 0, 0);
    });
  };
  for (int kt = 0; kt < KT; kt += 2) {
    stage(std::integral_constant<int, 0>{});
    if (kt + 1 < KT) stage(std::integral_constant<int, 1>{});
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  barrier();  // every DMA has landed
  gemm_epilogue<BM, BN, MB, 1, EPI, true>(p, acc, m0, n0, wave, 0, (int)threadIdx.x, ring, vec,
                                          epi_lora(EPI) ? lora_d : nullptr);
}

// rows: 32 or 64 per workgroup.
template <int EPI>
hipError_t launch_skinny(const GemmParams& p, int rows, hipStream_t s) {
  const int64_t tiles = (p.m + rows - 1) / rows * ((p.n + 31) / 32);
  if (rows == 32)
    fp8_gemm_skinny<EPI, 1, 8><<<dim3((unsigned)tiles), dim3(192), 0, s>>>(p);
  else
    fp8_gemm_skinny<EPI, 2, 6><<<dim3((unsigned)tiles), dim3(256), 0, s>>>(p);
  return hipGetLastError();
}

}  // namespace vfa
