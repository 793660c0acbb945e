// A 256x256 grid of the W8A8 E4M3 GEMM whose last round is split into smaller
// tiles (instantiated per epilogue in fp8_gemm_mixed_bias.hip, fp8_gemm_mixed_gate.hip
// and fp8_gemm_mixed_swiglu.hip; fp8_gemm.hip chooses it, mixed_tail and
// swiglu_main_tiles).  Kernel-side only; not part of the C-ABI.
#pragma once
#include "fp8_gemm_pipe.h"

namespace vfa {

enum { MIXED_NONE = 0, MIXED_256x128 = 1, MIXED_128x128 = 2, MIXED_64x256 = 3 };

// A 256x256 grid whose last round would leave most of the CUs idle: the first
// main_tiles tiles (whole rounds of one tile per CU) run as 256x256, each of the
// remaining ones as 256/SBM x 256/SBN tiles of the SBM x SBN pipeline, which
// follow in the same launch and take the CUs as they come free.  K % 128 == 0.
template <int EPI, int SBM, int SBN, int SNS, int SPRE>
__global__ void __launch_bounds__(256, 1) fp8_gemm_mixed(const GemmParams p, int main_tiles) {
  constexpr int RING = pipe_lds(256, 256, SPLIT_RING), SRING = pipe_lds(SBM, SBN, SNS);
  // SwiGLU tiles are 128 value and 128 gate columns wide, whole or split.
  static_assert(!epi_swiglu(EPI) || SBN == 256, "value and gate columns stay paired");
  static_assert(SRING + VEC_LDS + (epi_swiglu(EPI) ? SILU_LDS : 0) <= RING,
                "the small tile's LDS fits the ring");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[RING];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  const int tiles_m = (int)((p.m + 255) / 256), tiles_n = (int)((p.n + 255) / 256);
  int tm, tn;
  if ((int)blockIdx.x < main_tiles) {
    grouped_tile(xcd_order((int)blockIdx.x, main_tiles), tiles_m, tiles_n, p.group_m, tm, tn);
    uint8_t* vec = ring + (2 * 256 + 2 * 256) * 128;
    pipe_tile<EPI, 256, 256, SPLIT_RING, 0, true>(p, tm, tn, ring, ring_lds, vec,
                                                  __builtin_amdgcn_readfirstlane(lds_addr(vec)), wave);
    return;
  }
  constexpr int PM = 256 / SBM, PN = 256 / SBN;
  const int sub = xcd_order((int)blockIdx.x - main_tiles, (int)gridDim.x - main_tiles);
  grouped_tile(main_tiles + sub / (PM * PN), tiles_m, tiles_n, p.group_m, tm, tn);
  tm = tm * PM + sub % PM;
  tn = tn * PN + sub % (PM * PN) / PM;
  if ((int64_t)tm * SBM >= p.m || (int64_t)tn * SBN >= p.n) return;  // past the edge of the output
  uint8_t* vec = ring + SRING;
  pipe_tile<EPI, SBM, SBN, SNS, SPRE, true>(p, tm, tn, ring, ring_lds, vec,
                                            __builtin_amdgcn_readfirstlane(lds_addr(vec)), wave);
}

template <int EPI, int SBM, int SBN, int SNS, int SPRE>
static hipError_t launch_mixed_as(const GemmParams& p, int64_t main_tiles, hipStream_t s) {
  const int64_t tiles = ((p.m + 255) / 256) * ((p.n + 255) / 256);
  const int64_t grid = main_tiles + (tiles - main_tiles) * (256 / SBM) * (256 / SBN);
  fp8_gemm_mixed<EPI, SBM, SBN, SNS, SPRE><<<dim3((unsigned)grid), dim3(256), 0, s>>>(p, (int)main_tiles);
  return hipGetLastError();
}

// tail: the tiles of the last round (256x128 or 128x128; SwiGLU 64x256).
template <int EPI>
hipError_t launch_mixed(const GemmParams& p, int64_t main_tiles, int tail, hipStream_t s) {
  if constexpr (epi_swiglu(EPI)) return launch_mixed_as<EPI, 64, 256, 3, 0>(p, main_tiles, s);
  else return tail == MIXED_256x128 ? launch_mixed_as<EPI, 256, 128, 3, 0>(p, main_tiles, s)
                               : launch_mixed_as<EPI, 128, 128, 3, -1>(p, main_tiles, s);
}

}  // namespace vfa
