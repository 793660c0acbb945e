// W8A8 E4M3 GEMM with fused epilogues for gfx950 (CDNA4): the choice of tiling
// and the dispatch.  The kernel is the pipelined tile of fp8_gemm_pipe.h.
//
//   acc[m, n] = sum_k A[m, k] * W[n, k]          (E4M3 x E4M3, binary32 accumulate)
//   base      = bf16(bf16(acc * sa[m] * sw[n]) + bias[n])
//
// This replaces torch._scaled_mm(codes, weight.t(), scale_a, scale_b, bf16)
// followed by the separate "+ bias" of RowFP8Execution.linear
// (reference src/vflash/native/h3_fp8_linear.py:109-121); the two bf16
// roundings are kept in that order.  Epilogue variants:
//   EPI_BIAS   out = base                                   (also merged QKV planes)
//   EPI_GATE   out = bf16(residual + bf16(gate * base))
//              (h3_fused_ops.py:124-170 strict_gate_residual_kernel)
//   EPI_LORA   out = bf16(base + delta), delta = bf16(t . B^T) with the optional
//              bf16(delta * scale), bf16(delta * strength) steps
//              (adapters/h3_reference_lora.py:75-90)
//   EPI_SWIGLU h = bf16(value * bf16(silu(gate))) with value = base[:, f] and
//              gate = base[:, half_n + f], plus per-row |h| maxima per 128
//              columns (h3_native_denoiser.py:369-376, h3_fused_ops.py:184-224)
//   EPI_LORA_GATE   EPI_GATE on bf16(base + delta): the adapted gate-residual
//              (h3_native_denoiser.py:327-338, h3_fused_ops.py:341-418)
//   EPI_SWIGLU_LORA EPI_SWIGLU on bf16(base + delta) for value and gate columns
//              alike (h3_fused_ops.py:229-286, strict_ffn_adapter_silu_kernel)
// The LoRA delta may come from up to three adapter branches with their own
// scales, each owning a contiguous run of output columns (the Q/K/V adapters of
// a merged projection, h3_native_denoiser.py:301-316, h3_fused_ops.py:900-980).
#include "fp8_gemm_mixed.h"
#include "fp8_gemm_skinny.h"

namespace vfa {

extern template hipError_t launch_skinny<EPI_BIAS>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_skinny<EPI_GATE>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_skinny<EPI_LORA>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_skinny<EPI_LORA_GATE>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_mixed<EPI_BIAS>(const GemmParams&, int64_t, int, hipStream_t);
extern template hipError_t launch_mixed<EPI_SWIGLU>(const GemmParams&, int64_t, int, hipStream_t);
extern template hipError_t launch_mixed<EPI_GATE>(const GemmParams&, int64_t, int, hipStream_t);
extern template hipError_t launch_tiling<EPI_BIAS>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_tiling<EPI_GATE>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_tiling<EPI_LORA>(const GemmParams&, int, hipStream_t);
extern template hipError_t launch_tiling<EPI_LORA_GATE>(const GemmParams&, int, hipStream_t);

// Compute units of the current device (cached per device id).
int compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// The tiling of a call, from its shape alone.
//
// A tiling's cost is the work of the busiest CU: ceil(tiles / CUs) tiles of
// BM x BN outputs (two co-resident tiles share one CU's throughput), divided
// by the tiling's relative throughput per output (larger tiles read fewer
// operand bytes per MFMA).  The cheapest wins, larger tiles first on ties.
// The 3-slot 128x128 form runs only where the grid fits one round; with more
// tiles the 2-slot form, two per CU, hides each tile's latency behind the
// other's.  The throughputs come from a sweep of every tiling over the
// skinny, adapter, 4096x3072x3072 and 32760x5120x13824 shapes, and of the
// 256-row and 128x128 tilings over 2048-8192 rows of K = 5120 linears.
struct Tiling {
  int bm, bn;
  double rate;          // relative throughput per output
  bool one_round_only;  // only where every tile gets a CU of its own
};
constexpr Tiling kTilings[GEMM_TILINGS] = {
    {256, 256, 1.00, false}, {256, 192, 0.92, false}, {256, 128, 0.82, false},
    {128, 192, 0.85, false}, {128, 128, 0.75, false}, {128, 128, 0.85, true},
    {128, 64, 0.60, false},  {64, 64, 0.50, false},
};

// branch_cols > 0 (a LoRA epilogue with several adapter branches of that many
// columns): only tilings whose wave width (BN / 2) divides branch_cols, so that
// each wave's columns belong to one branch.  The 128x64 and 64x64 tilings
// (32-column waves) serve every multiple of 32.
int pick_tiling(int64_t m, int64_t n, int64_t cus, int64_t branch_cols) {
  auto allowed = [&](int t) { return branch_cols <= 0 || branch_cols % (kTilings[t].bn / 2) == 0; };
  // Grids of three or more rounds of 256x256 tiles are MFMA-bound, and there
  // the largest tile's operand reuse wins: at 4095 x 5120 x 13824 it takes
  // 0.246 ms against 0.251 for 256x192, 0.265 for 256x128 and 0.272-0.274 for
  // the 128-row tiles (whose throughputs below come from one-round grids).
  if (((m + 255) / 256) * ((n + 255) / 256) >= 3 * cus && allowed(GEMM_256x256))
    return GEMM_256x256;
  int best = -1;
  double best_cost = 0.0;
  for (int t = 0; t < GEMM_TILINGS; ++t) {
    const Tiling& c = kTilings[t];
    if (!allowed(t)) continue;
    const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
    if (c.one_round_only && tiles > cus) continue;
    const double cost = (double)((tiles + cus - 1) / cus) * c.bm * c.bn / c.rate;
    if (best < 0 || cost < best_cost) {
      best = t;
      best_cost = cost;
    }
  }
  return best;
}

// Tile-order group height.  The 256x256 tiling sweeps four tile rows at a time
// when the output has at most 48 tile columns (N <= 12288) and three when it
// has more; the tiles resident on one XCD then share a few A and W panels in
// that XCD's L2.  Measured at M = 32760 against heights 2, 3 and 4 in
// alternating runs: height 4 is the fastest or within 0.3 % for N of 3072 to
// 10240 and the FFN down projection (height 3 up to 2.5 % slower there);
// height 3 is 0.5-0.8 % faster than 2 at N = 13824 and 15360 and 2.5-3 % at
// N = 28672 and the SwiGLU projection (112 column tiles).  The other tilings,
// on grids of one or a few rounds, use eight.
int tiling_group_m(int tiling, int64_t tile_cols) {
  if (tiling != GEMM_256x256) return 8;
  return tile_cols <= 48 ? 4 : 3;
}

// Whether the last round of a 256x256 grid is split into smaller tiles, so that
// its few tiles spread over all CUs (bit-identical: every tiling is).  With two
// or more whole rounds and at most half a round left, as 256x128 (one round of
// them), in microseconds: 4095 x 5120 x 13824 235 -> 225 (3.375 rounds), 8190 x
// 5376 x 7168 251 -> 234 (3.5), 20000 x 3072 x 5120 271 -> 261 (6.17), gate-residual
// 32760 x 14336 x 5376 1941 -> 1913 (10.5).  With one whole round, where the
// 256x192 tiling's 1.5 rounds beat two, with at most a quarter round left, as
// 128x128: 4095 x 5120 x 5120 93 -> 88.5 (1.25 rounds), with gate-residual 123 ->
// 111 and at K = 13824 259 -> 241.  More left than that is slower: 4200 x 5376 x
// 5376 102 -> 115 (1.40 rounds), 12000 x 5120 x 13824 606 -> 618 (9.91), 5000 x 5120
// x 5120 112 -> 124 (1.56).
// Only K % 128 == 0, whose whole tiles run the split ring: any other K takes the
// two-slot ring in every tile, and no mixed kernel is built or measured on that
// one.  The adapter epilogues have none either: their tiles of either size would
// need the adapter products in both halves of the kernel, which was not tried.
static int mixed_tail(const GemmParams& p, int tiling, int64_t tiles, int64_t cus) {
  const int64_t full = tiles / cus, rem = tiles % cus;
  if (p.k % 128 || rem == 0 || full < 1) return MIXED_NONE;
  if (full >= 2) return tiling == GEMM_256x256 && 2 * rem <= cus ? MIXED_256x128 : MIXED_NONE;
  return tiling == GEMM_256x192 && 4 * rem <= cus ? MIXED_128x128 : MIXED_NONE;
}

// SwiGLU: the 256x256 tiles that run whole when the rest runs as 64x256 tiles, or
// -1 where splitting does not pay: only while the 64x256 tiles fit one round.
// Microseconds whole and split at K 5376, F 14336: 9 rows 52.4, 44.8; 100 rows
// 55.0, 48.6; 1100 179, 155 (two rounds and 48 tiles); 3000 382, 356; at 300 x 2048
// x 4096 28.8, 15.1.  With more than a round of them: 300 rows 59.3, 91.7; 777
// rows 127, 140; 1024 131, 149.
// The limit of eight whole rounds is no measured crossing: past it the share that a
// split can save only shrinks.  Without the limit, whole and split: 5376 rows 659,
// 634 (9.2 rounds); 7680 925, 902 (13.1); 14080 1664, 1638 (24.1); 30464 3590, 3554
// (52.1).  Other K than multiples of 128, and the adapter form: as at mixed_tail.
static int64_t swiglu_main_tiles(const GemmParams& p, int64_t cus) {
  if (p.k % 128) return -1;
  const int64_t tiles_m = (p.m + 255) / 256, tiles_n = p.half_n / 128, tiles = tiles_m * tiles_n;
  const int64_t main = tiles / cus * cus;
  if (tiles == main || main >= 8 * cus) return -1;
  // 64-row tiles of the last round that hold any row (grouped_tile's order).
  int64_t live = 0;
  for (int64_t t = main; t < tiles; ++t) {
    const int64_t group = t / (p.group_m * tiles_n), first = group * p.group_m;
    const int64_t rows = tiles_m - first < p.group_m ? tiles_m - first : p.group_m;
    const int64_t tm = first + (t - group * p.group_m * tiles_n) % rows;
    const int64_t left = (p.m - tm * 256 + 63) / 64;
    live += left < 4 ? left : 4;
  }
  return live <= cus ? main : -1;
}

// Rows per workgroup (32 or 64) of the few-row kernel, or 0: the smaller one whose
// workgroups all get a CU of their own.  Two on a CU share its LDS and L1 and lose
// what the split of roles gains.  Microseconds, 64x64 tiles -> 32 rows, 64 rows:
// 17 x 5120 x 5120 11.1 -> 7.6, 8.5; 17 x 14336 x 5376 24.1 -> 14.8, 16.4; 64 x
// 3072 x 3072 8.8 -> 6.1, 6.6; 64 x 5120 x 5120 12.4 -> 13.4 (320 workgroups), 9.6;
// 17 x 5120 x 13824 13.4 -> 13.5 (432), 14.5; 128 x 5120 x 5120 12.5 -> 20.4, 15.8.
static int skinny_rows(const GemmParams& p, int64_t cus) {
  const int64_t cols = (p.n + 31) / 32;
  if ((p.m + 31) / 32 * cols <= cus) return 32;
  return (p.m + 63) / 64 * cols <= cus ? 64 : 0;
}

// GemmParams::group_m is set here from the tiling.
hipError_t launch_fp8_gemm(const GemmParams& params, int epi, hipStream_t s) {
  GemmParams p = params;
  if (epi_swiglu(epi)) {
    // One tiling: 128 value + 128 gate columns, the 256x256 schedule.
    p.group_m = tiling_group_m(GEMM_256x256, (p.half_n + 127) / 128);
    if (epi == EPI_SWIGLU_LORA) return launch_pipe<EPI_SWIGLU_LORA, PipeCfg<256, 256, SPLIT_RING, 0>>(p, s);
    const int64_t whole = swiglu_main_tiles(p, compute_units());
    if (whole >= 0) return launch_mixed<EPI_SWIGLU>(p, whole, MIXED_64x256, s);
    return launch_pipe<EPI_SWIGLU, PipeCfg<256, 256, SPLIT_RING, 0>>(p, s);
  }
  const int skinny = skinny_rows(p, compute_units());
  if (skinny) {
    p.group_m = 1;
    switch (epi) {
      case EPI_BIAS: return launch_skinny<EPI_BIAS>(p, skinny, s);
      case EPI_GATE: return launch_skinny<EPI_GATE>(p, skinny, s);
      case EPI_LORA: return launch_skinny<EPI_LORA>(p, skinny, s);
      case EPI_LORA_GATE: return launch_skinny<EPI_LORA_GATE>(p, skinny, s);
      default: return hipErrorInvalidValue;
    }
  }
  int tiling =
      pick_tiling(p.m, p.n, compute_units(), epi_lora(epi) ? p.lora_branch_cols : 0);
  if (tiling < 0) return hipErrorInvalidValue;
  // Adapter branches that 256x192 tiles would cut inside a wave: the query's
  // choice leaves that tiling out, but its epilogue takes each 32-column block's
  // branch by itself, so the launch may use it where it is the best one.  Merged
  // QKV of 1024 rows at K 5376, 3 x 7168 columns, rank 128: 139 us as 256x128, 126
  // as 256x192 (148 with the adapter gathered block by block in the epilogue);
  // rank 16 121 and 112.
  if (epi_lora(epi) && p.lora_branch_cols % 32 == 0 &&
      pick_tiling(p.m, p.n, compute_units(), 0) == GEMM_256x192)
    tiling = GEMM_256x192;
  // That tile stages adapter rows through 32-bit buffer offsets.
  if (epi_lora(epi) && tiling == GEMM_256x192 && (p.ldt >= (1 << 21) || p.ldb >= (1 << 21)))
    tiling = p.lora_branch_cols % 64 ? GEMM_128x64 : GEMM_256x128;
  p.group_m = tiling_group_m(tiling, (p.n + kTilings[tiling].bn - 1) / kTilings[tiling].bn);
  if (epi == EPI_BIAS || epi == EPI_GATE) {
    const int64_t tiles = ((p.m + 255) / 256) * ((p.n + 255) / 256), cus = compute_units();
    const int tail = mixed_tail(p, tiling, tiles, cus);
    if (tail != MIXED_NONE) {
      p.group_m = tiling_group_m(GEMM_256x256, (p.n + 255) / 256);
      return epi == EPI_BIAS ? launch_mixed<EPI_BIAS>(p, tiles / cus * cus, tail, s)
                             : launch_mixed<EPI_GATE>(p, tiles / cus * cus, tail, s);
    }
  }
  switch (epi) {
    case EPI_BIAS: return launch_tiling<EPI_BIAS>(p, tiling, s);
    case EPI_GATE: return launch_tiling<EPI_GATE>(p, tiling, s);
    case EPI_LORA: return launch_tiling<EPI_LORA>(p, tiling, s);
    case EPI_LORA_GATE: return launch_tiling<EPI_LORA_GATE>(p, tiling, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vfa
