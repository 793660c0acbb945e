// Weight-only linear for gfx950: bf16 activations times a weight restored from
// its E4M3 row codes inside the GEMM.
//
//   w[n, k]  = bf16(e4m3(code[n, k]) * scale[n])      (binary32 product, one rounding)
//   out      = bf16(sum_k x[m, k] * w[n, k] + bias[n]) (binary32 accumulate, one rounding)
//
// The default mode of RowFP8Execution (reference
// src/vflash/native/h3_fp8_linear.py:75-108): the restored weight is bit for bit
// what (weight.float() * scale).to(bfloat16) gives, but it never exists in
// memory.  The eager form writes and reads the weight as binary32 twice and as
// bf16 once, about 18 bytes per element, before its GEMM reads it again; here a
// weight costs its one byte.
//
// Each stage holds 64 K of the tile: activation rows of 128 bytes and code rows
// of 64 bytes, in an NS-slot LDS ring filled by buffer-load-to-LDS DMA.  For
// MFMA step v (0..3) of a stage, lanes 0-31 supply K 8v .. +7 and lanes 32-63
// K 32 + 8v .. +7 of both operands (the sum does not depend on the K order), so
// a lane reads 64 contiguous bytes of an activation row and 32 contiguous codes
// of a weight row.  A weight fragment costs 16 VALU instructions per lane (four
// paired conversions, eight multiplies, four paired roundings) against 32
// cycles for each MFMA it feeds: tiles of several 32-row activation blocks per
// wave share it, and the conversion of step v + 1 is interleaved with the MFMAs
// of step v.
#include "gemm_epilogue.h"

namespace vfa {

template <int BM, int BN, int NS>
struct W16Layout {
  static constexpr int A = BM * 128, W = BN * 64, SLOT = A + W;
  static constexpr int OUT = BM * BN * 2;  // the epilogue's bf16 staging tile
  static constexpr int RING = NS * SLOT > OUT ? NS * SLOT : OUT;
  static constexpr int DMA = SLOT / 4096;  // DMA instructions per wave and stage
  static constexpr int PER_CU = 2 * (RING + VEC_LDS) <= 160 * 1024 ? 2 : 1;
};

template <int BM, int BN, int NS, int WGM>
__global__ void __launch_bounds__(256, (W16Layout<BM, BN, NS>::PER_CU)) w8a16_gemm_pipe(
    const GemmParams p) {
  using L = W16Layout<BM, BN, NS>;
  constexpr int WGN = 4 / WGM;
  static_assert(BM % (32 * WGM) == 0 && BN % (32 * WGN) == 0 && BM % 64 == 0 && BN % 64 == 0 &&
                NS % 2 == 0 && (NS - 1) * L::DMA < 64, "tiling");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[L::RING];
  __shared__ __attribute__((aligned(1024))) uint8_t vec[VEC_LDS];
  constexpr int WM = BM / WGM, WN = BN / WGN, MB = WM / 32, NB = WN / 32;
  int tm, tn;
  tile_coords((int)((p.m + BM - 1) / BM), (int)((p.n + BN - 1) / BN), p.group_m, tm, tn);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = (int)threadIdx.x & 63;
  const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(lds_addr(ring));
  const int wm = wave % WGM, wn = wave / WGM;
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t rows_a = min((int64_t)BM, p.m - m0), rows_w = min((int64_t)BN, p.n - n0);
  // p.lda counts bytes here as everywhere; resources end with the tile's last
  // whole row, so rows past the operand read as zeros.
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a + m0 * p.lda, (uint32_t)(rows_a * p.lda));
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w + n0 * p.ldw, (uint32_t)(rows_w * p.ldw));
  const int64_t ka = 2 * p.k;  // activation row bytes
  const int KT = (int)((p.k + 63) / 64);

  // DMA lane maps (those of the NVFP4 GEMM): 128-byte rows in the lds_swizzle
  // chunk order, 64-byte rows with chunk c in slot c ^ ((row >> 2) & 3).
  const int drow = lane >> 3;
  const int ach0 = (lane & 7) ^ lds_swizzle(drow), ach1 = (lane & 7) ^ lds_swizzle(drow + 8);
  const uint32_t a_base0 = (uint32_t)((wave * (BM / 4) + drow) * p.lda + ach0 * 16);
  const uint32_t a_base1 = (uint32_t)((wave * (BM / 4) + drow + 8) * p.lda + ach1 * 16);
  const uint32_t a_step = (uint32_t)(16 * p.lda);
  const int wch = (lane & 3) ^ ((lane >> 4) & 3);
  const uint32_t w_base = (uint32_t)((wave * (BN / 4) + (lane >> 2)) * p.ldw + wch * 16);
  const uint32_t w_step = (uint32_t)(16 * p.ldw);
  const uint32_t dst_a = ring_lds + wave * (L::A / 4), dst_w = ring_lds + L::A + wave * (L::W / 4);
  // Stage s into slot j; chunks past K and stages past the end read as zeros.
  auto issue = [&](int j, int s) {
    const uint32_t slot = (uint32_t)j * L::SLOT;
    const int64_t kb = (int64_t)s * 128, kw = (int64_t)s * 64;
    const uint32_t kill0 = kb + ach0 * 16 < ka ? 0u : VFA_OOB;
    const uint32_t kill1 = kb + ach1 * 16 < ka ? 0u : VFA_OOB;
    const uint32_t killw = kw + wch * 16 < p.k ? 0u : VFA_OOB;
    static_for<BM / 32>([&](auto i) {
      const uint32_t off = (i % 2 ? a_base1 : a_base0) + (i / 2) * a_step + (uint32_t)kb;
      lds_dma16(ra, dst_a + slot + i * 1024, off | (i % 2 ? kill1 : kill0));
    });
    static_for<BN / 64>([&](auto i) {
      lds_dma16(rw, dst_w + slot + i * 1024, (w_base + i * w_step + (uint32_t)kw) | killw);
    });
  };

  const int fr = lane & 31, fh = lane >> 5;
  const int asw = lds_swizzle(fr), wsw = (fr >> 2) & 3;
  // The scale of each weight row this lane restores (rows past N: zero codes).
  float sc[NB];
  static_for<NB>([&](auto nb) {
    const int64_t n = n0 + wn * WN + nb * 32 + fr;
    sc[nb] = n < p.n ? p.sw[n] : 0.0f;
  });
  struct Raw {
    v4i a[MB][4];
    v4i w[NB][2];
  };
  auto read_raw = [&](Raw& r, int j) {
    const uint8_t* base = ring + j * L::SLOT;
    static_for<NB>([&](auto nb) {
      const uint8_t* row = base + L::A + (wn * WN + nb * 32 + fr) * 64;
      static_for<2>([&](auto c) {
        r.w[nb][c] = *reinterpret_cast<const v4i*>(row + (((2 * fh + c) ^ wsw) << 4));
      });
    });
    static_for<MB>([&](auto mb) {
      const uint8_t* row = base + (wm * WM + mb * 32 + fr) * 128;
      static_for<4>([&](auto c) {
        r.a[mb][c] = *reinterpret_cast<const v4i*>(row + (((4 * fh + c) ^ asw) << 4));
      });
    });
  };
  v16f acc[NB][MB];
  static_for<NB>([&](auto i) { static_for<MB>([&](auto jj) { acc[i][jj] = v16f{}; }); });
  struct Ops {
    v4i w[NB];
  };
  // The restored weight fragments of step v of stage kt, held in r.  A 16-code
  // chunk past K multiplies by zero instead of its row's scale, which may be
  // infinite.
  auto convert = [&](const Raw& r, int kt, auto v) {
    Ops o;
    const bool live = (int64_t)kt * 64 + 32 * fh + 16 * (v / 2) < p.k;
    static_for<NB>([&](auto nb) {
      const float s = live ? sc[nb] : 0.0f;
      static_for<2>([&](auto h) {
        const int d = r.w[nb][v / 2][(v % 2) * 2 + h];
        const v2f lo = __builtin_amdgcn_cvt_pk_f32_fp8(d, false);
        const v2f hi = __builtin_amdgcn_cvt_pk_f32_fp8(d, true);
        o.w[nb][2 * h] = (int)pack_bf16x2(lo[0] * s, lo[1] * s);
        o.w[nb][2 * h + 1] = (int)pack_bf16x2(hi[0] * s, hi[1] * s);
      });
    });
    return o;
  };
  constexpr int VALU = (16 * NB + MB * NB - 1) / (MB * NB);
  // The MFMAs of step v of the stage in r, with the conversion of the next step
  // (step nv of stage nkt, in rn) interleaved.
  auto step = [&](const Ops& cur, const Raw& r, auto v, const Raw& rn, int nkt, auto nv) {
    const Ops nxt = convert(rn, nkt, nv);
    static_for<NB>([&](auto nb) {
      static_for<MB>([&](auto mb) {
        acc[nb][mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(v8bf, cur.w[nb]), __builtin_bit_cast(v8bf, r.a[mb][v]), acc[nb][mb],
            0, 0, 0);
      });
    });
    static_for<NB * MB>([&](auto) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
    });
    __builtin_amdgcn_sched_barrier(0);
    return nxt;
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  Raw r[2];
  stage_vectors<BM, BN>(p, m0, n0, wave, lane, __builtin_amdgcn_readfirstlane(lds_addr(vec)));
  static_for<NS>([&](auto s) { issue((int)s, (int)s); });
  wait_vmcnt<(NS - 1) * L::DMA, true>();  // stage 0 and the vectors, issued before it
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_raw(r[0], 0);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the same pending reads on both loop entries
  Ops cur = convert(r[0], 0, I0{});
  // Stage kt in slot jc, its operands already in r[jc % 2].
  auto stage = [&](int kt, auto jc) {
    constexpr int j = jc;
    Raw &rc = r[j % 2], &rn = r[(j + 1) % 2];
    cur = step(cur, rc, I0{}, rc, kt, I1{});
    // Stage kt+1 has landed for every wave, and every wave has read stage kt.
    wait_vmcnt<(NS - 2) * L::DMA, true>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(j, kt + NS);
    read_raw(rn, (j + 1) % NS);
    cur = step(cur, rc, I1{}, rc, kt, I2{});
    cur = step(cur, rc, I2{}, rc, kt, I3{});
    cur = step(cur, rc, I3{}, rn, kt + 1, I0{});  // zeros past the last stage, never multiplied
  };
  for (int kt = 0; kt < KT; kt += NS)
    static_for<NS>([&](auto i) {
      if (kt + i < KT) stage(kt + i, i);
    });
  wait_vmcnt<0, true>();  // every DMA has landed before the ring becomes the staging tile
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  gemm_epilogue<BM, BN, WGM, WGN, EPI_LINEAR, true>(p, acc, m0, n0, wm, wn, (int)threadIdx.x, ring, vec);
}

int compute_units();

template <int BM, int BN, int NS, int WGM>
static void launch_w16(const GemmParams& p, hipStream_t s) {
  const int64_t tiles = ((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN);
  w8a16_gemm_pipe<BM, BN, NS, WGM><<<dim3((unsigned)tiles), dim3(256), 0, s>>>(p);
}

// The tiling, as in the NVFP4 GEMM: the least estimated time of the busiest CU
// (microseconds at K = 5120; a first tile, and each further one).  Measured at
// N = 5120 as 64x64, 128x64, 128x128 and 128x256: M = 17 26.7, 31.6, 41.1, 63.0;
// M = 200 38.9, 33.5, 43.3, 63.3; M = 512 60.3, 64.5, 44.9, 65.4; M = 1024 98.7,
// 96.9, 89.2, 67.5.  The two widest put their four waves side by side, so that no
// weight fragment is converted twice (2x2 waves: M = 512 50.3, 1024 x 7168 as
// 256x128 83.1 against 81.9).
hipError_t launch_w8a16(const GemmParams& params, hipStream_t s) {
  GemmParams p = params;
  p.group_m = 8;
  const int64_t cus = compute_units();
  auto cost = [&](int bm, int bn, int first, int more) {
    const int64_t tiles = ((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn);
    return first + more * ((tiles + cus - 1) / cus - 1);
  };
  const int64_t c[4] = {cost(128, 256, 66, 77), cost(128, 128, 45, 46), cost(128, 64, 32, 32),
                        cost(64, 64, 27, 14)};
  int best = 0;
  for (int t = 1; t < 4; ++t)
    if (c[t] < c[best]) best = t;
  switch (best) {
    case 0: launch_w16<128, 256, 4, 1>(p, s); break;
    case 1: launch_w16<128, 128, 4, 1>(p, s); break;
    case 2: launch_w16<128, 64, 6, 2>(p, s); break;
    default: launch_w16<64, 64, 6, 2>(p, s); break;
  }
  return hipGetLastError();
}

// The restored weight itself, for products that run on it as a plain bf16
// matrix: 16 codes per lane, out[n, k] = bf16(e4m3(code) * scale[n]).  Bound by
// its three bytes per element.
__global__ void __launch_bounds__(256) restore_rows(const uint8_t* __restrict__ w,
                                                    const float* __restrict__ sw, int64_t n,
                                                    int64_t k, int64_t ldw,
                                                    uint16_t* __restrict__ out) {
  const int64_t row = grid_row();
  if (row >= n) return;
  const float s = sw[row];
  const v4i* src = reinterpret_cast<const v4i*>(w + row * ldw);
  v4i* dst = reinterpret_cast<v4i*>(out + row * k);
  const int vecs = (int)(k / 16);
  for (int j = threadIdx.x; j < vecs; j += 256) {
    const v4i c = __builtin_nontemporal_load(src + j);
    v4i o[2];
    static_for<4>([&](auto i) {
      const v2f lo = __builtin_amdgcn_cvt_pk_f32_fp8(c[(int)i], false);
      const v2f hi = __builtin_amdgcn_cvt_pk_f32_fp8(c[(int)i], true);
      o[i / 2][(i % 2) * 2] = (int)pack_bf16x2(lo[0] * s, lo[1] * s);
      o[i / 2][(i % 2) * 2 + 1] = (int)pack_bf16x2(hi[0] * s, hi[1] * s);
    });
    dst[2 * j] = o[0];
    dst[2 * j + 1] = o[1];
  }
}

hipError_t launch_restore_rows(const uint8_t* w, const float* sw, int64_t n, int64_t k, int64_t ldw,
                               uint16_t* out, hipStream_t s) {
  restore_rows<<<row_grid(n), dim3(256), 0, s>>>(w, sw, n, k, ldw, out);
  return hipGetLastError();
}

}  // namespace vfa
