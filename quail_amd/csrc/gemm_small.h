// The promotion form of the FP8 block-scaled GEMM for few token rows (the
// 256 x 256 and 256 x 320 tiles of gemm_fp8.hip are for full packs): the
// same 16x16x128 MFMA per 128-K block summed from zero and the same
// total = fma(sA * sW, partial, total) in K order, so every tile here gives
// the bits of configs 30 and 31.
//
// What bounds it. At 46 rows Qwen3-4B's down projection is 8 (256 x 320) or
// 10 tiles: 10 of 256 CUs read 25 MB of weights, 97 us where the bytes take
// 5. Smaller tiles put every CU to work; then a tile's time is its chain of
// K blocks (76 of them): a barrier, the fragments' LDS reads (a 64 x 64 tile
// reads 48 KiB of fragments for 16 KiB of operands), the MFMAs and the direct
// loads, measured 0.17 (16 x 32) to 0.98 us (256 x 128) a block with one
// workgroup per CU. The reads and the MFMAs run one after the other: the next
// block's scales are multiplied as they are read, ahead of the current
// block's MFMAs, and LDS reads return in order, so a wave waits for most of
// the next block's reads first (s_waitcnt lgkmcnt(5) and (2) of 19 reads on
// 256 x 128 and 128 x 256, of 13 on 192 x 64; (10) of 14 on 64 x 64, where
// the scales come early). A 128 x 256 block reads 128 KiB, about 0.5 us, and
// has 0.5 us of MFMAs in its measured 1.0-1.4. Memory is not what they wait
// for: with every operand already in L2 the mid tiles run only 5-15% faster,
// and a copy of the loads alone draws 120 GB/s per CU from L2 where the tiles
// draw 41-61; the 76 gate_up tiles of 256 weight rows are the exception (12
// us with the weights in L2, 23 without).
//   46 rows, K = 9728, N = 2560:  97 -> 14.5 us (16 x 32 tiles)
//   333 rows, same:               98 -> 25 us (64 x 64)
//   1003 rows, same:              98 -> 44 us (192 x 64)
//   46 rows, gate_up + SiLU-quant (K = 2560, 2 x 9728): 41 -> 24 us (64 x 256)
// Measured and not kept: weights loaded straight into registers with only
// the tokens in LDS (1.2-1.5x the time), the K blocks of one tile spread
// over eight waves whose partials meet in LDS (faster below 8 rows at long
// K only: 11.8 against 14.1 us at one row), no fragments read ahead, 16
// waves on the 64- and 128-wide tiles (0.97-1.05x), 4 waves (1.2-1.7x), one
// scale load per stage instead of per block (0.97-1.05x).
#pragma once

#include "qx_common.h"

namespace qx {

// LDS reads of this wave done (vmcnt and expcnt unconstrained), then the
// workgroup barrier
__device__ __forceinline__ void lds_reads_barrier() {
  __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));
  asm volatile("s_barrier" ::: "memory");
}

__device__ __forceinline__ v8i frag16(v4i lo, v4i hi) {
  return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// this workgroup's tile id: a contiguous band of ids per XCD (blockIdx mod
// 8), so that the tiles that share weight rows share an L2
__device__ __forceinline__ int xcd_tile(int total) {
  const int per = (total + 7) / 8;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int full = total - (per - 1) * 8;
  return xcd < full ? xcd * per + local : full * per + (xcd - full) * (per - 1) + local;
}

constexpr int kSwigluRow = 528;  // a staged row of 128 gate and 128 up bf16, padded over the banks

// SiLU, product and per-128 quant of a staged tile's rows (16 lanes each)
template <int BM, int NW>
__device__ __forceinline__ void swiglu_quant_rows(const uint8_t* smem, int wave, int lane, int m0,
                                                  int j0, int M, uint8_t* __restrict__ Q,
                                                  int64_t q_ld, float* __restrict__ Qs,
                                                  int64_t qs_ld) {
  const int seg = lane & 15;
  for (int g4 = wave; g4 < BM / 4; g4 += NW) {
    const int prow = g4 * 4 + (lane >> 4);
    const int m = m0 + prow;
    swiglu_quant_row<false>(smem + prow * kSwigluRow, seg, m < M,
                            Q + (int64_t)m * q_ld + j0 + seg * 8,
                            Qs + (int64_t)(j0 >> 7) * qs_ld + m);
  }
}

// BM tokens x BN weights by WM x WN waves; the operands of KPB 128-K blocks
// make a stage, STAGES of them a ring
template <int BM, int BN, int WM, int WN, int STAGES, int KPB>
struct RingCfg {
  static constexpr int kWaves = WM * WN;
  static constexpr int kSlabs = (BM + BN) / 8;                       // 1 KiB loads per block
  static constexpr int kPer = (kSlabs + kWaves - 1) / kWaves;        // of which a wave issues
  static constexpr int kOps = KPB * (kPer + 1);                      // and its scale load
  static constexpr int kBlock = (BM + BN) * 128 + kWaves * 256;
  static constexpr int kStage = KPB * kBlock;
  static constexpr int kLds = STAGES * kStage;
  static_assert(BM % 16 == 0 && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "16 x 16 tiles");
  static_assert(BN / WN <= 128 && 128 % (BN / WN) == 0, "a wave's rows lie in one scale block");
  static_assert(kWaves * 64 >= BM + 2, "scale slots");
  static_assert(kLds <= 160 * 1024, "LDS");
  static_assert(STAGES >= 2 && (STAGES - 1) * kOps < 64, "vmcnt");
};

// One workgroup per tile. Operands go memory -> LDS by direct loads the
// compiler does not track (its own waits would drain the ring), rows of 128
// bytes with chunk c at position c ^ (row % 8). KPB blocks share one
// barrier: behind it the next group's fragments are read into registers, the
// current group's MFMAs run (behind most of those reads: see above), and the
// stage just left is refilled.
// Two or four blocks per barrier on the small tiles, whose block is shorter
// than a barrier's skew (16 x 32 with four: 16.3 -> 14.1 us at K = 9728);
// the wide tiles have neither the LDS nor the need.
template <int BM, int BN, int WM, int WN, int STAGES, int KPB, bool SWIGLU>
__global__ __launch_bounds__(64 * WM * WN) void gemm_fp8_promo_ring_kernel(
    const uint8_t* __restrict__ A, const float* __restrict__ sA, const uint8_t* __restrict__ W,
    const float* __restrict__ sW, uint16_t* __restrict__ C, int M, int N, int K, int64_t lda,
    int64_t ldc, int64_t sa_ld, int tiles_m, int tiles_n, uint8_t* __restrict__ Q, int64_t q_ld,
    float* __restrict__ Qs, int64_t qs_ld) {
  using Cfg = RingCfg<BM, BN, WM, WN, STAGES, KPB>;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int NW = Cfg::kWaves;
  static_assert(!SWIGLU || BN == 256, "SwiGLU tiles: 128 gate + 128 up rows");
  // The refill goes out behind the reads, and behind the MFMAs as well where
  // the registers allow it (in front of both before: 277 rows of 5120 x 25600
  // under 128 x 64 tiles 92.5 -> 88.2 us, 600 under 192 x 128 164 -> 157, 1260
  // of 2560 x 4096 under 128 x 128 25.5 -> 24.1; the 256 x 128 and the
  // SiLU-quant tiles spill with it last: 30 -> 64 us, behind the reads 29.3).
  constexpr bool kIssueLast = !SWIGLU && BM * BN < 256 * 128;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Cfg::kLds];

  const int id = xcd_tile(tiles_m * tiles_n);
  const int m0 = (id % tiles_m) * BM;  // the tiles of one weight band are neighbours
  const int n0 = (id / tiles_m) * BN;
  const int KT = K >> 7;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wm = wave / WN;
  const int r16 = lane & 15, q16 = lane >> 4;

  // this lane's part of the wave's loads: slab i of a block is tile rows
  // 8 i .. 8 i + 7, token rows first; lane l brings chunk (l % 8) ^ (l / 8)
  // of row l / 8 to LDS position l
  const uint8_t* src[Cfg::kPer];
  const int w_row0 = SWIGLU ? n0 >> 1 : n0;
#pragma unroll
  for (int j = 0; j < Cfg::kPer; ++j) {
    const int slab = min(wave * Cfg::kPer + j, Cfg::kSlabs - 1);  // repeats rewrite their bytes
    const int chunk = ((lane & 7) ^ (lane >> 3)) * 16;
    if (slab < BM / 8) {
      const int row = min(m0 + slab * 8 + (lane >> 3), M - 1);
      src[j] = A + (int64_t)row * lda + chunk;
    } else {
      const int r = (slab - BM / 8) * 8 + (lane >> 3);
      const int row = w_row0 + r + (SWIGLU && r >= 128 ? (N >> 1) - 128 : 0);
      src[j] = W + (int64_t)row * K + chunk;
    }
  }
  // scale slots: the tile's token scales, then its weight scales (one per
  // 128-row block)
  const float* ssrc;
  int64_t sstep;
  {
    constexpr int kBlocks = SWIGLU ? 2 : (BN + 127) / 128;
    const int slot = wave * 64 + lane;
    if (slot < BM) {
      ssrc = sA + min(m0 + slot, M - 1);
      sstep = sa_ld;
    } else {
      const int nb = min(slot - BM, kBlocks - 1);
      ssrc = sW + (int64_t)(SWIGLU ? (w_row0 + nb * (N >> 1)) >> 7 : (n0 >> 7) + nb) * KT;
      sstep = 1;
    }
  }
  // a group's blocks past the last are not loaded
  int issued = 0;  // blocks issued
  int ist = 0;     // the stage of the next group
  auto issue = [&]() {
#pragma unroll
    for (int g = 0; g < KPB; ++g) {
      if (KPB > 1 && issued >= KT) break;
      uint8_t* buf = smem + ist * Cfg::kStage + g * Cfg::kBlock;
#pragma unroll
      for (int j = 0; j < Cfg::kPer; ++j) {
        const int slab = min(wave * Cfg::kPer + j, Cfg::kSlabs - 1);
        lds_dma16_stream(src[j], buf + slab * 1024);
        src[j] += 128;
      }
      lds_dma4(ssrc, buf + (BM + BN) * 128 + wave * 256);
      ssrc += sstep;
      ++issued;
    }
    ist = ist + 1 == STAGES ? 0 : ist + 1;
  };

  struct Frags {
    v8i w[TN], a[TM];
    float s[TM];
  };
  const int lo = r16 * 128 + ((q16 ^ (r16 & 7)) * 16);
  const int hi = r16 * 128 + (((q16 + 4) ^ (r16 & 7)) * 16);
  const int sw_slot = BM + (wn * (BN / WN)) / 128;
  int rst = 0;  // the stage read next
  auto read = [&](Frags (&f)[KPB]) {
#pragma unroll
    for (int g = 0; g < KPB; ++g) {
      const uint8_t* blk = smem + rst * Cfg::kStage + g * Cfg::kBlock;
      const uint8_t* al = blk + wm * TM * 2048;
      const uint8_t* wl = blk + BM * 128 + wn * TN * 2048;
      const float* sl = reinterpret_cast<const float*>(blk + (BM + BN) * 128);
#pragma unroll
      for (int a = 0; a < TN; ++a)
        f[g].w[a] = frag16(*reinterpret_cast<const v4i*>(wl + a * 2048 + lo),
                           *reinterpret_cast<const v4i*>(wl + a * 2048 + hi));
#pragma unroll
      for (int b = 0; b < TM; ++b)
        f[g].a[b] = frag16(*reinterpret_cast<const v4i*>(al + b * 2048 + lo),
                           *reinterpret_cast<const v4i*>(al + b * 2048 + hi));
      const float sw = sl[sw_slot];
#pragma unroll
      for (int b = 0; b < TM; ++b) f[g].s[b] = sl[(wm * TM + b) * 16 + r16] * sw;
    }
    rst = rst + 1 == STAGES ? 0 : rst + 1;
  };

  v4f tot[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b) tot[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
  auto block = [&](const Frags& f) {
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        const v4f part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
            f.w[a], f.a[b], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) tot[a][b][e] = __builtin_fmaf(f.s[b], part[e], tot[a][b][e]);
      }
  };

#pragma unroll
  for (int st = 0; st < STAGES; ++st)
    if (issued < KT) issue();
  if (STAGES * KPB <= KT) wait_vmcnt<(STAGES - 1) * Cfg::kOps>(); else wait_vmcnt<0>();
  lds_barrier();
  Frags f0[KPB], f1[KPB];
  read(f0);
  // one group: cur is in registers, nxt the next group's
  auto step = [&](int g, Frags (&cur)[KPB], Frags (&nxt)[KPB]) {
    // group g + 1 has landed (the later ones may be in flight: whole ones, or
    // the wait is for everything), and every wave holds group g in registers:
    // its stage takes group g + STAGES
    if ((g + STAGES) * KPB <= KT) wait_vmcnt<(STAGES - 2) * Cfg::kOps>(); else wait_vmcnt<0>();
    lds_reads_barrier();
    if ((g + 1) * KPB < KT) read(nxt);  // past the last block: bytes never used
    if (!kIssueLast && issued < KT) issue();
    if ((g + 1) * KPB <= KT) {
#pragma unroll
      for (int u = 0; u < KPB; ++u) block(cur[u]);
    } else {
#pragma unroll
      for (int u = 0; u < KPB - 1; ++u)
        if (g * KPB + u < KT) block(cur[u]);
    }
    if (kIssueLast && issued < KT) issue();
  };
  const int groups = (KT + KPB - 1) / KPB;
  for (int g = 0; g < groups; g += 2) {
    step(g, f0, f1);
    if (g + 1 < groups) step(g + 1, f1, f0);
  }

  if constexpr (SWIGLU) {
    static_assert(BM * kSwigluRow <= Cfg::kLds, "the tile is staged in the ring");
    __syncthreads();
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      uint8_t* row = smem + ((wm * TM + b) * 16 + r16) * kSwigluRow;
#pragma unroll
      for (int a = 0; a < TN; ++a)
        *reinterpret_cast<uint2*>(row + (wn * TN * 16 + a * 16 + q16 * 4) * 2) =
            make_uint2(pack2_bf16(tot[a][b][0], tot[a][b][1]), pack2_bf16(tot[a][b][2], tot[a][b][3]));
    }
    __syncthreads();
    swiglu_quant_rows<BM, NW>(smem, wave, lane, m0, n0 >> 1, M, Q, q_ld, Qs, qs_ld);
  } else {
#pragma unroll
    for (int b = 0; b < TM; ++b) {
      const int m = m0 + (wm * TM + b) * 16 + r16;
      if (m < M) {
        uint16_t* dst = C + (int64_t)m * ldc + n0 + wn * TN * 16 + q16 * 4;
#pragma unroll
        for (int a = 0; a < TN; ++a)
          *reinterpret_cast<uint2*>(dst + a * 16) = make_uint2(
              pack2_bf16(tot[a][b][0], tot[a][b][1]), pack2_bf16(tot[a][b][2], tot[a][b][3]));
      }
    }
  }
}

}  // namespace qx
