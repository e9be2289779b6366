// BF16 GEMM for outputs that are too small to fill the GPU with 256 x 256 tiles.
//
// The same operands, LDS layouts, MFMA (v_mfma_f32_16x16x32_bf16), accumulator layout and
// epilogues as gemm_fast.h, on smaller macro-tiles: each output element sums its products in
// the same order, so the results are the same bits. One workgroup per tile; S LDS stages in
// a ring, both operands of a k-tile loaded S - 1 k-tiles ahead:
//   wait for this wave's loads of the k-tile (the S - 2 later tiles' stay in flight),
//   s_barrier, issue the loads of the tile S - 1 ahead into the stage that every wave has
//   finished reading, then the two k32 steps on this stage.
// The ring keeps S - 1 tiles of operands in flight: a BM x BN tile moves (BM + BN) x 128 bytes
// per 64 k from L2 into LDS, at 44 bytes per clock and CU at most, against BM BN 128 / 4096
// clocks of MFMA. Neither is at its limit in the counters (10 to 31 bytes per clock and CU, the
// matrix pipe 8 to 45 % busy, over products of 512 to 4096 rows): a 64 x 64 tile alone on a CU
// takes 0.28 us per k-tile where its loads need 0.17 and its MFMAs 0.06. What is left is the
// chain from a barrier through the fragment reads to the MFMAs, with two workgroups at most to
// hide it, and last rounds that leave CUs idle.
#pragma once

#include "gemm_fast.h"

namespace ws {

// A wait for every LDS read issued so far that also redefines the N fragment registers, so
// that no MFMA reading them can be scheduled ahead of it (tie_wait of gemm_fast.h).
template <int N>
__device__ __forceinline__ void tie_frags(bf16x8_t (&f)[N]) {
  static_assert(N == 4 || N == 6 || N == 8, "fragment counts of the ring tiles");
  if constexpr (N == 4)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3])::"memory");
  else if constexpr (N == 6)
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5])::"memory");
  else
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]),
                   "+v"(f[7])::"memory");
}

// Macro-tile of the ring kernel: BM x BN outputs on WM x WN waves, S LDS stages.
template <int BM_, int BN_, int WM_, int WN_, int S_>
struct RingCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_;
  static constexpr int NT = WM * WN * kWave;
  static constexpr int TM = BM / WM, TN = BN / WN, FA = TM / 16, FB = TN / 16;
  static constexpr int kTileA = BM * 128, kTileB = BN * 128, kStage = kTileA + kTileB;
  static constexpr int kEpi = WM * WN * epi_wave<FA, FB>();
  static constexpr int kLds = S * kStage > kEpi ? S * kStage : kEpi;
  static_assert(S >= 2 && kLds <= 160 * 1024, "the stages fit a CU's LDS");
};

// Fragment i (A blocks, then B blocks) of k32 step STEP as an assembly read. K-contiguous
// blocks are 16 rows (2048 bytes) apart at one base address per step; M/N-contiguous ones
// have a base each (the swizzle mixes the block index into the address).
template <class Cfg, int AMODE, int BMODE, int STEP, int I>
__device__ __forceinline__ bf16x8_t ring_read(const unsigned (&abase)[Cfg::FA],
                                              const unsigned (&bbase)[Cfg::FB], unsigned st) {
  constexpr bool kA = I < Cfg::FA;
  constexpr int mode = kA ? AMODE : BMODE, j = kA ? I : I - Cfg::FA;
  if constexpr (mode == kKContig) {
    // Step 1 is chunk c ^ 4: 64 bytes away in the swizzled row.
    const unsigned base = (kA ? abase[0] : bbase[0]) ^ (STEP * 64);
    return b128_read<j * 2048>(base + st);
  } else {
    const unsigned base = kA ? abase[kA ? j : 0] : bbase[kA ? 0 : j];
    return tr_frag<STEP>(base + st);
  }
}

template <class Cfg, int AMODE, int BMODE, int STEP, int I>
__device__ __forceinline__ void ring_read_all(bf16x8_t (&f)[Cfg::FA + Cfg::FB],
                                              const unsigned (&abase)[Cfg::FA],
                                              const unsigned (&bbase)[Cfg::FB], unsigned st) {
  if constexpr (I < Cfg::FA + Cfg::FB) {
    f[I] = ring_read<Cfg, AMODE, BMODE, STEP, I>(abase, bbase, st);
    ring_read_all<Cfg, AMODE, BMODE, STEP, I + 1>(f, abase, bbase, st);
  }
}

// MFMA n of step 0, with step 1's fragment r read after MFMA ceil(r NM / NF).
template <class Cfg, int AMODE, int BMODE, int N>
__device__ __forceinline__ void ring_step0(Acc16<Cfg::FA, Cfg::FB>& acc,
                                           bf16x8_t (&f0)[Cfg::FA + Cfg::FB],
                                           bf16x8_t (&f1)[Cfg::FA + Cfg::FB],
                                           const unsigned (&abase)[Cfg::FA],
                                           const unsigned (&bbase)[Cfg::FB], unsigned st) {
  constexpr int NM = Cfg::FA * Cfg::FB, NF = Cfg::FA + Cfg::FB;
  static_assert(NF <= NM, "a read slot per MFMA");
  if constexpr (N < NM) {
    constexpr int i = N / Cfg::FB, j = N % Cfg::FB;
    acc.v[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f0[Cfg::FA + j], f0[i], acc.v[i][j], 0, 0, 0);
    if constexpr ((N * NF) % NM < NF) {
      constexpr int r = N * NF / NM;
      f1[r] = ring_read<Cfg, AMODE, BMODE, 1, r>(abase, bbase, st);
    }
    __builtin_amdgcn_sched_barrier(0);
    ring_step0<Cfg, AMODE, BMODE, N + 1>(acc, f0, f1, abase, bbase, st);
  }
}

// Workgroups that run at once (two on each of 256 CUs): the XCD remap deals each such window
// of the raster out in eight runs of neighbouring tiles (against one run per XCD over the
// whole grid, the paired tiles are 0.5-1 % faster).
constexpr int kRingWindow = 512;

template <class Cfg, int AMODE, int BMODE, bool PAIRED, class Epi>
__global__ void __launch_bounds__(Cfg::NT) gemm_ring_kernel(const GemmParams p) {
  static_assert(AMODE != kGeneric && BMODE != kGeneric, "vector operands only");
  constexpr int FA = Cfg::FA, FB = Cfg::FB, NM = FA * FB, NF = FA + FB, S = Cfg::S;
  constexpr int TM = Cfg::TM, TN = Cfg::TN;
  constexpr bool kAsm = AMODE == kMNContig || BMODE == kMNContig;

  extern __shared__ __attribute__((aligned(1024))) unsigned char rsmem[];
  if (p.skip_if != nullptr && *p.skip_if != 0) return;  // uniform: the whole grid exits

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int kb = blockIdx.y * p.k_tiles_per_split;
  const int ke = min(cdiv(p.K, kFBK), kb + p.k_tiles_per_split);

  int tm, tn;
  tile_position(xcd_remap(blockIdx.x, p.total_tiles, kRingWindow), p.tiles_m, p.tiles_n, tm, tn);
  const int row0_a = tm * Cfg::BM;
  const int row0_b = tn * (PAIRED ? Cfg::BN / 2 : Cfg::BN);

  RingTile<Cfg::BM, Cfg::NT, AMODE, false> la;
  RingTile<Cfg::BN, Cfg::NT, BMODE, PAIRED> lb;
  la.init(p.a, row0_a, p.M, 0, wave, lane);
  lb.init(p.b, row0_b, PAIRED ? p.H : p.N, PAIRED ? p.H : 0, wave, lane);
  constexpr int kWaitLoads = (RingTile<Cfg::BM, Cfg::NT, AMODE, false>::kIns +
                              RingTile<Cfg::BN, Cfg::NT, BMODE, PAIRED>::kIns) * (S - 2);

  // Tile rows of this wave's B blocks (paired tiles: up blocks, then gate blocks).
  int b_rb[FB];
#pragma unroll
  for (int j = 0; j < FB; ++j)
    b_rb[j] = PAIRED ? (j < FB / 2 ? wn * (TN / 2) + 16 * j
                                   : Cfg::BN / 2 + wn * (TN / 2) + 16 * (j - FB / 2))
                     : wn * TN + 16 * j;

  Acc16<FA, FB> acc;
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) acc.v[i][j] = f32x4_v{0.f, 0.f, 0.f, 0.f};

  // Loads ahead past the end of K land as zeros. A slice that ends before K loads the next
  // slice's first S - 1 tiles there, which nothing reads: ending the loads with the slice costs
  // more than that traffic (768 x 512 over 15360 tokens in four slices 38.5 -> 40.5 us).
  auto issue = [&](int kt, int stage) {
    unsigned char* st = rsmem + stage * Cfg::kStage;
    la.issue(p.a, row0_a, kt * kFBK, p.K, st, wave, lane);
    lb.issue(p.b, row0_b, kt * kFBK, p.K, st + Cfg::kTileA, wave, lane);
  };
  if (kb < ke) {
#pragma unroll
    for (int s = 0; s + 1 < S; ++s) issue(kb + s, s);
    unsigned abase[FA], bbase[FB];
    if constexpr (kAsm) {
      const unsigned lds0 =
          (unsigned)(unsigned long)(__attribute__((address_space(3))) unsigned char*)rsmem;
      auto base = [&](int mode, int rb) -> unsigned {
        if (mode == kMNContig) return tr_base(rb, lane);
        const int r = rb + (lane & 15);
        return r * 128 + (((lane >> 4) ^ swz(r)) << 4);
      };
#pragma unroll
      for (int i = 0; i < FA; ++i) abase[i] = lds0 + base(AMODE, wm * TM + 16 * i);
#pragma unroll
      for (int j = 0; j < FB; ++j) bbase[j] = lds0 + Cfg::kTileA + base(BMODE, b_rb[j]);
    }
    int rd = 0, wr = S - 1;
    for (int kt = kb; kt < ke; ++kt) {
      __builtin_amdgcn_s_waitcnt(wait_vmcnt(kWaitLoads));
      __builtin_amdgcn_s_barrier();
      // Stage wr was read in the previous k-tile, which every wave has left (barrier).
      issue(kt + S - 1, wr);
      wr = wr + 1 == S ? 0 : wr + 1;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kAsm) {
        const unsigned char* sa = rsmem + rd * Cfg::kStage;
        const unsigned char* sb = sa + Cfg::kTileA;
        bf16x8_t af[2][FA], bf[2][FB];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
          for (int i = 0; i < FA; ++i) af[s][i] = read_frag(sa, wm * TM + 16 * i, s, lane);
#pragma unroll
          for (int j = 0; j < FB; ++j) bf[s][j] = read_frag(sb, b_rb[j], s, lane);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < FA; ++i)
#pragma unroll
            for (int j = 0; j < FB; ++j)
              acc.v[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[s][j], af[s][i], acc.v[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, NF, 0);
#pragma unroll
        for (int r = 0; r < NF; ++r) {
          __builtin_amdgcn_sched_group_barrier(0x008, NM / NF > 0 ? NM / NF : 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      } else {
        const unsigned st = (unsigned)(rd * Cfg::kStage);
        bf16x8_t f0[NF], f1[NF];
        ring_read_all<Cfg, AMODE, BMODE, 0, 0>(f0, abase, bbase, st);
        tie_frags(f0);
        __builtin_amdgcn_sched_barrier(0);
        ring_step0<Cfg, AMODE, BMODE, 0>(acc, f0, f1, abase, bbase, st);
        tie_frags(f1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < FA; ++i)
#pragma unroll
          for (int j = 0; j < FB; ++j)
            acc.v[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f1[FA + j], f1[i], acc.v[i][j], 0, 0, 0);
      }
      rd = rd + 1 == S ? 0 : rd + 1;
      // This wave's fragment reads are complete (its MFMAs have issued) before the barrier
      // that lets other waves' loads overwrite the stage.
      __builtin_amdgcn_sched_barrier(0);
    }
    // The loads past the last k-tile land, and every wave is done reading, before the
    // epilogue's staging writes.
    __builtin_amdgcn_s_waitcnt(wait_vmcnt(0));
    __builtin_amdgcn_s_barrier();
  }
  Epi::run(p, acc, row0_a + wm * TM, row0_b + (PAIRED ? wn * (TN / 2) : wn * TN), lane, tm, tn, wn,
           rsmem + wave * epi_wave<FA, FB>());
}

}  // namespace ws
