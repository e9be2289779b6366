// Host-side launch helpers shared by the C-ABI translation units.
#pragma once

#include <stdarg.h>
#include <stdio.h>

#include "gemm_ring.h"

namespace ws {

// Status codes returned by every entry point.
enum Status { kOk = 0, kInvalid = 1, kHipError = 2 };

int set_error(int code, const char* fmt, ...);  // records the thread's last error, returns code
int device_cus();                               // compute units of the current device
int ensure_lds(const void* kernel, int bytes);  // raises the kernel's dynamic LDS limit on this device to >= bytes

// Whether a pointer is aligned to `bytes`.
inline bool al(const void* p, int bytes) { return reinterpret_cast<unsigned long>(p) % bytes == 0; }

inline int hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) return set_error(kHipError, "%s: %s", what, hipGetErrorString(e));
  return kOk;
}

// Storage mode of a GEMM operand: `rows` is the operand's M (A) or N (B) extent and
// `K` the reduction length. The vector modes need 16-byte aligned rows and runs whose
// length is a multiple of 8 along the contiguous dimension.
inline int classify(const void* ptr, long s_row, long s_k, long rows, long K) {
  const unsigned long p = reinterpret_cast<unsigned long>(ptr);
  if (s_k == 1 && p % 16 == 0 && s_row % 8 == 0 && K % 8 == 0) return kKContig;
  if (s_row == 1 && p % 16 == 0 && s_k % 8 == 0 && rows % 8 == 0) return kMNContig;
  return kGeneric;
}

// The generic loader computes 64-bit addresses; the vector loaders use 32-bit offsets
// relative to a per-tile base, bounded here.
inline bool offsets_fit(int mode, long s_row, long s_k, int tile_rows) {
  const long lim = 0x7fffffffL;
  if (mode == kKContig) return (long)tile_rows * s_row * 2 + 2 * kBK < lim;
  if (mode == kMNContig) return (long)kBK * s_k * 2 + 2L * tile_rows < lim;
  return true;
}

struct LaunchCfg {
  int persistent;  // grid = resident workgroups instead of one per tile
  int splits;      // split-K slices (blockIdx.y)
  int workers;     // > 0: exactly this many workgroups (balanced accumulation)
};
// The fused entry points' 256 x 256 launches: one workgroup per CU looping over the tiles.
// A workgroup that ends and a new one that starts on the freed CU leave it idle for
// about 3 us per tile; the persistent grid keeps that to about 1 us (the forward
// projections and the LM-head GEMMs 2-4 % faster, results bit-identical).
constexpr LaunchCfg kFusedCfg{1, 1, 0};

template <int BM, int BN, int WM, int WN, int AM, int BMD, bool PAIRED, class Epi>
int run_gemm(GemmParams p, LaunchCfg cfg, hipStream_t stream) {
  constexpr int NT = WM * WN * kWave;
  constexpr int lds = gemm_lds_bytes<BM, BN>();
  const void* kern = reinterpret_cast<const void*>(&gemm_kernel<BM, BN, WM, WN, AM, BMD, PAIRED, Epi>);
  if (int rc = ensure_lds(kern, lds)) return rc;
  const int cols = PAIRED ? p.H : p.N;
  const int bn_cols = PAIRED ? BN / 2 : BN;
  p.tiles_m = cdiv(p.M, BM);
  p.tiles_n = cdiv(cols, bn_cols);
  p.total_tiles = p.tiles_m * p.tiles_n;
  const int k_tiles = cdiv(p.K, kBK);
  const int splits = cfg.splits < 1 ? 1 : cfg.splits;
  p.k_tiles_per_split = cdiv(k_tiles, splits);
  if (p.k_tiles_per_split < 1) p.k_tiles_per_split = 1;
  const int resident = device_cus() * (lds > 80 * 1024 ? 1 : 2);
  dim3 grid(cfg.persistent ? (p.total_tiles < resident ? p.total_tiles : resident) : p.total_tiles,
            splits);
  hipLaunchKernelGGL((gemm_kernel<BM, BN, WM, WN, AM, BMD, PAIRED, Epi>), grid, dim3(NT), lds,
                     stream, p);
  return hip_check(hipGetLastError(), "gemm launch");
}

// Large tile: 256 x 256 with 8 waves (64 x 128 per wave). Small tile: 128 x 128 with
// 4 waves (64 x 64 per wave), two workgroups per CU.
enum TileCfg { kTileLarge = 0, kTileSmall = 1 };

#define WS_TILE_ARGS_LARGE 256, 256, 4, 2
#define WS_TILE_ARGS_SMALL 128, 128, 2, 2

}  // namespace ws

namespace ws {

// Layout-combination bit for (A mode, B mode).
constexpr unsigned ab_bit(int am, int bm) { return 1u << (am * 3 + bm); }
constexpr unsigned kMaskKK = ab_bit(kKContig, kKContig);
constexpr unsigned kMaskGG = ab_bit(kGeneric, kGeneric);
constexpr unsigned kMaskMM = kMaskKK | ab_bit(kKContig, kMNContig) | ab_bit(kMNContig, kKContig) |
                             ab_bit(kMNContig, kMNContig) | kMaskGG;

// Runs the instantiation for (am, bm) if MASK holds it, demoting an operand to the
// generic loader otherwise.
template <unsigned MASK, int BM, int BN, int WM, int WN, bool PAIRED, class Epi>
int dispatch(const GemmParams& p, int am, int bm, LaunchCfg cfg, hipStream_t s) {
  auto has = [](int a, int b) { return (MASK & ab_bit(a, b)) != 0; };
  if (!has(am, bm)) {
    if (has(am, kGeneric)) bm = kGeneric;
    else if (has(kGeneric, bm)) am = kGeneric;
    else { am = kGeneric; bm = kGeneric; }
  }
#define WS_CASE(A_, B_)                                                            \
  case A_ * 3 + B_:                                                                \
    if constexpr ((MASK & ab_bit(A_, B_)) != 0)                                    \
      return run_gemm<BM, BN, WM, WN, A_, B_, PAIRED, Epi>(p, cfg, s);             \
    break;
  switch (am * 3 + bm) {
    WS_CASE(0, 0) WS_CASE(0, 1) WS_CASE(0, 2)
    WS_CASE(1, 0) WS_CASE(1, 1) WS_CASE(1, 2)
    WS_CASE(2, 0) WS_CASE(2, 1) WS_CASE(2, 2)
  }
#undef WS_CASE
  return set_error(kInvalid, "no GEMM instantiation for operand layouts (%d, %d)", am, bm);
}

inline bool fits_i32(long v) { return v >= 0 && v < 0x7fffffffL; }

// Epilogues address an output tile through a buffer resource of at most 2 GiB that starts
// at the tile's first row, so 256 rows of an output (row stride `ld` elements of
// `elem_bytes`) must span less than that; wider outputs are rejected instead of losing
// stores past the limit.
inline int check_out_stride(long ld, int elem_bytes, const char* what) {
  if ((long)kFBM * ld * elem_bytes + (long)kFBN * elem_bytes >= 0x7fffffffL)
    return set_error(kInvalid, "%s row stride %ld is too large: a 256-row tile spans 2 GiB or more",
                     what, ld);
  return kOk;
}

// Fast path (gemm_fast.h): 256 x 256 tiles, direct-to-LDS loads, 16x16x32 MFMA.
template <int AM, int BMD, bool PAIRED, class Epi>
int run_fast(GemmParams p, LaunchCfg cfg, hipStream_t stream) {
  const void* kern = reinterpret_cast<const void*>(&gemm_fast_kernel<AM, BMD, PAIRED, Epi>);
  if (int rc = ensure_lds(kern, kFLdsBytes)) return rc;
  const int cols = PAIRED ? p.H : p.N;
  const int bn_cols = PAIRED ? kFBN / 2 : kFBN;
  p.tiles_m = cdiv(p.M, kFBM);
  p.tiles_n = cdiv(cols, bn_cols);
  p.total_tiles = p.tiles_m * p.tiles_n;
  const int k_tiles = cdiv(p.K, kFBK);
  const int splits = cfg.splits < 1 ? 1 : cfg.splits;
  p.k_tiles_per_split = cdiv(k_tiles, splits);
  if (p.k_tiles_per_split < 1) p.k_tiles_per_split = 1;
  const int resident = device_cus();
  dim3 grid(cfg.persistent ? (p.total_tiles < resident ? p.total_tiles : resident) : p.total_tiles,
            splits);
  if (cfg.workers > 0) grid = dim3(cfg.workers, 1);
  hipLaunchKernelGGL((gemm_fast_kernel<AM, BMD, PAIRED, Epi>), grid, dim3(kFNT), kFLdsBytes, stream, p);
  return hip_check(hipGetLastError(), "gemm launch");
}

// True when both operand modes can take the fast path for a 256-row tile. The vector
// modes already guarantee 16-byte aligned chunks and whole-chunk edges; the per-tile
// 32-bit offsets are bounded here (paired B tiles reach `half` rows further).
inline bool fast_ok(const GemmParams& p, int am, int bm, bool paired) {
  if (am == kGeneric || bm == kGeneric || !p.vec_out) return false;
  const long lim = 0x7fffffffL;
  const long half = paired ? p.H : 0;
  if (am == kKContig && (256L + 1) * p.a.s_row * 2 >= lim) return false;
  if (am == kMNContig && 2L * 256 + 64L * p.a.s_k * 2 >= lim) return false;
  if (bm == kKContig && (256L + half + 1) * p.b.s_row * 2 >= lim) return false;
  if (bm == kMNContig && 2L * (256 + half) + 64L * p.b.s_k * 2 >= lim) return false;
  return true;
}

template <bool PAIRED, class Epi>
int dispatch_fast(const GemmParams& p, int am, int bm, LaunchCfg cfg, hipStream_t s) {
  switch (am * 2 + bm) {
    case 0: return run_fast<kKContig, kKContig, PAIRED, Epi>(p, cfg, s);
    case 1: return run_fast<kKContig, kMNContig, PAIRED, Epi>(p, cfg, s);
    case 2: return run_fast<kMNContig, kKContig, PAIRED, Epi>(p, cfg, s);
    default: return run_fast<kMNContig, kMNContig, PAIRED, Epi>(p, cfg, s);
  }
}

// Macro-tiles of the vector-operand GEMMs: 256 x 256 (gemm_fast.h) and the ring kernel's
// smaller ones (gemm_ring.h). Two 64 to 80 KiB workgroups fit a CU except for kTile128x1,
// which takes the CU alone with eight waves and four stages.
typedef RingCfg<128, 128, 2, 2, 2> Ring128x2;
typedef RingCfg<128, 128, 4, 2, 4> Ring128x1;
typedef RingCfg<64, 128, 2, 2, 3> Ring64x128;
typedef RingCfg<64, 64, 2, 2, 4> Ring64;
enum FastTile { kTile256 = 0, kTile128x2, kTile128x1, kTile64x128, kTile64, kFastTiles };

// Cost of one launch of each macro-tile in microseconds, fitted to sweeps of 150 shapes and
// epilogues (128 to 16384 rows, 512 to 32768 columns, K 512 to 16384; outputs of all tiles the
// same bits). Over 1600 others (128 to 16384 rows, 256 to 16384 columns, K 128 to 16384) the
// picks are 1.3 to 3.3 % behind the best tile in the mean, by layout, and at most 47 %. A CU
// runs its workgroups in rounds of one (`pair` 0) or two at a time; a round takes `alone` us per
// 64-deep k-tile for one workgroup, `pair` us for two that share the CU, and `fixed` us
// around the k-loop. The 256 x 256 tile costs less per product with every CU busy; below about
// one round of its tiles most CUs idle, and a smaller tile wins although it loads its operands
// more often. Measured, us (256 x 256 against the choice): 512 x 1280 x 8960 130 / 41 (64 x 64),
// 1999 x 1280 x 8960 131 / 78 (64 x 128; 128 x 128 alone would take 73), 4096 x 2048 x 5632
// 98 / 78 and 4096 x 1280 x 6400 102 / 72 (128 x 128 paired), 128 x 4800 x 960 20 / 7.5
// (64 x 64); and where it stays: 1999 x 8960 x 1280 56 / 55, 8192 x 10240 x 2048 238 / 294,
// 8192 x 2048 x 2048 51 / 60 (the best smaller tile).
struct TileCost {
  int bm, bn;
  float alone, pair, fixed;  // pair 0: one workgroup per CU
  // Over several rounds of pairs the workgroups drift apart and share less in L2: `pair`
  // starts `settle` lower and grows by `drift` per k-tile beyond 32, to `most` at the end.
  float settle, drift, most;
  // Rows off whole 128-byte lines: the k-loop's factor when the contiguous reduction is no
  // multiple of 64 (each row piece spans two lines), and us per round for such outputs.
  float ragged_k, ragged_n;
};
inline const TileCost& tile_cost(int tile, int am, int bm) {
  static const TileCost kk[kFastTiles] = {
      {256, 256, 1.43f, 0.0f, 4.0f, 0, 0, 0, 1.05f, 5.0f},
      {128, 128, 0.62f, 0.87f, 3.2f, 0.07f, 0.006f, 0.18f, 1.25f, 5.0f},
      {128, 128, 0.50f, 0.0f, 3.6f, 0, 0, 0, 1.1f, 1.7f},
      {64, 128, 0.34f, 0.50f, 3.6f, 0.0f, 0.005f, 0.16f, 1.2f, 1.0f},
      {64, 64, 0.28f, 0.33f, 3.4f, 0.0f, 0.0015f, 0.09f, 1.4f, 0.5f}};
  static const TileCost kmn[kFastTiles] = {
      {256, 256, 1.48f, 0.0f, 4.0f, 0, 0, 0, 1.05f, 5.0f},
      {128, 128, 0.64f, 0.89f, 3.2f, 0.07f, 0.006f, 0.18f, 1.25f, 5.0f},
      {128, 128, 0.53f, 0.0f, 3.6f, 0, 0, 0, 1.1f, 1.7f},
      {64, 128, 0.38f, 0.53f, 3.6f, 0.0f, 0.005f, 0.16f, 1.2f, 1.0f},
      {64, 64, 0.31f, 0.36f, 3.4f, 0.0f, 0.0015f, 0.09f, 1.4f, 0.5f}};
  static const TileCost mnmn[kFastTiles] = {
      {256, 256, 1.52f, 0.0f, 4.0f, 0, 0, 0, 1.0f, 5.0f},
      {128, 128, 0.60f, 1.00f, 3.2f, 0, 0, 0, 1.0f, 5.0f},
      {128, 128, 0.54f, 0.0f, 3.6f, 0, 0, 0, 1.0f, 1.7f},
      {64, 128, 0.39f, 0.70f, 3.6f, 0, 0, 0, 1.0f, 1.0f},
      {64, 64, 0.29f, 0.42f, 3.4f, 0, 0, 0, 1.0f, 0.5f}};
  if (am == kKContig && bm == kKContig) return kk[tile];
  return (am == kMNContig && bm == kMNContig ? mnmn : kmn)[tile];
}
// What an epilogue costs beside a plain BF16 store, us per round of 256 x 256 tiles (every CU
// in it at once, bound by HBM): the SwiGLU backward reads and writes the packed projection,
// 8192 x 4096 x 1024 97 us against 56. A smaller tile's round pays by its area; two
// workgroups on a CU hide a tenth of it behind each other's k-loop.
enum EpiCost { kEpiStore = 0, kEpiSigmoid = 2, kEpiSwiglu = 4, kEpiF32 = 6, kEpiF32Add = 18, kEpiSwigluBwd = 20 };

// An [m, n] output (n the packed width of a paired GEMM) with reduction k in `copies` split-K
// slices. A last round in which only some CUs hold a pair is priced between a lone workgroup's
// time and a pair's, or with `some_pairs` us per k-tile.
inline float tile_time(int tile, long m, long n, long k, int am, int bm, int cus, bool paired,
                       float epi, long copies = 1, float some_pairs = 0.0f) {
  const TileCost& c = tile_cost(tile, am, bm);
  const long tiles = (long)cdiv(m, c.bm) * cdiv(n, c.bn) * copies;
  const float kt = (float)cdiv(cdiv(k, kFBK), copies), area = (float)(c.bm * c.bn) / 65536.0f;
  const float slow = k % kFBK ? c.ragged_k : 1.0f;
  const float fixed = c.fixed + ((paired ? n / 2 : n) % kFBK ? c.ragged_n : 0.0f);
  const float alone = c.alone * slow;
  if (c.pair == 0.0f) {
    const long rounds = tiles / cus, rest = tiles % cus;
    if (tile != kTile256) return (float)(rounds + (rest != 0)) * (alone * kt + fixed + epi * area);
    // With most CUs idle in the last round its tiles' loads meet less traffic.
    float t = (float)rounds * (alone * kt + fixed + epi);
    if (rest) t += alone * (0.65f + 0.30f * (float)rest / (float)cus) * kt + fixed + epi;
    return t;
  }
  const long rounds = tiles / (2 * cus), rest = tiles % (2 * cus);
  const float around = fixed + epi * area * 1.8f;
  const float pair = c.pair * slow > some_pairs ? c.pair * slow : some_pairs;
  float drift = 0.0f;
  if (tiles > 2 * cus) {
    drift = -c.settle + c.drift * (kt - 32.0f);
    drift = drift < -c.settle ? -c.settle : drift > c.most ? c.most : drift;
  }
  float t = (float)rounds * ((pair + drift) * kt + around);
  if (rest > cus)  // some CUs hold a pair
    t += (some_pairs > 0.0f ? some_pairs : alone + (pair - alone) * (float)(rest - cus) / (float)cus) * kt +
         around;
  else if (rest)
    t += alone * kt + fixed + epi * area;
  return t;
}
// The macro-tile with the lowest cost; a smaller one must promise 5 % over 256 x 256.
inline int pick_tile(long m, long n, long k, int am, int bm, bool paired, float epi,
                     float* time = nullptr) {
  const int cus = device_cus();
  int best = kTile256;
  const float whole = tile_time(kTile256, m, n, k, am, bm, cus, paired, epi);
  float t = 0.95f * whole;
  // A paired 64 x 64 tile would write 32-byte row pieces.
  for (int i = 1; i < (paired ? kTile64 : kFastTiles); ++i) {
    const float ti = tile_time(i, m, n, k, am, bm, cus, paired, epi);
    if (ti < t) {
      best = i;
      t = ti;
    }
  }
  if (time) *time = best == kTile256 ? whole : t;
  return best;
}

template <class Cfg, int AM, int BMD, bool PAIRED, class Epi>
int run_ring(GemmParams p, int splits, hipStream_t stream) {
  const void* kern = reinterpret_cast<const void*>(&gemm_ring_kernel<Cfg, AM, BMD, PAIRED, Epi>);
  if (int rc = ensure_lds(kern, Cfg::kLds)) return rc;
  p.tiles_m = cdiv(p.M, Cfg::BM);
  p.tiles_n = cdiv(PAIRED ? p.H : p.N, PAIRED ? Cfg::BN / 2 : Cfg::BN);
  p.total_tiles = p.tiles_m * p.tiles_n;
  p.k_tiles_per_split = cdiv(cdiv(p.K, kFBK), splits);
  hipLaunchKernelGGL((gemm_ring_kernel<Cfg, AM, BMD, PAIRED, Epi>), dim3(p.total_tiles, splits),
                     dim3(Cfg::NT), Cfg::kLds, stream, p);
  return hip_check(hipGetLastError(), "gemm launch");
}

template <int AM, int BMD, bool PAIRED, class Epi>
int run_ring_tile(const GemmParams& p, int tile, hipStream_t s, int splits = 1) {
  switch (tile) {
    case kTile128x2: return run_ring<Ring128x2, AM, BMD, PAIRED, Epi>(p, splits, s);
    case kTile128x1: return run_ring<Ring128x1, AM, BMD, PAIRED, Epi>(p, splits, s);
    case kTile64x128: return run_ring<Ring64x128, AM, BMD, PAIRED, Epi>(p, splits, s);
    default:
      if constexpr (!PAIRED) return run_ring<Ring64, AM, BMD, PAIRED, Epi>(p, splits, s);
  }
  return set_error(kInvalid, "no GEMM macro-tile %d", tile);
}

// The fast path with the macro-tile picked by tile_time. A rule's mask holds the operand layouts
// (ab_bit) the smaller tiles are built for; the others run on 256 x 256 tiles.
constexpr unsigned kMaskKRows = ab_bit(kKContig, kKContig) | ab_bit(kKContig, kMNContig);
constexpr unsigned kMaskVector = kMaskKRows | ab_bit(kMNContig, kKContig) | ab_bit(kMNContig, kMNContig);
struct TileRule {
  unsigned mask;
  bool paired;
  EpiCost epi;
};
// By WsEpilogue (include/warpstate_hip.h).
constexpr TileRule kTileRules[] = {{kMaskVector, false, kEpiStore},
                                   {kMaskKRows, false, kEpiStore},
                                   {kMaskKRows, false, kEpiSigmoid},
                                   {kMaskKRows, true, kEpiSwiglu},
                                   {kMaskKRows, false, kEpiSwigluBwd}};
inline int rule_tile(const TileRule& r, long m, long n, long k, int am, int bm) {
  return (r.mask & ab_bit(am, bm)) ? pick_tile(m, n, k, am, bm, r.paired, r.epi) : kTile256;
}

template <int RULE, class Epi>
int dispatch_tiles(const GemmParams& p, int am, int bm, LaunchCfg cfg, hipStream_t s) {
  constexpr unsigned MASK = kTileRules[RULE].mask;
  constexpr bool PAIRED = kTileRules[RULE].paired;
  const int tile = rule_tile(kTileRules[RULE], p.M, p.N, p.K, am, bm);
  if (tile == kTile256) return dispatch_fast<PAIRED, Epi>(p, am, bm, cfg, s);
#define WS_RING(A_, B_)                                                          \
  if constexpr ((MASK & ab_bit(A_, B_)) != 0)                                    \
    if (am == A_ && bm == B_) return run_ring_tile<A_, B_, PAIRED, Epi>(p, tile, s);
  WS_RING(0, 0) WS_RING(0, 1) WS_RING(1, 0) WS_RING(1, 1)
#undef WS_RING
  return set_error(kInvalid, "no GEMM instantiation for operand layouts (%d, %d)", am, bm);
}

}  // namespace ws
