// Dense MFMA GEMM of the decode + GEMM band: y = x @ W^T (+ bias) on a weight that the one-pass decode has just
// written, f32 accumulate.
//
// What bounds the band's small shapes in a library GEMM is not the arithmetic: a few dozen output tiles leave most compute
// units idle, each walks all of K with little in flight, and the call costs the host more than both kernels together.  Two
// kernels serve the band here.  The wide tiles (wide_gemm.hpp, 64 x 64 to 256 x 256) have a wave per 16 MT x 16 NT of the tile and one ring of
// 64-k steps; which of them a shape takes, and whether K is split over blocks, the plan below estimates.  The kernel in this file splits K over groups of
// waves inside the block (group g takes every KG-th step), and the groups' sums meet in LDS, in their order, without a second kernel or a workspace.  It has two tiles.
// 32 x 64 in four groups of a wave is for what is left without a tile for every compute unit even at 64 x 64, or is a long chain of steps for few: 8 KiB of operands per
// step on their way three steps deep (47 x 384 x 8320 unsplit 16.3 us, the library's product 19.0; 90 x 609 x 13312 28).  64 x 128 in two groups of
// four waves is for long K over few tiles, next to parts of K over blocks: half as many steps one behind the other as in a part of a wide tile.  Decode + product, us, best of all wide
// tiles and splits / this: 548 x 320 x 9728 20.0 / 17.6, 444 x 352 x 9856 19.7 / 17.2, 370 x 659 x 12800 28.9 / 26.6, 601 x 432 x 9344 22.1 / 19.8.
//
// Long reductions over few output tiles leave most of the chip idle all the same, here as in the library.  There K is split over blocks
// too (`splits` parts of equal length, give or take a step): every block stores its f32 tile to the workspace and splitk_reduce_kernel adds
// the parts in their order.  In this kernel the parts of a column tile stay on the die that decoded its rows.
//
// Both operand tiles are loaded straight into LDS (global_load_lds_dwordx4; rows of 128 bytes, 16-byte piece p of
// row r in slot p ^ ((r >> 1) & 7), so that a read of 32 consecutive rows touches every bank group twice), a ring of
// kDenseRing steps per group; one in-order counter tracks a wave's loads and the waits are written by hand.  A wave
// computes 32 x 64 of the tile (MFMA 32x32x16), reading the operands of a k group while it multiplies the one
// before.
// Rows that end inside a step (SHORT) are read where they lie: residual VQ 1157 x 272 at 471 tokens 21.7 -> 9.1 us per call (the library's product
// before), VQ 1920 x 288 at 1590 tokens 13.1 -> 10.8 (x copied to rows of whole steps).
// The row tiles of a column tile go to one die (workgroups go to the eight dies in turn), so that a die's L2
// fetches a column tile of W once for all row tiles.
#include <math.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "dense_gemm.hpp"
#include "gemm_tile.hpp"
#include "lds_transfer.hpp"
#include "table_gemm.hpp"

namespace npamd {

namespace {

constexpr int kDenseRing = 3;  // steps of a group of waves in LDS

// WGM x WGN waves of 32 x 64 and KG groups of them, each with a part of the steps.
template <int WGM, int WGN, int KG>
struct DenseTile {
  static constexpr int kBM = 32 * WGM, kBN = 64 * WGN;
  static constexpr int kWaves = WGM * WGN;  // of one K group
  static constexpr int kThreads = 64 * kWaves * KG;
  static constexpr int kStageBytes = (kBM + kBN) * 128;
  static constexpr int kPiecesX = kBM / 8, kPiecesW = kBN / 8;  // a load's worth of rows
  static constexpr int kLoadsX = (kPiecesX + kWaves - 1) / kWaves, kLoadsW = (kPiecesW + kWaves - 1) / kWaves;  // per wave and step
  static constexpr int kRedBytes = (KG - 1) * kBM * kBN * 4;
  static constexpr int kEpBytes = kBM * kBN * 2;
  static constexpr int kRingBytes = KG * kDenseRing * kStageBytes;
  static constexpr int kLds = kRingBytes > kRedBytes + kEpBytes ? kRingBytes : kRedBytes + kEpBytes;
  static_assert(kLds <= kLdsPerBlockMax, "the block's tiles do not fit LDS");
};

// SHORT: rows end inside the last step.  Loads past their end bring the last piece again, and the operands there are zeroed
// as they are used, in the one step that has any.
template <int ACT, int WGM, int WGN, int KG, bool SHORT>
__global__ void __launch_bounds__((DenseTile<WGM, WGN, KG>::kThreads))
dense_gemm_kernel(const DenseShape s) {
  using T = DenseTile<WGM, WGN, KG>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // blockIdx.x % 8 names the die; a die takes an eighth of the units, counted down the columns
  const int unit = (blockIdx.x & 7) * s.units_per_die + (blockIdx.x >> 3);
  const int rt = unit % s.row_tiles, part = unit / s.row_tiles % s.splits, ct = unit / s.row_tiles / s.splits;
  if (ct >= s.col_tiles) return;
  const int step0 = (int)((int64_t)s.steps * part / s.splits);
  const int steps = (int)((int64_t)s.steps * (part + 1) / s.splits) - step0;  // of this part
  const int m0 = rt * T::kBM, n0 = ct * T::kBN;

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave_all / T::kWaves, wave = wave_all % T::kWaves;
  const int wm = wave % WGM, wn = wave / WGM;
  const int c = lane & 31, h = lane >> 5;

  const int steps_g = (steps - g + KG - 1) / KG;  // this group's steps: g, g + KG, ... of the part
  const int base = steps / KG;                    // steps every group has
  const int64_t part_at = SHORT ? 0 : (int64_t)step0 * 128;
  const uint8_t* const xb = reinterpret_cast<const uint8_t*>(s.x) + (int64_t)m0 * s.ldx * 2 + part_at;
  const uint8_t* const wb = reinterpret_cast<const uint8_t*>(s.w) + (int64_t)n0 * s.ldw * 2 + part_at;
  // The piece of its operand that load i brings.  Where the waves don't divide the pieces, the last is brought more than once.
  auto piece_of = [&](int i) {
    return i < T::kLoadsX ? min(wave + T::kWaves * i, T::kPiecesX - 1) : min(wave + T::kWaves * (i - T::kLoadsX), T::kPiecesW - 1);
  };
  uint32_t voff[T::kLoadsX + T::kLoadsW];
#pragma unroll
  for (int i = 0; i < T::kLoadsX + T::kLoadsW; ++i) {
    const bool is_x = i < T::kLoadsX;
    const int r = piece_of(i) * 8 + (lane >> 3);
    const int row = is_x ? min(r, s.M - 1 - m0) : min(r, s.N - 1 - n0);  // rows past the end: a valid row nobody stores
    voff[i] = (uint32_t)((int64_t)row * (is_x ? s.ldx : s.ldw) * 2) + (SHORT ? 0u : (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16));
  }
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + (uint32_t)(g * kDenseRing * T::kStageBytes);
  auto load = [&](int i, int slot, int it) {
    const bool is_x = i < T::kLoadsX;
    const uint32_t piece = (uint32_t)((is_x ? 0 : T::kPiecesX) + piece_of(i));
    if constexpr (SHORT) {
      const int p = (lane & 7) ^ ((piece_of(i) * 4 + (lane >> 4)) & 7);  // of the step, as above
      const uint32_t at = voff[i] + (uint32_t)min((step0 + g + KG * it) * 8 + p, s.pieces - 1) * 16u;
      lds_load16(ring + (uint32_t)(slot * T::kStageBytes) + piece * 1024u, at, uniform_ptr(is_x ? xb : wb));
      return;
    }
    const uint8_t* src = uniform_ptr((is_x ? xb : wb) + (int64_t)(g + KG * it) * 128);
    lds_load16(ring + (uint32_t)(slot * T::kStageBytes) + piece * 1024u, voff[i], src);
  };

  f32x16 acc[1][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[0][t][i] = 0.f;

  constexpr int kLoads = T::kLoadsX + T::kLoadsW;
#pragma unroll
  for (int p = 0; p < kDenseRing - 1; ++p)
    if (p < steps_g) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) load(i, p, p);
    }

  uint32_t slot_off[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) slot_off[j] = (uint32_t)((((h << 2) | j) ^ ((c >> 1) & 7)) << 4);
  const uint8_t* const ring_p = lds + g * kDenseRing * T::kStageBytes;
  const uint32_t a_off = (uint32_t)((wm * 32 + c) * 128), b_off = (uint32_t)((T::kBM + wn * 64 + c) * 128);
  u32x4 ao[2], bo[2][2];
  auto read_ops = [&](int set, const uint8_t* stage, int j) {
#pragma unroll
    for (int t = 0; t < 2; ++t) bo[set][t] = *reinterpret_cast<const u32x4*>(stage + b_off + t * 4096 + slot_off[j]);
    ao[set] = *reinterpret_cast<const u32x4*>(stage + a_off + slot_off[j]);
  };

  // One step out of ring slot `slot`: the operands of k group j + 1 are read in front of the MFMAs of group j, and with
  // LOADS the pieces of step `ahead` are requested behind them, into the slot of the step before this one.  `there`: pieces of the step
  // in front of the rows' end (SHORT).
  auto compute = [&](auto loads, int slot, int ahead, int there) {
    constexpr bool LOADS = decltype(loads)::value;
    const uint8_t* const stage = ring_p + slot * T::kStageBytes;
    const int into = slot == 0 ? kDenseRing - 1 : slot - 1;
    read_ops(0, stage, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) read_ops((j + 1) & 1, stage, j + 1);
      if constexpr (SHORT && !LOADS) {  // the last step is never one that requests another
        const bool dead = 4 * h + j >= there;
#pragma unroll
        for (int t = 0; t < 2; ++t) bo[j & 1][t] = dead ? u32x4{0, 0, 0, 0} : bo[j & 1][t];
        ao[j & 1] = dead ? u32x4{0, 0, 0, 0} : ao[j & 1];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        acc[0][t] = mfma32<ACT>(ao[j & 1], bo[j & 1][t], acc[0][t]);
        if constexpr (LOADS) {
#pragma unroll
          for (int i = (j * 2 + t) * kLoads / 8; i < (j * 2 + t + 1) * kLoads / 8; ++i) load(i, into, ahead);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto pieces_there = [&](int it) { return s.pieces - (step0 + g + KG * it) * 8; };
  int slot = 0;
  auto next_slot = [&] { slot = slot == kDenseRing - 1 ? 0 : slot + 1; };
  int it = 0;
  // Steps every group has, while there is something left to request.
  for (; it < base - (kDenseRing - 1); ++it) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kDenseRing - 2) * kLoads) : "memory");
    block_sync_lds();  // everybody's pieces have arrived, and nobody reads the slot of the step before any more
    compute(std::true_type{}, slot, it + kDenseRing - 1, 8);
    next_slot();
  }
  for (; it < base; ++it) {
    // The step's pieces have arrived when only those of the one behind it are still on their way.
    if (it == base - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    block_sync_lds();
    if (it + kDenseRing - 1 < steps_g) {  // the last step of a group that has one more than the others
#pragma unroll
      for (int i = 0; i < kLoads; ++i) load(i, slot == 0 ? kDenseRing - 1 : slot - 1, it + kDenseRing - 1);
    }
    compute(std::false_type{}, slot, 0, pieces_there(it));
    next_slot();
  }
  if (steps % KG) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    block_sync_lds();
    if (base < steps_g) compute(std::false_type{}, slot, 0, pieces_there(base));
  }

  // The groups' sums meet in group 0, in group order.
  __syncthreads();
  if (g > 0) {
    float* mine = reinterpret_cast<float*>(lds) + ((size_t)(g - 1) * T::kWaves + wave) * 2048 + lane * 4;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(mine + (t * 4 + q) * 256) =
            f32x4{acc[0][t][4 * q], acc[0][t][4 * q + 1], acc[0][t][4 * q + 2], acc[0][t][4 * q + 3]};
  }
  __syncthreads();
  if (g > 0) return;
#pragma unroll
  for (int o = 0; o < KG - 1; ++o) {
    const float* theirs = reinterpret_cast<const float*>(lds) + ((size_t)o * T::kWaves + wave) * 2048 + lane * 4;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(theirs + (t * 4 + q) * 256);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0][t][4 * q + e] += v[e];
      }
  }
  if (s.splits > 1) {
    // D[m = 8 (i / 4) + 4 h + i % 4][n = c] of each 32 x 32 tile
    float* const mine = s.partials + (size_t)part * s.M * s.N;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int n = n0 + wn * 64 + t * 32 + c;
      if (n >= s.N) continue;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + wm * 32 + 8 * (i / 4) + 4 * h + (i % 4);
        if (m < s.M) mine[(size_t)m * s.N + n] = acc[0][t][i];
      }
    }
    return;
  }
  store_wave_tile<ACT, 1, 2>(acc, lds + T::kRedBytes + wave * 4096, lane, s.y, s.ldy, m0 + wm * 32, n0 + wn * 64, s.M, s.N, s.bias);
}

template <int ACT, int WGM, int WGN, int KG>
int launch_dense_tile(DenseShape s, hipStream_t st) {
  using T = DenseTile<WGM, WGN, KG>;
  s.row_tiles = (s.M + T::kBM - 1) / T::kBM;
  s.col_tiles = (s.N + T::kBN - 1) / T::kBN;
  const int64_t units = (int64_t)s.col_tiles * s.row_tiles * s.splits, blocks = (units + 7) / 8 * 8;
  s.units_per_die = (int)(blocks / 8);
  if (blocks > 0x7FFFFFFF) return fail(NPAMD_ERR_UNSUPPORTED, "npamd_dense_gemm: too many tiles");
  static LdsLatch latches[2];
  const bool ends_inside = s.pieces % 8 != 0;
  const auto kernel = ends_inside ? dense_gemm_kernel<ACT, WGM, WGN, KG, true> : dense_gemm_kernel<ACT, WGM, WGN, KG, false>;
  const hipError_t e = enable_dynamic_lds(latches[ends_inside], reinterpret_cast<const void*>(kernel), T::kLds);
  if (e != hipSuccess)
    return fail(NPAMD_ERR_LAUNCH, "npamd_dense_gemm: cannot reserve %d bytes of LDS: %s", T::kLds, hipGetErrorString(e));
  launch(kernel, (unsigned)blocks, T::kThreads, T::kLds, st, s);
  return check_launch("npamd_dense_gemm");
}

// The tiles there are and what a launch on each costs, us: fixed + per round of workgroups + hypot(step time, bytes
// loaded / rate), fitted to 700 shapes of 17 to 4096 rows, 256 to 14336 columns and K of 256 to 14336, fp16 and bf16 (the tile of least
// estimate is 0.2 % slower than the best of them in the mean, 13 % at most; each tile is there because without it that is 0.4 to 7 % in the mean or 15 % and
// more on some shape; estimates are within 4 to 9 %).  A round is one tile per compute unit of every die.  The two legs of the hypot
// are coefficients of the fit, no times of a unit: together a 64-k step of 256 x 256 on every compute unit takes 1.5 us (4096 x 4096 x 4096), of which its 2048 cycles of MFMAs are 1.0
// to 1.2 at the 1.7 to 2.0 GHz that the chip runs at under them.
struct DenseCost {
  int bm, bn, groups;
  float fixed, per_step, per_mb, per_round;
};
constexpr DenseCost kDenseCost[] = {
    {32, 64, 4, 1.438f, 0.420f, 0.040f, 2.328f},   // the kernel above; from here on the wide tiles, numbered as in launch_wide
    {64, 64, 1, 1.319f, 0.164f, 0.028f, 2.617f},
    {64, 128, 1, 1.287f, 0.232f, 0.030f, 3.028f},
    {128, 128, 1, 1.342f, 0.288f, 0.043f, 4.153f},
    {160, 128, 1, 1.179f, 0.342f, 0.047f, 5.014f},
    {256, 128, 1, 1.316f, 0.450f, 0.052f, 5.727f},
    {192, 128, 1, 1.100f, 0.342f, 0.050f, 4.627f},
    {96, 128, 1, 1.275f, 0.265f, 0.037f, 3.473f},
    {160, 256, 1, 0.773f, 0.600f, 0.057f, 7.067f},
    {192, 256, 1, 0.926f, 0.748f, 0.059f, 7.195f},
    {256, 224, 1, 2.348f, 0.814f, 0.067f, 6.872f},
    {256, 256, 1, 2.163f, 0.853f, 0.073f, 7.682f},
    {96, 64, 1, 1.473f, 0.198f, 0.038f, 2.770f},
    {192, 192, 1, 0.000f, 0.487f, 0.055f, 8.035f},
    {64, 128, 2, 2.000f, 0.400f, 0.040f, 0.000f},  // the kernel above again; where the plan looks at it
};
constexpr int kDenseTiles = sizeof(kDenseCost) / sizeof(kDenseCost[0]), kDenseTwoGroups = kDenseTiles - 1;

template <int ACT>
int launch_dense(const DenseShape& s, int tile, hipStream_t st) {
  const int rc = tile == 0 ? launch_dense_tile<ACT, 1, 1, 4>(s, st)
                 : tile == kDenseTwoGroups ? launch_dense_tile<ACT, 2, 2, 2>(s, st)
                                           : launch_wide(s, ACT, tile, st);
  if (rc != NPAMD_OK || s.splits == 1) return rc;
  launch_splitk_reduce<ACT>(s.partials, s.splits, s.M, s.N, s.bias, s.y, s.ldy, st);
  return check_launch("npamd_dense_gemm");
}

constexpr int kDenseMaxSplits = 16;
constexpr int64_t kDenseStrideMax = NPAMD_TILE_MAX_STRIDE;
constexpr int kDenseMinSplitSteps = 4;  // 64-k steps of a part
// What a split of this product adds: the reduction kernel and the gap in front of it, and its bytes, us and us per MB (200 shapes of
// long K, 2 to 16 parts, within 1.4 us in the median).  A ninth part costs the sum another round trip of loads, some 4 us: by itself the plan takes no more than eight.
constexpr float kDenseSplitFixed = 3.5f, kDenseSplitPerMb = 0.6f, kDenseTwoGroupsPerMb = 0.8f;  // that tile's parts leave a value at a time
constexpr int kDensePlannedSplits = 8;
// The same for the tile GEMM's (estimates of npamd_gemv_blocks_preferred).
constexpr float kSplitFixed = 4.5f, kSplitPerMb = 0.45f;

struct DensePlan {
  int tile, splits;
  float us;
};

template <size_t... I>
void count_tiles(int M, int N, int64_t* tiles, std::index_sequence<I...>) {
  ((tiles[I] = (int64_t)((M - 1) / kDenseCost[I].bm + 1) * ((N - 1) / kDenseCost[I].bn + 1)), ...);
}

// The tile and split of least estimate.  64 x 128 in two groups is looked at in parts of one round where y has no fewer rows than columns, K from 4096 on; on wider products it loses as
// many calls as it gains.  Against the tiles of 32x32x16 MFMAs that were here before, behind a decode: of 859 products of 150 to 1700 rows, 256 to 2200 columns and K of 4096 to 14336 55 take
// more than 6 % longer (104 without the tile, 3 with the best of all tiles and parts) at 0.97 of the time in the mean, of 607 of any size up to 60 GFLOP 19 (47) at 0.914.  The wide tiles address their part of the result with 31 bits: with rows of y, or columns, that
// could lie further apart than that, the other kernel's.
//
// Every call of the band is planned, one at a new token count three times: sizes are divided by constants, and the parts of a tile are looked at only while what they cannot go
// below (their bytes, their share of the walk and the sum) is less than the best so far.  us on the host, all tiles and parts in turn / so: 384 x 4096 x 4096
// 0.61 / 0.17, 77 x 3003 x 2176 0.83 / 0.16, 64 x 1024 x 4096 0.87 / 0.32, 528 x 336 x 13440 0.94 / 0.56.
DensePlan plan_dense(int M, int N, int K, int forced_tile, int max_splits, bool wide = true) {
  DensePlan best{0, 1, 1e30f};
  const int steps = K / 64;
  const int forced = tuning().dense_splits, most = max_splits < steps ? max_splits : steps;
  const int forced_splits = forced < most ? forced : most;
  wide = wide && N < kDenseStrideMax;
  const int only = wide && forced_tile > 0 && forced_tile <= kDenseTiles ? forced_tile - 1 : wide ? -1 : 0;
  int64_t tiles[kDenseTiles];
  count_tiles(M, N, tiles, std::make_index_sequence<kDenseTiles>{});
  const bool two_groups = only >= 0 || (M >= N && steps >= 64);
  auto load = [&](int i) { return (float)tiles[i] * steps * (kDenseCost[i].bm + kDenseCost[i].bn) * 128e-6f * kDenseCost[i].per_mb; };
  auto look = [&](int i, int splits, int part, float bytes, float sum) {
    const DenseCost& c = kDenseCost[i];
    const int64_t rounds = ((tiles[i] * splits + 7) / 8 + 31) / 32;
    if (i == kDenseTwoGroups && only < 0 && (splits == 1 || rounds > 1 || !two_groups)) return;
    const float walk = (float)rounds * ((part + c.groups - 1) / c.groups) * c.per_step;
    float t = c.fixed + (float)rounds * c.per_round + sum;
    if (t + fmaxf(walk, bytes) >= best.us) return;
    t += sqrtf(walk * walk + bytes * bytes);
    if (t < best.us) best = {i, splits, t};
  };
  const int first = only < 0 ? 0 : only, last = only < 0 ? kDenseTiles : only + 1;
  if (forced_splits <= 1)
    for (int i = first; i < last; ++i) look(i, 1, steps, load(i), 0.f);
  if (forced_splits == 1 || max_splits < 2) return best;
  const float mb = 4e-6f * M * N;
  auto per_mb = [](int i) { return i == kDenseTwoGroups ? kDenseTwoGroupsPerMb : kDenseSplitPerMb; };
  if (forced_splits > 1) {
    const int part = (steps + forced_splits - 1) / forced_splits;
    for (int i = first; i < last; ++i) look(i, forced_splits, part, load(i), kDenseSplitFixed + per_mb(i) * mb * forced_splits);
    return best;
  }
  const int parts = std::min(std::min(max_splits, kDensePlannedSplits), steps / kDenseMinSplitSteps);
  int part_of[kDensePlannedSplits + 1];
  for (int splits = 2; splits <= parts; ++splits) part_of[splits] = (steps + splits - 1) / splits;
  for (int i = first; i < last; ++i) {
    const DenseCost& c = kDenseCost[i];
    const float bytes = load(i), least = c.fixed + c.per_round + kDenseSplitFixed + fmaxf(bytes, tiles[i] * steps / (256.f * c.groups) * c.per_step);
    for (int splits = 2; splits <= parts && tiles[i] * splits <= 512; ++splits) {
      const float sum = per_mb(i) * mb * splits;
      if (least + sum >= best.us) break;
      look(i, splits, part_of[splits], bytes, kDenseSplitFixed + sum);
    }
  }
  return best;
}

}  // namespace
}  // namespace npamd

using namespace npamd;

extern "C" int64_t npamd_dense_gemm_workspace_bytes(int M, int N, int K) {
  if (M < 1 || N < 1 || K < 64) return 0;
  const DensePlan p = plan_dense(M, N, K, tuning().dense_tile, kDenseMaxSplits);
  return p.splits > 1 ? (int64_t)p.splits * M * N * 4 : 0;
}

static int dense_gemm(const char* what, const void* x, int64_t ldx, const void* w, int64_t ldw, const float* bias, void* y, int64_t ldy,
                      int M, int N, int K, int act_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  NPAMD_REQUIRE(act_dtype == NPAMD_F16 || act_dtype == NPAMD_BF16, "%s: f16 or bf16 only", what);
  NPAMD_REQUIRE(ldx >= K && ldw >= K && ldy >= N && ldx % 8 == 0 && ldw % 8 == 0, "%s: bad row stride", what);
  if (M == 0 || N == 0) return NPAMD_OK;
  NPAMD_REQUIRE(x && w && y && (((uintptr_t)x | (uintptr_t)w) & 15) == 0, "%s: null or unaligned pointer", what);
  NPAMD_REQUIRE(ldx < kDenseStrideMax && ldw < kDenseStrideMax, "%s: row stride too large", what);
  hipStream_t st = (hipStream_t)stream;
  const int64_t room = workspace && ((uintptr_t)workspace & 3) == 0 ? workspace_bytes / ((int64_t)M * N * 4) : 1;
  const int width = (K + 63) / 64 * 64;
  const bool wide = ldy < kDenseStrideMax;
  DensePlan p = plan_dense(M, N, width, tuning().dense_tile, kDenseMaxSplits, wide);
  if (p.splits > room) p = plan_dense(M, N, width, tuning().dense_tile, 1, wide);  // too little workspace: unsplit
  const DenseShape s{x, w, bias, y, ldx, ldw, ldy, M, N, width / 64, 0, 0, p.splits, 0, (float*)workspace, K / 8, 0};
  const int tile = p.tile;
  return act_dtype == NPAMD_BF16 ? launch_dense<NPAMD_BF16>(s, tile, st) : launch_dense<NPAMD_F16>(s, tile, st);
}

extern "C" int npamd_dense_gemm(const void* x, int64_t ldx, const void* w, int64_t ldw, const float* bias, void* y, int64_t ldy,
                                int M, int N, int K, int act_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const char* what = "npamd_dense_gemm";
  NPAMD_REQUIRE(M >= 0 && N >= 0 && K >= 64 && K % 64 == 0, "%s: bad shape M=%d N=%d K=%d (K has to be a multiple of 64)", what, M, N, K);
  return dense_gemm(what, x, ldx, w, ldw, bias, y, ldy, M, N, K, act_dtype, workspace, workspace_bytes, stream);
}

// Rows of x and w that end inside a 64-k step, K a multiple of 8: neither is copied to whole steps first.
extern "C" int npamd_dense_gemm_ragged(const void* x, int64_t ldx, const void* w, int64_t ldw, const float* bias, void* y, int64_t ldy,
                                       int M, int N, int K, int act_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const char* what = "npamd_dense_gemm_ragged";
  NPAMD_REQUIRE(M >= 0 && N >= 0 && K >= 8 && K % 8 == 0, "%s: bad shape M=%d N=%d K=%d (K has to be a multiple of 8)", what, M, N, K);
  return dense_gemm(what, x, ldx, w, ldw, bias, y, ldy, M, N, K, act_dtype, workspace, workspace_bytes, stream);
}

// Whether a call of more than 16 tokens goes to the GEMV with a block per 32 tokens (npamd_*_gemv_blocks), or the table GEMM behind the same
// entry (table_gemm.hip), rather than to decode + product or the tile GEMM.  Up to a round or two of its blocks it is one short launch in the place of two that follow each
// other; past that every block of tokens decodes its weights again.  All three are estimated.  kind: 0 VQ, 1 residual VQ, 4 and 8 bits
// per weight.  Codebooks in memory and residual VQ are estimated as with indices that are all as frequent, and with the tables of four layers in turn.  Of 3015 calls
// near the line, 17 to 4096 tokens, two fifths of them seen by no fit, those that it sends to the slower side lose 0.8 % in the mean of all, 109 of them more than 8 % (the line before this
// one, with corrections by format and range of K on the decode's side: 3.2 %, 416).  us, before / blocks, at 64 and 256 tokens: int4 512 x 512 6.9 / 4.0 and 6.9 / 4.1,
// 1024 x 4096 11.8 / 6.4 and 13.3 / 9.5, 3072 x 3072 14.8 / 8.2; 256 rows 1024 x 1024 7.9 / 4.7 and 8.0 / 5.7, 2048 x 2048 10.4 / 5.7 and 11.1 / 11.2;
// 4096 rows 1024 x 1024 8.1 / 4.7 and 8.1 / 6.6; 65536 rows 512 x 512 7.0 / 4.2 and 7.1 / 4.8, 1024 x 4096 13.2 / 10.0 and 16.5 / 24.8.
namespace npamd {
// What the library's product takes, us (see npamd_dense_gemm_preferred).
static double library_us(int M, int N, int K) {
  const double big_tiles = ceil(M / 256.0) * ceil(N / 256.0);
  const double rate = big_tiles >= 180 ? 1.3 : big_tiles >= 64 ? (K < 4096 ? 1.2 : 1.05) : 0.85;
  return 5.0 + 2e-9 * M * N * K / rate + fmax(0.0, (K - 4096) / 1024.0) * 1.5;
}

// The blocks entry, us.  Of int4 / int8, of residual VQ and of tables that LDS does not hold: a start, what a round of the blocks that LDS holds at a time takes, and what its waves do, the
// longest of them one step behind the other and all of a compute unit's together.  As their launchers choose them (launch_q_gemv; launch_fused_gemv with one
// staged row tile); fitted to 1758 calls near the line, each format and table apart, K of 128 to 14336: within 4 to 6 % in the median of 725 others, 12 % in nine of ten.
float gemv_blocks_us(int kind, int table_rows, int M, int N, int K) {
  constexpr int cus = 256;
  const int tokens = (M + kGemvTokens - 1) / kGemvTokens, rows = (N + 15) / 16, tiles = rows * tokens;
  const int steps = (K + 255) / 256, chunks = (K + 63) / 64, load = (tiles + cus - 1) / cus;
  auto per = [](int a, int b) { return (a + b - 1) / b; };
  if (kind >= 4) {
    const int item = 512 * kind + 256, load2 = per((rows + 1) / 2 * tokens, cus), four = std::min(steps, 4);  // LDS of a row tile's step; of pairs of row tiles
    auto held = [&](int waves, int R) { return std::max(1, kGemvLdsPerBlockMax / (waves * (16384 + R * item))); };
    bool two = steps >= 8 && load > 1 && 16 * load2 <= 9 * load;
    if (tokens > 1) {
      const int rounds1 = per(load, held(four, 1)), rounds2 = per(load2, held(four, 2));
      two = rounds2 < rounds1 || (two && rounds2 == rounds1);
    }
    const int R = two ? 2 : 1, blocks = two ? load2 : load;
    const int spw = per(steps, !two && load <= 1 && 8 * (16384 + item) <= kGemvLdsPerBlockMax ? 8 : 4), waves = per(steps, spw);
    const int rounds = per(blocks, held(waves, R));
    if (kind == 4) return 2.63f + 1.11f * rounds + 0.081f * blocks * R + hypotf(0.296f * spw * rounds, 0.212f * blocks * R * steps);
    return 2.12f + 2.01f * rounds + hypotf(0.563f * spw * rounds, 0.205f * blocks * R * steps);
  }
  const int table = table_rows * 16;
  if (kind == 0 && table <= kGemvLdsCodebookMax) {
    if (gemv_wide_looks_up_in_memory(M, tiles, chunks, table)) {
      const float lookups = 2.0f * K, served = table_rows <= 2048 ? 1100e3f : 275e3f;  // of a block; by the L1s, by the L2s
      return 3.3f + load * lookups / 2400.f + tiles * lookups / served;
    }
    const int R = gemv_wide_row_tiles(M, tiles, table);
    const int waves = R < 4 && table > 32 * 1024 ? 6 : 8, spw = per(steps, waves), rounds = per(per(rows, R) * tokens, cus);
    return 1.8f + rounds * (R == 1 ? 1.4f + 2.1f * spw : R == 2 ? 2.7f + 2.0f * spw : 8.5f + 3.0f * spw);
  }
  // Lookups in memory.
  int spw = std::max(per((kind == 1 ? rows : tiles) * steps, 16 * cus), per(steps, 8)), waves = 0, lds = 0;
  for (;; ++spw) {
    waves = per(steps, spw);
    const int sums = waves * std::min(M, kGemvTokens) * 64;
    lds = (kind == 1 ? std::max(sums, 4096) : sums) + waves * 2 * GemvStage<1>::kBytes;
    if (lds <= kGemvLdsPerBlockMax) break;
  }
  const int rounds = per(load, std::max(1, std::min(kGemvLdsPerBlockMax / lds, 32 / waves)));
  // Tables by who serves them: the L1s (up to 2048 rows, the main table of residual layers), an L2 next to the weights, an L2 that other layers' tables share.
  struct { float start, round, step, lookups, block; } c =
      kind == 0 ? table_rows <= 16384 ? decltype(c){2.50f, 0.59f, 0.619f, 0.444f, 0.144f} : decltype(c){3.26f, 0.33f, 0.803f, 0.471f, 0.150f}
                : table_rows <= 2048    ? decltype(c){2.14f, 1.86f, 0.681f, 0.306f, 0.182f}
                  : table_rows <= 8192  ? decltype(c){2.47f, 1.46f, 0.476f, 0.395f, 0.191f}
                  : table_rows <= 16384 ? decltype(c){2.24f, 1.52f, 0.f, 0.586f, 0.265f}
                                        : decltype(c){3.72f, 1.44f, 0.515f, 0.535f, 0.115f};
  return c.start + (c.round + c.step * spw) * rounds + c.lookups * load * K / 256 + c.block * load;
}
}  // namespace npamd

extern "C" int npamd_gemv_blocks_preferred(int M, int N, int K, int kind, int table_rows, int gathered, int tile) {
  if (M <= 16 || N < 1 || K < 64 || K % 64) return 0;
  const float gather = gathered ? 3.0f + M * (float)K * 4 / 4.4e6f : 0.f;
  float blocks = gemv_blocks_us(kind, table_rows, M, N, K);
  const bool in_lds = kind == 0 && table_rows <= 4096;
  if (in_lds && table_rows > 16) blocks = fminf(blocks, plan_table_gemm(M, N, K, table_rows).us);  // up to 16 rows: indices of 4 bits
  // Near the line the blocks' figures are 3 % high at fewer tokens (2483 calls of 17 to 1024 tokens: 0.70 % lost in the mean so, with 1 0.81, with 1.03 1.04), and not past 512.
  // Residual layers with large main tables: between indices that are all as frequent and Zipf's, whose lookups the blocks gain more from (mean loss, uniform / Zipf, 317 calls: 0.94 0.7 / 1.0 %, 0.97 0.5 / 1.7).
  blocks = (kind == 1 && table_rows > 8192 ? 0.94f : M > 512 ? 1.f : 0.97f) * (blocks + gather);
  // The decode, us: what it takes by itself and per million weights, behind it the product, and what K in parts takes there past the plan's figure (or less).  Fitted to the same calls
  // as the blocks' figures, 0.1 to 45 million weights: within 3 to 5 % in the median, 10 % in nine of ten.
  const float weights = 1e-6f * N * K;
  const float decode = kind == 4 ? 2.4f + 0.26f * weights
                     : kind == 8 ? 2.45f + 0.33f * weights
                     : kind == 1 ? 2.8f + (table_rows <= 4096 ? 0.77f : 1.0f) * weights
                                 : in_lds ? 2.1f + 0.0002f * table_rows + 0.30f * weights
                                 : 2.2f + (table_rows <= 16384 ? 0.69f : 0.93f) * weights;
  const float in_parts = kind == 4 ? 0.7f : in_lds ? 0.9f : kind == 0 && table_rows <= 16384 ? 0.f : kind == 8 ? -0.1f : -0.6f;
  // The library's rate here is what it reaches, 1.25 PFLOP/s from 100 of its tiles on; below, with less of a risk in the other direction.
  const bool own = npamd_dense_gemm_preferred(M, N, K), many = ceil(M / 256.0) * ceil(N / 256.0) >= 100;
  const float library = many ? 5.f + 2e-9f * M * N * K / 1.25f : (float)library_us(M, N, K);
  const DensePlan p = plan_dense(M, N, K, 0, kDenseMaxSplits);
  const float host = own ? (p.splits > 1 ? 10.3f : 7.0f) : 33.f;  // of two or three launches
  const float product = fmaxf(host, decode + (own ? p.us + (p.splits > 1 ? in_parts : 0.f) : library));
  if (blocks >= product) return 0;
  if (!tile || (in_lds && M > 256)) return 1;  // past 256 tokens such layers have no tile GEMM
  const int columns = (N + 63) / 64 * ((M + 383) / 384), chunks = K / 64;
  int splits = columns * 10 < 256 * 7 ? 256 / columns : 1;
  splits = splits > chunks / 8 ? chunks / 8 : splits;
  splits = splits > 16 ? 16 : splits < 1 ? 1 : splits;
  if (in_lds) {
    // us of a step at 64 / 128 / 192 / 256 tokens: 0.23, 0.27, 0.45, 0.53, with 4096 rows a fifth more
    const int rounds = (columns * splits + 255) / 256;
    const float step = (M <= 128 ? 0.19f + 0.0006f * M : 0.30f + 0.0009f * M) * (1.f + 0.2f * table_rows / 4096);
    const float us = gather + 3.3f + rounds * step * ((chunks + splits - 1) / splits) + (splits > 1 ? kSplitFixed + kSplitPerMb * (4e-6f * splits * M * N) : 0.f);
    return blocks < us ? 1 : 0;
  }
  const float us = gather + (kind >= 4 ? 1.05f : 1.15f) * (7.8f + 0.25f * chunks / splits + (splits > 1 ? 2.5f : 0.f));
  return blocks < us ? 1 : 0;
}

// Where this product is the better one against the library's.  That takes 18.3-19 us per eager call whatever its size and 33 us go by between two calls of
// decode + library product, whatever the GPU does meanwhile: below 64 GFLOP this one.  Past that the library's kernels are ahead where its tiles of 256 x 256, those at the edges
// counted whole, fill their rounds of all compute units, the more of a product the less they have to.  Of 3728 products of 10 to 5000 GFLOP, K from 64 to 28672, fp16 and bf16, this one's time over the library's
// (median, quarters): rounds at least 0.98 full, 64 to 300 GFLOP 1.05 (1.03 to 1.06), to 1600 1.08, past that 1.13; 0.9 to 0.98 full, to 300 GFLOP 0.97 (0.87 to 1.04), to
// 800 1.03 (0.92 to 1.08), to 1600 1.05, past that 1.08; 0.86 to 0.9 full, past 1600 GFLOP 1.11; less full 0.87 to 0.97 (the library is 10 % and more ahead on one in twenty of those, by
// no size that tells which: 1024 x 9728 x 14336 239 / 299 us, 1024 x 13824 x 13824 479 / 327).  Rounds of exactly seven eighths are level up to 14336 columns and the library's by 7 % past them, unlike their
// neighbours (4096 x 14336 x 4096 a thousand in a row bf16 329 / 341, fp16 346 / 359, three after a pause 343 to 351 / 347 to 354;
// 2048 x 14336 x 4096 170 / 174, 179 / 182 and 178 / 178; 4096 x 11008 x 4096, 0.896 full, 405 / 262); there is no difference between the types.  Where K is short (512 to 768: 0.81 up to
// 64 GFLOP, 1.05 up to 300) or N no multiple of 8 (0.95 up to 300 GFLOP) the line is at 300.  Library / this, us: 4095 x 4096 x 4096 bf16 92.7 / 97.9, 8000 x 4096 x 14336 590 / 695,
// 2842 x 64000 x 4992 1265 / 1652, 5000 x 128256 x 2048 1957 / 2282; 4096 x 6144 x 4096 174.5 / 177.6 and bf16 166.3 / 157.8, 1646 x 13120 x 11136 690 / 444.
extern "C" int npamd_dense_gemm_preferred(int M, int N, int K) {
  if (M < 1 || N < 1 || K < 64 || K % 64 || K >= kDenseStrideMax) return 0;
  const int forced = tuning().dense_tile;
  if (forced) return forced > 0;
  if (N >= kDenseStrideMax) return 0;  // the wide tiles do not take it
  const double gflop = 2e-9 * M * N * K;
  const int64_t tiles = (((int64_t)M + 255) / 256) * ((N + 255) / 256), rounds = (tiles + 255) / 256;
  const double full = tiles / (256.0 * rounds);
  const bool whole = full >= 0.98 || 8 * tiles == 7 * 256 * rounds;
  if (gflop < 300) return gflop >= 64 && K >= 768 && N % 8 == 0 && whole ? 0 : 1;
  return whole || (gflop >= 800 && full >= 0.9) || (gflop >= 1600 && full >= 0.86) ? 0 : 1;
}
