// Dense product on wide tiles: y = x @ W^T (+ bias), f32 accumulate.  wide_gemm.hip has the tiles, dense_gemm.hip what chooses them.
//
// A wave computes 16 MT x 16 NT of the block's tile (MFMA 16x16x32), at most 128 x 64 or 64 x 112: an operand then serves four to eight MFMAs, where waves of
// 64 x 64 keep LDS as busy as the matrix pipes.  x and W come straight into LDS, rows of 128 bytes, a ring of steps of 64 k; half a step's operands are
// read between the MFMAs of the half before, and a step's place is loaded again as soon as its second half is in registers: one barrier a step.
// What bounds it, at 4096 x 14336 x 4096 (bf16, tiles of 256 x 224): the matrix pipes, busy 78 % of all cycles, and the power they draw, which holds the clock at
// 1.7 to 2.0 GHz; 6 us of each round of tiles are its start and its end, half of that the result on its way to memory.  The time goes with the clock: 341 us (1.41 PFLOP/s) each
// of a thousand in a row, 347 to 354 for three after a pause, 398 to 407 for thirty, the library's product 329, 343 to 351 and 390.
// What counted, us of that product in one process (the kernel before, 256 x 128 on MFMAs of 32x32x16, 422 there, this one 332): loads right behind the barrier into the place just read, instead of in front of the next one 415 -> 370; spread over 24 of
// the 64 MFMAs of a step, not one behind each 371 -> 363; 16x16x32 instead of 32x32x16, in as many cycles but less power 388 -> 352; a
// tile width that fills the last round (256 x 224 for 256 x 256) 352 -> 337.  Tried without gain: four waves of 128 x 128 (one per SIMD: 354), steps of 32 k in
// four or five places (half lines: 387), a block per compute unit that walks several tiles (358: its stores and the next tile's loads wait
// for each other in one counter).
#pragma once

#include <type_traits>

#include "dense_gemm.hpp"
#include "gemm_tile.hpp"
#include "lds_transfer.hpp"

namespace npamd {

// Lambdas over a kernel's registers: called several times, the compiler would leave them out of line and the registers in memory.
#define NPAMD_INLINE __attribute__((always_inline))

// WGM x WGN waves of 16 MT x 16 NT, a ring of ST steps of 64 k; the loads of a step go out behind the SPAN MFMAs of a wave
// that follow the step's barrier.
template <int WGM_, int WGN_, int MT_, int NT_, int ST_, int SPAN_>
struct WideTile {
  static constexpr int WGM = WGM_, WGN = WGN_, MT = MT_, NT = NT_, ST = ST_, SPAN = SPAN_;
  static constexpr int kBM = 16 * MT * WGM, kBN = 16 * NT * WGN;
  static constexpr int kWaves = WGM * WGN, kThreads = 64 * kWaves;
  static constexpr int kPiecesX = kBM / 8, kPieces = (kBM + kBN) / 8;  // a load's worth of rows
  static constexpr int kLoads = (kPieces + kWaves - 1) / kWaves;       // per wave and step
  static constexpr int kStageBytes = (kBM + kBN) * 128;
  static constexpr int kEpRow = 32 * NT + 16;  // bytes of a row of a wave's tile on its way out
  static constexpr int kEpBytes = 16 * MT * kEpRow;
  static constexpr int kLds = ST * kStageBytes > kWaves * kEpBytes ? ST * kStageBytes : kWaves * kEpBytes;
  static constexpr int kMfmas = MT * NT;  // of a wave and half a step
  static_assert(kLds <= kLdsPerBlockMax && SPAN <= 2 * kMfmas && (ST - 1) * kLoads < 64);
};

template <int ACT, class T>
__global__ void __launch_bounds__(T::kThreads, T::kThreads == 256 ? 2 : 1)
wide_gemm_kernel(const DenseShape s) {
  constexpr int MT = T::MT, NT = T::NT, ST = T::ST, L = T::kLoads, kM = T::kMfmas, SPAN = T::SPAN;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // blockIdx.x % 8 names the die; a die takes an eighth of the units, counted down the columns of a group of row tiles (launch_wide_tile).
  const int unit = (blockIdx.x & 7) * s.units_per_die + (blockIdx.x >> 3), columns = s.col_tiles * s.splits;
  if (unit >= s.row_tiles * columns) return;
  const int group = unit / (s.group * columns), in = unit - group * (s.group * columns), group_rows = min(s.group, s.row_tiles - group * s.group);
  const int column = in / group_rows, rt = group * s.group + in - column * group_rows;
  const int ct = s.splits > 1 ? column / s.splits : column, part = column - ct * s.splits;
  const int m0 = rt * T::kBM, n0 = ct * T::kBN;
  const int step0 = (int)((int64_t)s.steps * part / s.splits);
  const int steps = (int)((int64_t)s.steps * (part + 1) / s.splits) - step0;  // of this part

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % T::WGM, wn = wave / T::WGM;
  const int c = lane & 15, h = lane >> 4;

  // The rows of 8 that load i brings: L neighbours a wave, so that most waves load only x or only W.  Past the last, it or the one before again.
  auto piece_of = [&](int i) NPAMD_INLINE { return min(wave * L + i, T::kPieces - 2 + ((wave * L + i) & 1)); };
  // Piece p of row r lies in place p ^ ((r >> 1) & 7): a lane's differs between even and odd i only.
  auto piece_in_row = [&](int i) NPAMD_INLINE { return (lane & 7) ^ ((((wave * L + i) & 1) * 4 + (lane >> 4)) & 7); };
  uint32_t voff[L];
  const uint8_t* from[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int q = piece_of(i);
    const bool is_x = q < T::kPiecesX;
    const int r = (is_x ? q : q - T::kPiecesX) * 8 + (lane >> 3);
    const int row = is_x ? min(r, s.M - 1 - m0) : min(r, s.N - 1 - n0);  // rows past the end: a valid row nobody stores
    voff[i] = (uint32_t)((int64_t)row * (is_x ? s.ldx : s.ldw) * 2) + (uint32_t)(piece_in_row(i) * 16);
    from[i] = uniform_ptr(is_x ? reinterpret_cast<const uint8_t*>(s.x) + ((int64_t)m0 * s.ldx + (int64_t)step0 * 64) * 2
                               : reinterpret_cast<const uint8_t*>(s.w) + ((int64_t)n0 * s.ldw + (int64_t)step0 * 64) * 2);
  }
  const uint32_t ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  auto load = [&](int i, int slot, int step) NPAMD_INLINE {
    lds_load16(ring + (uint32_t)(slot * T::kStageBytes + piece_of(i) * 1024), voff[i], from[i] + (int64_t)step * 128);
  };
  // Rows that end inside the last step: its loads bring the last piece again for those past the end, and the operands there are zeroed.
  const int there = s.pieces - (step0 + steps - 1) * 8;  // pieces of this part's last step
  auto end_rows = [&](int first, int last) NPAMD_INLINE {
#pragma unroll
    for (int i = 0; i < L; ++i)
      if (i >= first && i < last) voff[i] -= (uint32_t)(max(piece_in_row(i) - (there - 1), 0) * 16);
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 xo[2][MT], wo[2][NT];
  const uint32_t x_off = (uint32_t)((wm * 16 * MT + c) * 128), w_off = (uint32_t)((T::kBM + wn * 16 * NT + c) * 128);
  const uint32_t place[2] = {(uint32_t)((h ^ ((c >> 1) & 7)) << 4), (uint32_t)(((4 | h) ^ ((c >> 1) & 7)) << 4)};
  auto read_one = [&](int j, const uint8_t* stage, int i) NPAMD_INLINE {
    if (i < NT) wo[j][i] = *reinterpret_cast<const u32x4*>(stage + w_off + i * 2048 + place[j]);
    else xo[j][i - NT] = *reinterpret_cast<const u32x4*>(stage + x_off + (i - NT) * 2048 + place[j]);
  };
  auto blank = [&](int j) NPAMD_INLINE {
    const bool dead = 4 * j + h >= there;
#pragma unroll
    for (int b = 0; b < NT; ++b) wo[j][b] = dead ? u32x4{0, 0, 0, 0} : wo[j][b];
#pragma unroll
    for (int a = 0; a < MT; ++a) xo[j][a] = dead ? u32x4{0, 0, 0, 0} : xo[j][a];
  };
  // The wave's own pieces of a step have arrived when only those of `young` younger steps are still on their way.
  auto wait_young = [&](int young) NPAMD_INLINE {
    if (young >= 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * L < 63 ? 3 * L : 63) : "memory");
    else if (young == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory");
    else if (young == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  int slot = 0;
  // One step of two halves; between the MFMAs of a half the reads of the next half's operands.  At the middle the next step has arrived,
  // and nobody reads this one's place any more: the loads of step it + ST take it, the first of them behind the MFMAs of this step's second half, the others
  // behind those of the next step's first half.  MODE 2: all of that; 1: nothing is left to load but the others of step it + ST - 1; 0: nothing at all.
  auto step = [&](auto mode, int it) NPAMD_INLINE {
    constexpr int MODE = decltype(mode)::value;
    constexpr int kReads = MT + NT, kReadSpots = kM * 3 / 4;
    const uint8_t* const stage = lds + slot * T::kStageBytes;
    const int behind = slot == ST - 1 ? 0 : slot + 1, before = slot == 0 ? ST - 1 : slot - 1;
    const uint8_t* const next = lds + behind * T::kStageBytes;
    const bool ends = MODE == 0 && it == steps - 1 && there < 8;
    if (ends) blank(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (j == 1) {
        if constexpr (MODE == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * L) : "memory");
        else wait_young(steps - 2 - it);
        block_sync_lds();
        __builtin_amdgcn_sched_barrier(0);
        if (ends) blank(1);
      }
#pragma unroll
      for (int q = 0; q < kM; ++q) {
        acc[q / NT][q % NT] = mfma16<ACT>(wo[j][q % NT], xo[j][q / NT], acc[q / NT][q % NT]);
        if (q < kReadSpots) {
#pragma unroll
          for (int i = q * kReads / kReadSpots; i < (q + 1) * kReads / kReadSpots; ++i) read_one(j ^ 1, j ? next : stage, i);
        }
        const int at = j ? q : kM + q;
        if (at < SPAN && (j ? MODE == 2 : MODE >= 1)) {
#pragma unroll
          for (int i = at * L / SPAN; i < (at + 1) * L / SPAN; ++i) load(i, j ? slot : before, j ? it + ST : it + ST - 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    slot = behind;
  };
  constexpr int kFirstLoads = SPAN <= kM ? L : kM * L / SPAN;  // of a step, behind its barrier

#pragma unroll
  for (int p = 0; p < ST; ++p) {
    if (p < steps) {
      const int loads = p < ST - 1 ? L : kFirstLoads;
      if (p == steps - 1 && there < 8) end_rows(0, loads);
#pragma unroll
      for (int i = 0; i < loads; ++i) load(i, p, p);
    }
  }
  if (steps >= ST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * L + kFirstLoads) : "memory");
  else wait_young(steps - 1);
  block_sync_lds();
#pragma unroll
  for (int i = 0; i < MT + NT; ++i) read_one(0, lds, i);
  int it = 0;
  for (const int ragged = there < 8 ? steps - 1 - ST : -1; it < steps - ST; ++it) {
    if (it == ragged) end_rows(0, kFirstLoads);
    step(std::integral_constant<int, 2>{}, it);
  }
  if (SPAN > kM && it == steps - ST) {
    if (there < 8) end_rows(kFirstLoads, L);
    step(std::integral_constant<int, 1>{}, it);
    ++it;
  }
  for (; it < steps; ++it) step(std::integral_constant<int, 0>{}, it);

  // What lies outside the result is stored past the end of the buffer, which the hardware drops: no branches.
  constexpr uint32_t kBuffer = 0x80000000u, kNowhere = kBuffer;  // bytes
  constexpr int kRaw = 0x00020000;                               // of a buffer descriptor: bytes as they lie
  const int wm0 = m0 + wm * 16 * MT, wn0 = n0 + wn * 16 * NT, rows = s.M - wm0, cols = s.N - wn0;  // of the wave's tile
  // A lane has the columns 16 b + 4 h .. + 3 of row 16 a + c.
  if (s.splits > 1) {
    float* const to = s.partials + ((int64_t)part * s.M + wm0) * s.N + wn0;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(to, 0, (int)kBuffer, kRaw);
    const bool whole = s.N % 4 == 0 && (reinterpret_cast<uintptr_t>(s.partials) & 15) == 0;
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        const int m = 16 * a + c, n = 16 * b + 4 * h;
        const uint32_t off = (uint32_t)(m * s.N + n) * 4u;
        if (whole) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[a][b]), rsrc, m < rows && n < cols ? off : kNowhere, 0, 0);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = acc[a][b][e];  // a copy: the cast of an element itself takes the first one's bits
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc, m < rows && n + e < cols ? off + 4u * e : kNowhere, 0, 0);
          }
        }
      }
    return;
  }
  // Through LDS, each wave in a part of its own: rows of 16 NT columns then leave whole.
  uint8_t* const ep = lds + wave * T::kEpBytes;
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    f32x4 bv{0.f, 0.f, 0.f, 0.f};
    if (s.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[e] = s.bias[min(wn0 + 16 * b + 4 * h + e, s.N - 1)];
    }
#pragma unroll
    for (int a = 0; a < MT; ++a) {
      uint32_t bits[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = acc[a][b][e] + bv[e];
        bits[e] = ACT == NPAMD_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
      }
      *reinterpret_cast<u32x2*>(ep + (16 * a + c) * T::kEpRow + 32 * b + 8 * h) = u32x2{bits[0] | (bits[1] << 16), bits[2] | (bits[3] << 16)};
    }
  }
  uint16_t* const to = reinterpret_cast<uint16_t*>(s.y) + (int64_t)wm0 * s.ldy + wn0;
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(to, 0, (int)kBuffer, kRaw);
  const uint32_t ldy = (uint32_t)s.ldy;
  if (s.ldy % 8 == 0 && s.N % 8 == 0 && (reinterpret_cast<uintptr_t>(s.y) & 15) == 0) {
    constexpr int kPerRow = 2 * NT, kRowsAtOnce = 64 / kPerRow;  // 16-byte pieces; NT = 3, 7: a few lanes idle
    const int r = lane / kPerRow, p = lane % kPerRow;
#pragma unroll 8
    for (int i = 0; i < (16 * MT + kRowsAtOnce - 1) / kRowsAtOnce; ++i) {
      const int m = i * kRowsAtOnce + r;
      const u32x4 v = *reinterpret_cast<const u32x4*>(ep + min(m, 16 * MT - 1) * T::kEpRow + p * 16);
      const bool in = r < kRowsAtOnce && m < min(rows, 16 * MT) && p * 8 < cols;
      __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, in ? ((uint32_t)m * ldy + (uint32_t)p * 8u) * 2u : kNowhere, 0, 0);
    }
    return;
  }
  // Rows at odd addresses: a value at a time, a row's side by side.
#pragma unroll 8
  for (int m = 0; m < 16 * MT; ++m) {
#pragma unroll
    for (int n0 = 0; n0 < 16 * NT; n0 += 64) {
      const int n = n0 + lane;
      const uint16_t v = *reinterpret_cast<const uint16_t*>(ep + m * T::kEpRow + min(n, 16 * NT - 1) * 2);
      __builtin_amdgcn_raw_buffer_store_b16(v, rsrc, m < rows && n < 16 * NT && n < cols ? ((uint32_t)m * ldy + (uint32_t)n) * 2u : kNowhere, 0, 0);
    }
  }
}

template <int ACT, class T>
int launch_wide_tile(DenseShape s, hipStream_t st) {
  s.row_tiles = (s.M + T::kBM - 1) / T::kBM;
  s.col_tiles = (s.N + T::kBN - 1) / T::kBN;
  const int64_t units = (int64_t)s.col_tiles * s.row_tiles * s.splits, blocks = (units + 7) / 8 * 8;
  if (blocks > 0x7FFFFFFF) return fail(NPAMD_ERR_UNSUPPORTED, "npamd_dense_gemm: too many tiles");
  s.units_per_die = (int)(blocks / 8);
  // Units are counted down the columns of 2048 rows, so that the rows of W that a die's decode wrote (see die_block) are read through its L2 and, past
  // 2048 rows, x does not come into the L2s again for every column tile; where x is the longer side, down four row tiles, as then it is what each die would
  // bring whole.  Decode + product of int4 layers with groups of 4 tiles / of 2048 rows, us: 656 x 1452 x 4608 27.2 / 22.7, 304 x 3690 x 2048 22.9 / 18.1, 1104 x 2714
  // x 1024 19.2 / 15.3; 1440 x 970 x 8832 53.4 / 59.2, 1956 x 1532 x 11008 102.2 / 108.5, 3575 x 703 x 1536 17.3 / 20.3.
  s.group = s.M > 1.2f * s.N ? 4 : 2048 / T::kBM;
  static LdsLatch latch;
  const auto kernel = wide_gemm_kernel<ACT, T>;
  const hipError_t e = enable_dynamic_lds(latch, reinterpret_cast<const void*>(kernel), T::kLds);
  if (e != hipSuccess) return fail(NPAMD_ERR_LAUNCH, "npamd_dense_gemm: cannot reserve %d bytes of LDS: %s", T::kLds, hipGetErrorString(e));
  launch(kernel, (unsigned)blocks, T::kThreads, T::kLds, st, s);
  return check_launch("npamd_dense_gemm");
}

}  // namespace npamd
