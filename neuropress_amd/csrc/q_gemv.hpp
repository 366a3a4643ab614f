// Fused GEMV of the group-affine formats (int4, int8) for up to 32 tokens, wave64 + MFMA 16x16x32.
//
// Operands and arithmetic are those of fused_gemv_kernel (gemv.hpp): D[16 x 16] += x[16 x 32] * W^T[32 x 16], weights
// dequantized and rounded to the activation type.  What differs is how the bytes come in.  An operand's 16 lanes are 16 rows of
// the weight, and a load that puts each lane's bytes into its own registers touches a cache line per lane: 64 cycles of the
// compute unit's address path for a KiB, scales as many again (14336 x 4096 int4: 6 us of 15).  Here a wave asks
// for whole lines, straight into an LDS area of its own (global_load_lds, 128 or 256 bytes of a row side by side, 16 cycles per
// KiB), and reads operands and scales from there; so do the activations, of which only the tokens there are are loaded.
// Bytes are moved to registers in one go and their place is requested again for the step after at once, so a wave has a step
// of 256 k of all its row tiles on the way while it decodes the one before; nothing is shared between waves and nothing
// waits at a barrier.  A block owns 16 R rows and all of K; its waves split the steps and their partial tiles are summed through LDS.
// Before (fused_gemv_kernel) / now, us at 1 / 8 / 16 / 32 tokens: 14336 x 4096 int4 bf16 with zero points 17.4 / 18.0 / 19.9 / 27.8 and
// 13.8 / 15.0 / 16.6 / 23.9, int8 bf16 22.4 / 21.7 / 22.7 / 31.3 and 15.7 / 16.6 / 17.8 / 24.7 (3.8 TB/s at one token); 4096 x 14336
// int4 fp16 15.3 / 16.6 / 19.0 / 25.3 and 10.1 / 12.6 / 15.7 / 21.3; 8944 x 2176 int8 13.9 / 14.9 / 16.7 / 22.7 and 8.2 / 9.1 / 10.4 / 14.5.
// What is left at many tokens is the vector instructions (decode) and LDS (codes in and out, activations per row tile).
// Requesting four items ahead without whole lines changed nothing (14.6 against 14.4 us); neither did sixteen waves.
#pragma once

#include "gemv.hpp"
#include "lds_transfer.hpp"

namespace npamd {

template <int N>
__device__ __forceinline__ void q_gemv_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS of one wave: the activations of a step, two tokens per KiB (16-byte piece p of token m in slot p ^ (m & 15) of its 512
// bytes, so that 16 tokens' reads of a piece fall into 16 bank groups), then per row tile its codes (16 rows, piece p of row
// r in slot p ^ (r >> 1) of eight or p ^ r of sixteen) and its scales and zero points (a dword per row and chunk).
template <int NBITS, bool ASYM, int R, int XI>
struct QGemvLds {
  static constexpr int kRow = 32 * NBITS;  // bytes of a row in a step
  static constexpr int kCodes = 16 * kRow;
  static constexpr int kItem = kCodes + (ASYM ? 512 : 256);
  static constexpr int kLoads = kCodes / 1024 + (ASYM ? 2 : 1);  // load instructions of an item
  static constexpr int kWave = XI * 1024 + R * kItem;
  static constexpr int kMaxWaves = kGemvLdsPerBlockMax / kWave < 8 ? kGemvLdsPerBlockMax / kWave : 8;
};

// The 32 tokens of a block, one behind the other along y; up to 16 are one block.
template <int MT>
__device__ __forceinline__ GemvShape q_gemv_tokens(GemvShape s) {
  if constexpr (MT == 1) return s;
  const int m0 = blockIdx.y * kGemvTokens;
  s.M = min(s.M - m0, kGemvTokens);
  s.x = reinterpret_cast<const uint16_t*>(s.x) + (int64_t)m0 * s.ldx;
  s.y = reinterpret_cast<uint16_t*>(s.y) + (int64_t)m0 * s.ldy;
  return s;
}

// XI: load instructions for a step's activations: up to 2 XI tokens.
template <int ACT, int NBITS, bool ASYM, class Provider, int R, int XI>
__global__ void __launch_bounds__(512)
q_gemv_kernel(const GemvShape all, const typename Provider::Args a) {
  constexpr int MT = XI > 8 ? 2 : 1;
  const GemvShape s = q_gemv_tokens<MT>(all);
  using L = QGemvLds<NBITS, ASYM, R, XI>;
  constexpr int kSlots = L::kRow / 16, kRowsPerLoad = 64 / kSlots, kCodeLoads = L::kCodes / 1024;
  extern __shared__ __attribute__((aligned(16))) uint8_t q_lds[];
  const Provider prov(a);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_waves = blockDim.x >> 6;
  const int c = lane & 15, q = lane >> 4;
  const int row0 = blockIdx.x * (16 * R);
  const int step_begin = wave * s.steps_per_wave;
  const int step_end = min(step_begin + s.steps_per_wave, s.steps);

  f32x4 acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (step_begin < step_end) {
    uint8_t* const mine = q_lds + wave * L::kWave;
    const uint32_t mine_lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)mine;
    const uint8_t* const wbase = a.w_pack + (int64_t)row0 * s.chunks * (NBITS * 8);
    const int64_t scale0 = (int64_t)row0 * a.groups_per_row;  // row0 is a multiple of 16: whole dwords
    const int last_row = s.N - 1 - row0;  // rows past the end: a valid row nobody stores
    uint32_t xoff[XI], woff[R][kCodeLoads], srow[R];
    int wpiece[kCodeLoads];
    const int xpiece = lane & 31;
#pragma unroll
    for (int i = 0; i < XI; ++i) xoff[i] = (uint32_t)(min(2 * i + (lane >> 5), s.M - 1) * s.ldx * 2);
#pragma unroll
    for (int t = 0; t < kCodeLoads; ++t) {
      const int row = t * kRowsPerLoad + lane / kSlots;
      wpiece[t] = (lane % kSlots) ^ (kSlots == 8 ? (row >> 1) & 7 : row);
#pragma unroll
      for (int r = 0; r < R; ++r) woff[r][t] = (uint32_t)min(16 * r + row, last_row) * (uint32_t)(s.chunks * NBITS * 8);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) srow[r] = (uint32_t)min(16 * r + (lane >> 2), last_row) * (uint32_t)a.groups_per_row;
    auto load_x = [&](int step) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        const int p = step * 32 + (xpiece ^ ((2 * i + (lane >> 5)) & 15));  // 16-byte piece of the row
        lds_load16(mine_lds + (uint32_t)(i * 1024), xoff[i] + (uint32_t)(min(p, s.chunks * 8 - 1) * 16), s.x);
      }
    };
    auto load_item = [&](int r, int step) {
      const uint32_t dst = mine_lds + (uint32_t)(XI * 1024 + r * L::kItem);
#pragma unroll
      for (int t = 0; t < kCodeLoads; ++t) {
        const int kc = min(step * 4 + wpiece[t] / (kSlots / 4), s.chunks - 1);
        lds_load16(dst + (uint32_t)(t * 1024),
                      woff[r][t] + (uint32_t)(kc * (NBITS * 8) + wpiece[t] % (kSlots / 4) * 16), wbase);
      }
      const int kc = min(step * 4 + (lane & 3), s.chunks - 1);
      const uint32_t at = ((srow[r] + (uint32_t)((2 * kc) >> a.gs_shift_chunks)) * 2u) & ~3u;
      lds_load4(dst + (uint32_t)L::kCodes, at, a.scale + scale0);
      if constexpr (ASYM) lds_load4(dst + (uint32_t)(L::kCodes + 256), at, a.zp + scale0);
    };

    load_x(step_begin);
#pragma unroll
    for (int r = 0; r < R; ++r) load_item(r, step_begin);

    auto one_step = [&](auto last_, int step) {
      constexpr bool LAST = decltype(last_)::value;
      const bool ragged = (step + 1) * 4 > s.chunks;       // uniform
      const bool dead = step * 4 + q >= s.chunks;  // a k slot past K: exactly zero, whatever its scale and activations
      q_gemv_wait<R * L::kLoads>();
      u32x4 xa[MT][8];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = min(16 * t + c, s.M - 1);  // rows of D past M: a token nobody stores again
#pragma unroll
        for (int j = 0; j < 8; ++j) xa[t][j] = *reinterpret_cast<const u32x4*>(mine + m * 512 + (((q * 8 + j) ^ (m & 15)) << 4));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (!LAST) load_x(step + 1);
      if (ragged) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int j = 0; j < 8; ++j) xa[t][j] = dead ? u32x4{0u, 0u, 0u, 0u} : xa[t][j];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        // younger: the other items of this step that are still to come, or their successors, and the activations
        if constexpr (LAST) {
          if (r == R - 1) q_gemv_wait<0>();
          else if (r == R - 2) q_gemv_wait<L::kLoads>();
          else if (r == R - 3) q_gemv_wait<2 * L::kLoads>();
          else q_gemv_wait<3 * L::kLoads>();
        } else {
          q_gemv_wait<(R - 1) * L::kLoads + XI>();
        }
        const uint8_t* const item = mine + XI * 1024 + r * L::kItem;
        typename Provider::Raw w;
        u32x4 piece[kSlots / 4];
#pragma unroll
        for (int i = 0; i < kSlots / 4; ++i)
          piece[i] = *reinterpret_cast<const u32x4*>(
              item + c * L::kRow + (((q * (kSlots / 4) + i) ^ (kSlots == 8 ? (c >> 1) & 7 : c)) << 4));
        if constexpr (NBITS == 4) w.w0 = piece[0], w.w1 = piece[1];
        else w.w[0] = piece[0], w.w[1] = piece[1], w.w[2] = piece[2], w.w[3] = piece[3];
        // groups of 32: both scales of a chunk in one dword; larger: one scale, in either half of it
        const int kc = min(step * 4 + q, s.chunks - 1);
        const uint32_t index = (uint32_t)min(16 * r + c, last_row) * (uint32_t)a.groups_per_row + (uint32_t)((2 * kc) >> a.gs_shift_chunks);
        const uint32_t sh_lo = a.gs_shift_chunks ? (index & 1u) * 16u : 0u, sh_hi = a.gs_shift_chunks ? sh_lo : 16u;
        const uint32_t sc = *reinterpret_cast<const uint32_t*>(item + L::kCodes + (c * 4 + q) * 4);
        w.s_lo = ((sc >> sh_lo) & 0xFFFFu) * 0x10001u;
        w.s_hi = ((sc >> sh_hi) & 0xFFFFu) * 0x10001u;
        if constexpr (ASYM) {
          const uint32_t zp = *reinterpret_cast<const uint32_t*>(item + L::kCodes + 256 + (c * 4 + q) * 4);
          w.z_lo = (zp >> sh_lo) & 0xFFFFu;
          w.z_hi = (zp >> sh_hi) & 0xFFFFu;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (!LAST) load_item(r, step + 1);
        u32x4 b[8];
        b[0] = prov.template operand<0>(w);
        b[1] = prov.template operand<1>(w);
        b[2] = prov.template operand<2>(w);
        b[3] = prov.template operand<3>(w);
        b[4] = prov.template operand<4>(w);
        b[5] = prov.template operand<5>(w);
        b[6] = prov.template operand<6>(w);
        b[7] = prov.template operand<7>(w);
        if (ragged) {
#pragma unroll
          for (int j = 0; j < 8; ++j) b[j] = dead ? u32x4{0u, 0u, 0u, 0u} : b[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[r][t] = mfma16<ACT>(xa[t][j], b[j], acc[r][t]);
      }
    };
    for (int step = step_begin; step < step_end - 1; ++step) one_step(std::false_type{}, step);
    one_step(std::true_type{}, step_end - 1);
  }

  // D layout: lane (c, q) holds D[m = 16 t + 4 q + i][n = c], i = 0..3.
  constexpr int kCols = 16 * R;
  float* const red = reinterpret_cast<float*>(q_lds);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 16 * t + 4 * q + i;
        if (m < s.M) red[(wave * s.M + m) * kCols + r * 16 + c] = acc[r][t][i];
      }
  __syncthreads();
  for (int o = threadIdx.x; o < s.M * kCols; o += blockDim.x) {
    const int m = o / kCols, n = row0 + o % kCols;
    if (n >= s.N) continue;
    float v = 0.f;
    for (int w = 0; w < n_waves; ++w) v += red[w * s.M * kCols + o];
    if (s.bias) v += s.bias[n];
    store_from_f32<ACT>(s.y, (int64_t)m * s.ldy + n, v);
  }
}

template <int ACT, int NBITS, bool ASYM, class Provider, int R, int XI>
int launch_q_gemv_rx(GemvShape s, const typename Provider::Args& a, int blocks_per_cu, hipStream_t st, const char* what) {
  using L = QGemvLds<NBITS, ASYM, R, XI>;
  // Four waves, one per SIMD, except where a compute unit has a single block of one row tile: us with four / eight, int4 at 8
  // tokens, 4096 x 14336 13.9 / 12.6, 4096 x 4096 5.4 / 5.2; 11008 x 4096 10.7 / 10.5 and with 16 tokens, where LDS holds
  // fewer blocks of eight, 13.0 / 15.1; 14336 x 4096 int8 16.6 / 19.0; 6 waves (two SIMDs with two) 15.8 where four take 13.1.
  const int waves_wanted = R == 1 && blocks_per_cu <= 1 && L::kMaxWaves >= 8 ? 8 : 4;
  s.steps_per_wave = (s.steps + waves_wanted - 1) / waves_wanted;
  if (tuning().gemv_spw > 0) s.steps_per_wave = max(tuning().gemv_spw, (s.steps + L::kMaxWaves - 1) / L::kMaxWaves);
  const int waves = (s.steps + s.steps_per_wave - 1) / s.steps_per_wave;
  const int blocks = (s.N + 16 * R - 1) / (16 * R);
  const int stage = waves * L::kWave, red = waves * (s.M < kGemvTokens ? s.M : kGemvTokens) * 16 * R * 4;
  const int lds = stage > red ? stage : red;
  if (lds > 64 * 1024) {
    static LdsLatch latch;  // per instantiation
    const hipError_t e =
        enable_dynamic_lds(latch, reinterpret_cast<const void*>(&q_gemv_kernel<ACT, NBITS, ASYM, Provider, R, XI>), lds);
    if (e != hipSuccess) return fail(NPAMD_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS: %s", what, lds, hipGetErrorString(e));
  }
  last_gemv_staged() = 1;
  launch(q_gemv_kernel<ACT, NBITS, ASYM, Provider, R, XI>, dim3(blocks, (s.M + kGemvTokens - 1) / kGemvTokens), waves * 64, lds, st, s, a);
  return check_launch(what);
}

template <int ACT, int NBITS, bool ASYM, class Provider, int R>
int launch_q_gemv_r(const GemvShape& s, const typename Provider::Args& a, int blocks_per_cu, hipStream_t st, const char* what) {
  if (s.M <= 2) return launch_q_gemv_rx<ACT, NBITS, ASYM, Provider, R, 1>(s, a, blocks_per_cu, st, what);
  if (s.M <= 8) return launch_q_gemv_rx<ACT, NBITS, ASYM, Provider, R, 4>(s, a, blocks_per_cu, st, what);
  if (s.M <= 16) return launch_q_gemv_rx<ACT, NBITS, ASYM, Provider, R, 8>(s, a, blocks_per_cu, st, what);
  return launch_q_gemv_rx<ACT, NBITS, ASYM, Provider, R, 16>(s, a, blocks_per_cu, st, what);
}

// One row tile per block, or two, which read the activations once, from three tokens on where K is long enough for four waves
// to have two steps each and pairs of tiles leave the fullest compute unit no more than an eighth more of them.  us with
// one / two tiles: 14336 x 4096 int4 at 1 / 8 / 16 / 32 tokens 11.0 / 11.1, 12.8 / 12.0, 16.0 / 13.6, 22.7 / 20.6; 14336 x 512
// 4.1 / 4.9 at 8; 11008 x 4096 (three tiles against two pairs) 10.7 / 11.3.
template <int ACT, int NBITS, bool ASYM, class Provider>
int launch_q_gemv(GemvShape s, const typename Provider::Args& a, int cus, hipStream_t st, const char* what) {
  s.steps = (s.chunks + 3) / 4;
  const int token_blocks = (s.M + kGemvTokens - 1) / kGemvTokens;
  const int tiles = (s.N + 15) / 16 * token_blocks, pairs = ((s.N + 15) / 16 + 1) / 2 * token_blocks;
  const int load1 = (tiles + cus - 1) / cus, load2 = (pairs + cus - 1) / cus;  // blocks of the fullest compute unit
  int R = s.M > 2 && s.steps >= 8 && load1 > 1 && 2 * load2 * 8 <= load1 * 9 ? 2 : 1;
  // More than 32 tokens: a block's activations take 16 KiB of LDS per wave whatever its row tiles.  Two where that saves a round of
  // blocks: int8 at 64 tokens, one / two, 4096 x 1024 6.9 / 5.4, 3072 x 3072 10.4 / 8.2; int4, two blocks of one tile to a compute unit,
  // 3072 x 3072 at 96 11.1 / 14.8, 4096 x 1024 at 128 8.3 / 9.1, 2048 x 2048 at 256 11.6 / 12.1.
  if (token_blocks > 1) {
    const int waves = s.steps < 4 ? s.steps : 4;
    const int fit1 = kGemvLdsPerBlockMax / (waves * QGemvLds<NBITS, ASYM, 1, 16>::kWave);
    const int fit2 = kGemvLdsPerBlockMax / (waves * QGemvLds<NBITS, ASYM, 2, 16>::kWave);
    const int rounds1 = (load1 + fit1 - 1) / fit1, rounds2 = (load2 + fit2 - 1) / fit2;
    R = rounds2 < rounds1 || (R == 2 && rounds2 == rounds1) ? 2 : 1;
  }
  if (tuning().gemv_r > 0) R = tuning().gemv_r > 1 ? 2 : 1;
  if (R == 2) return launch_q_gemv_r<ACT, NBITS, ASYM, Provider, 2>(s, a, load2, st, what);
  return launch_q_gemv_r<ACT, NBITS, ASYM, Provider, 1>(s, a, load1, st, what);
}

}  // namespace npamd
