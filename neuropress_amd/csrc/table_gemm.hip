// Product of more than 16 tokens with a plain VQ weight whose codebook LDS holds: y = x @ W^T (+ bias), wave64 + MFMA 32x32x16, f32
// accumulate, W never written.  Vector length 8, 8, 12 or 16 bits per index, up to 4096 rows, the codebook in the activation type.
//
// What it takes the place of is decode + dense product, two launches of which the second brings W back out of the L2s, and past
// 64 tokens the tile GEMM, whose producer waves write W into LDS for others to read.  A codebook row is an MFMA operand as it
// lies, so here a wave looks the operands of its 64 columns up in the block's LDS copy of the table and uses each for MT
// MFMAs; nothing but x and indices is loaded, 1 / 8 to 1 / 16 of W's bytes.
//
// A block keeps a tile of 32 MT x 64; its KG waves share out K, two 64-k steps at a time, and meet only in the end, in LDS, every
// wave adding up its share of the 32 x 32 tiles in the waves' order.  Each wave brings its own x (rows of 128 bytes, 16-byte piece p
// of row r in place p ^ ((r >> 1) & 7)) and its own indices straight into LDS (global_load_lds); there is no barrier in the loop.
// A step: its operands of x go into registers at once, which frees their place for the next step's while the MFMAs run; behind
// the MFMAs of a k group the rows of that group in the next step are looked up; the indices of the step after that are read.
//
// What bounds it: at 256 x 4096 x 4096 with 256 rows (12.3 us; start and end 4 of them) the matrix pipes are busy a third of the time, LDS 45 %; a
// wave's step is a chain of its x arriving, its LDS reads and its MFMAs, which two waves per SIMD (KG = 8) or larger tiles
// cover in part.  Tried without gain: two and three places for x, reads a step ahead, copies of the table side by side
// (fewer bank conflicts), column tiles that start K at different steps, loads between the single MFMAs (14.2 us for 11.9).
// us per call through the module, decode + product or tile GEMM / this kernel, 256 rows: 4096 x 4096 at 128 / 256 / 384 / 512 tokens 15.7 / 8.8,
// 24.8 / 12.3, 28.6 / 17.5, 31.5 / 22.0; 2048 x 2048 at 256 / 512 11.0 / 6.5, 13.5 / 8.8; 9856 x 12544 at 64 / 256 44.9 / 23.7, 169.6 / 82.1;
// 4096 rows: 4096 x 4096 at 128 / 256 / 512 17.8 / 12.1, 25.0 / 15.1, 31.9 / 24.6; 14336 x 14336 at 384 302 / 182.
// The line against the other kernels: npamd_gemv_blocks_preferred (dense_gemm.hip), which compares estimates of all of them.
#include "table_gemm.hpp"

#include "../../include/npamd_diag.h"

#include <math.h>

#include <type_traits>

#include "gemm_tile.hpp"
#include "lds_transfer.hpp"

namespace npamd {

namespace {

struct TableShape {
  const void* x;
  const uint8_t* packed;
  const void* cb;
  const float* bias;
  void* y;
  int64_t ldx, ldy;
  int M, N, steps, pieces;  // 64-k steps of an index row; 16-byte pieces of a row of x
  uint32_t nc_minus_1;
  int row_tiles, col_tiles, units_per_die;
};

constexpr int kTableCols = 64;
constexpr int kCodeSteps = 2;  // steps whose indices are brought together
constexpr int kTableMaxK = 1 << 20;

template <int BITS, int MT, int KG>
struct TableTile {
  static constexpr int kBM = 32 * MT;
  static constexpr int kThreads = 64 * KG;
  static constexpr int kSlotBytes = kBM * 128;
  static constexpr int kCodeRow = kCodeSteps * BITS;  // bytes: a step is eight indices
  static constexpr int kCodeBytes = kTableCols * kCodeRow;
  static constexpr int kXLoads = kBM / 8, kCodeLoads = BITS == 16 ? kCodeBytes / 1024 : kCodeBytes / 256;
  static constexpr int kWaveBytes = kSlotBytes + 2 * kCodeBytes;
  static constexpr int kTable = KG * kWaveBytes;  // where the table lies
  static constexpr int kEpRow = kTableCols * 2 + 16;
  static constexpr int kEp = KG * 2 * MT * 4096;
  static constexpr int kEnd = kEp + kBM * kEpRow;
  static constexpr int lds(int table_bytes) { return kTable + table_bytes > kEnd ? kTable + table_bytes : kEnd; }
};

template <int ACT, int BITS, int MT, int KG>
__global__ void __launch_bounds__((TableTile<BITS, MT, KG>::kThreads))
table_gemm_kernel(const TableShape s) {
  using T = TableTile<BITS, MT, KG>;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // blockIdx.x % 8 names the die; a die takes an eighth of the tiles, counted along their rows: its L2 brings few rows of x
  const int unit = (blockIdx.x & 7) * s.units_per_die + (blockIdx.x >> 3);
  const int rt = unit / s.col_tiles, ct = unit - rt * s.col_tiles;
  if (rt >= s.row_tiles) return;
  const int m0 = rt * T::kBM, n0 = ct * kTableCols;
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, h = lane >> 5;

  // This wave's steps: two at a time, every KG-th two.  The very last of all may be one.
  const int twos = (s.steps + 1) / 2;
  const int mine = twos > g ? (twos - g + KG - 1) / KG : 0;
  const int total = mine ? 2 * mine - (2 * (g + KG * (mine - 1)) + 1 == s.steps) : 0;
  auto step_of = [&](int t) { return ((t >> 1) * KG + g) * 2 + (t & 1); };

  const uint8_t* const xb = uniform_ptr(reinterpret_cast<const uint8_t*>(s.x) + (int64_t)m0 * s.ldx * 2);
  const int row_bytes = s.steps * BITS;
  const uint8_t* const wb = uniform_ptr(s.packed + (int64_t)n0 * row_bytes);
  uint32_t xoff[T::kXLoads];
#pragma unroll
  for (int i = 0; i < T::kXLoads; ++i) xoff[i] = (uint32_t)((int64_t)min(i * 8 + (lane >> 3), s.M - 1 - m0) * s.ldx * 2);
  const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + (uint32_t)(g * T::kWaveBytes);
  // Load i of a step of x whose rows begin at piece `at`: rows of 128 bytes, piece p of row r in place p ^ ((r >> 1) & 7).
  auto load_x = [&](int i, int at) {
    const int p = (lane & 7) ^ ((i * 4 + (lane >> 4)) & 7);
    lds_load16(base + (uint32_t)(i * 1024), xoff[i] + (uint32_t)min(at + p, s.pieces - 1) * 16u, xb);
  };
  // Indices of the wave's two steps `f` (past its end: the last two, which nobody uses), a row's side by side.
  auto load_code = [&](int i, int f) {
    const int two = min(f, mine - 1) * KG + g;
    const uint32_t to = base + (uint32_t)(T::kSlotBytes + (f & 1) * T::kCodeBytes);
    if constexpr (BITS == 16) {
      const int r = i * 32 + (lane >> 1), p = lane & 1;
      lds_load16(to + (uint32_t)(i * 1024), (uint32_t)(min(r, s.N - 1 - n0) * row_bytes + min(two * 2 + p, s.steps - 1) * 16), wb);
    } else {
      constexpr int kDwords = T::kCodeRow / 4;
      const int d = i * 64 + lane, r = d / kDwords, q = d - r * kDwords;
      lds_load4(to + (uint32_t)(i * 256), (uint32_t)(min(r, s.N - 1 - n0) * row_bytes + min(two * kDwords + q, row_bytes / 4 - 1) * 4), wb);
    }
  };

  if (mine) {
#pragma unroll
    for (int i = 0; i < 2 * T::kCodeLoads; ++i) load_code(i % T::kCodeLoads, i / T::kCodeLoads);
#pragma unroll
    for (int i = 0; i < T::kXLoads; ++i) load_x(i, step_of(0) * 8);
  }
  u32x4* const table = reinterpret_cast<u32x4*>(lds + T::kTable);
  {
    const u32x4* const src = reinterpret_cast<const u32x4*>(s.cb);
    for (int i = threadIdx.x; i <= (int)s.nc_minus_1; i += T::kThreads) table[i] = src[i];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  const uint8_t* const own = lds + g * T::kWaveBytes;
  const uint8_t* const codes = own + T::kSlotBytes;
  // The four indices of a lane's column and half of a step, 16 bits each.
  u32x2 idx[2];
  auto read_idx = [&](u32x2 (&idx)[2], int t) {
    const uint8_t* const at = codes + ((t >> 1) & 1) * T::kCodeBytes + (t & 1) * BITS;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const int r = ti * 32 + c;
      if constexpr (BITS == 16) {
        idx[ti] = *reinterpret_cast<const u32x2*>(at + r * T::kCodeRow + h * 8);
      } else if constexpr (BITS == 8) {
        idx[ti].x = *reinterpret_cast<const uint32_t*>(at + r * T::kCodeRow + h * 4);
      } else {
        const uint32_t* const p = reinterpret_cast<const uint32_t*>(at + r * T::kCodeRow + h * 4);
        idx[ti] = u32x2{p[0], p[1]};  // 48 bits, behind 16 others in the upper half
      }
    }
  };
  auto index = [&](const u32x2& v, int j) -> uint32_t {
    if constexpr (BITS == 16) return ((j & 1) ? (j & 2 ? v.y : v.x) >> 16 : (j & 2 ? v.y : v.x) & 0xFFFFu);
    else if constexpr (BITS == 8) return (v.x >> (8 * j)) & 0xFFu;
    else {
      const uint64_t all = (((uint64_t)v.y << 32) | v.x) >> (h ? 16 : 0);
      return (uint32_t)(all >> (12 * j)) & 0xFFFu;
    }
  };

  f32x16 acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][ti][i] = 0.f;

  u32x4 a[4][MT], b[4][2];
  uint32_t place[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) place[j] = (uint32_t)(c * 128 + ((((h << 2) | j) ^ ((c >> 1) & 7)) << 4));
  auto look_up = [&](int j, int ti) {
    b[j][ti] = table[min(index(idx[ti], j), s.nc_minus_1)];
  };
  if (total) {
    read_idx(idx, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) look_up(j, ti);
    read_idx(idx, 1);
  }
  // Nothing but loads and zeroes behind a branch: accumulators assigned on two sides of one are copied from register to register where
  // they join (64 moves a step).
  for (int t = 0; t < total; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[j][mt] = *reinterpret_cast<const u32x4*>(own + mt * 4096 + place[j]);
    u32x2 next[2];
    read_idx(next, t + 2);
    const int there = s.pieces - step_of(t) * 8;  // pieces in front of the end of x's rows
    if (there < 8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool dead = 4 * h + j >= there;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[j][mt] = dead ? u32x4{0, 0, 0, 0} : a[j][mt];
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) b[j][ti] = dead ? u32x4{0, 0, 0, 0} : b[j][ti];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < total) {  // into the place of this step's, which are in registers
      if ((t & 1) == 0) {
#pragma unroll
        for (int i = 0; i < T::kCodeLoads; ++i) load_code(i, (t >> 1) + 2);
      }
#pragma unroll
      for (int i = 0; i < T::kXLoads; ++i) load_x(i, step_of(t + 1) * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) acc[mt][ti] = mfma32<ACT>(a[j][mt], b[j][ti], acc[mt][ti]);
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) look_up(j, ti);  // the next step's
      __builtin_amdgcn_sched_barrier(0);
    }
    idx[0] = next[0];
    idx[1] = next[1];
  }

  // The waves' sums meet in LDS, in the waves' order; 32 x 32 tile q is added up by wave q % KG.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  float* const parts = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int q = 0; q < 2 * MT; ++q) {
    if (q % KG == g) continue;
    float* const to = parts + ((size_t)g * 2 * MT + q) * 1024 + lane * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<f32x4*>(to + e * 256) =
          f32x4{acc[q / 2][q % 2][4 * e], acc[q / 2][q % 2][4 * e + 1], acc[q / 2][q % 2][4 * e + 2], acc[q / 2][q % 2][4 * e + 3]};
  }
  __syncthreads();
  uint8_t* const ep = lds + T::kEp;
#pragma unroll
  for (int q = 0; q < 2 * MT; ++q) {
    if (q % KG != g) continue;
    const int n = n0 + (q % 2) * 32 + c;
    const float bv = s.bias && n < s.N ? s.bias[n] : 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < KG; ++z) {
        if (z == g) {
#pragma unroll
          for (int k = 0; k < 4; ++k) sum[k] += acc[q / 2][q % 2][4 * e + k];
        } else {
          const f32x4 v = *reinterpret_cast<const f32x4*>(parts + ((size_t)z * 2 * MT + q) * 1024 + e * 256 + lane * 4);
#pragma unroll
          for (int k = 0; k < 4; ++k) sum[k] += v[k];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int row = (q / 2) * 32 + 8 * e + 4 * h + k;
        const float v = sum[k] + bv;
        *reinterpret_cast<uint16_t*>(ep + row * T::kEpRow + ((q % 2) * 32 + c) * 2) =
            (uint16_t)(ACT == NPAMD_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v));
      }
    }
  }
  __syncthreads();
  const bool whole = s.ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(s.y) & 15) == 0;
  uint16_t* const y = reinterpret_cast<uint16_t*>(s.y);
  for (int i = threadIdx.x; i < T::kBM * 8; i += T::kThreads) {
    const int m = m0 + i / 8, n = n0 + i % 8 * 8;
    if (m >= s.M || n >= s.N) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(ep + i / 8 * T::kEpRow + i % 8 * 16);
    if (whole && n + 8 <= s.N) {
      *reinterpret_cast<u32x4*>(y + (int64_t)m * s.ldy + n) = v;
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < s.N) y[(int64_t)m * s.ldy + n + e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

constexpr int kTableTiles = 5;
constexpr struct { int mt, kg; } kTableTile[kTableTiles] = {{1, 8}, {2, 8}, {2, 4}, {3, 4}, {4, 4}};

int table_lds(int tile, int bits, int table_bytes) {
  const auto& t = kTableTile[tile];
  const int all = t.kg * (t.mt * 4096 + 2 * kTableCols * kCodeSteps * bits) + table_bytes;
  const int end = t.kg * 2 * t.mt * 4096 + 32 * t.mt * (kTableCols * 2 + 16);
  return all > end ? all : end;
}
template <int ACT, int BITS, int MT, int KG>
int launch_table_tile(const VqCall& c) {
  using T = TableTile<BITS, MT, KG>;
  TableShape s{c.x, c.packed, c.cb, c.bias, c.y, c.ldx, c.ldy, c.M, c.N, c.K / 64, (c.k_in ? c.k_in : c.K) / 8, (uint32_t)c.nc - 1u, 0, 0, 0};
  s.row_tiles = (s.M + T::kBM - 1) / T::kBM;
  s.col_tiles = (s.N + kTableCols - 1) / kTableCols;
  const int64_t units = (int64_t)s.row_tiles * s.col_tiles, blocks = (units + 7) / 8 * 8;
  if (blocks > 0x7FFFFFFF) return fail(NPAMD_ERR_UNSUPPORTED, "%s: too many tiles", c.what);
  s.units_per_die = (int)(blocks / 8);
  const int lds = T::lds(c.nc * 16);
  static LdsLatch latch;
  const auto kernel = table_gemm_kernel<ACT, BITS, MT, KG>;
  const hipError_t e = enable_dynamic_lds(latch, reinterpret_cast<const void*>(kernel), lds);
  if (e != hipSuccess) return fail(NPAMD_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS: %s", c.what, lds, hipGetErrorString(e));
  launch(kernel, (unsigned)blocks, T::kThreads, lds, c.st, s);
  return check_launch(c.what);
}

template <int ACT, int BITS>
int launch_table_bits(const VqCall& c, int tile) {
  switch (tile) {
    case 0: return launch_table_tile<ACT, BITS, 1, 8>(c);
    case 1: return launch_table_tile<ACT, BITS, 2, 8>(c);
    case 2: return launch_table_tile<ACT, BITS, 2, 4>(c);
    case 3: return launch_table_tile<ACT, BITS, 3, 4>(c);
    default: return launch_table_tile<ACT, BITS, 4, 4>(c);
  }
}

template <int ACT>
int launch_table(const VqCall& c, int tile) {
  switch (c.bits) {
    case 8: return launch_table_bits<ACT, 8>(c, tile);
    case 12: return launch_table_bits<ACT, 12>(c, tile);
    default: return launch_table_bits<ACT, 16>(c, tile);
  }
}

}  // namespace

// The tile of least estimate: fixed + share of the table + rounds * (per_round + steps of a wave * per step), fitted to 68 layers of 512 to
// 14336 rows, K of 256 to 14336 and tables of 256 to 4096 rows at 32 to 1024 tokens (rms 5 to 9 %).  Two workgroups that share a
// compute unit take `pair` times as long as one.  The figures are those of 16-bit indices, which take the most LDS.
TablePlan plan_table_gemm(int M, int N, int K, int nc) {
  TablePlan best{-1, 1e30f};
  const int forced = tuning().table_tile, twos = (K / 64 + 1) / 2;
  if (forced < 0 || M <= 16 || N < 1 || K < 64 || K % 64 || K > kTableMaxK || nc < 1 || nc * 16 > kTileLdsCodebookMax) return best;
  constexpr struct { float fixed, round, step, crowded, table, pair; } kCost[kTableTiles] = {
      {2.85f, 1.11f, 0.468f, 0.226f, 3.3f, 1.66f},
      {2.10f, 2.51f, 0.679f, 0.309f, 3.2f, 1.5f},
      {2.55f, 1.49f, 0.430f, 0.173f, 3.1f, 1.58f},
      {1.70f, 3.28f, 0.592f, 0.105f, 3.1f, 1.5f},
      {1.62f, 3.95f, 0.727f, 0.190f, 3.3f, 1.5f},
  };
  for (int i = 0; i < kTableTiles; ++i) {
    if (table_lds(i, 16, nc) > kLdsPerBlockMax || (forced > 0 && i != forced - 1)) continue;
    const auto& t = kTableTile[i];
    const auto& c = kCost[i];
    const int64_t blocks = (int64_t)((M + 32 * t.mt - 1) / (32 * t.mt)) * ((N + kTableCols - 1) / kTableCols), load = ((blocks + 7) / 8 + 31) / 32;
    const float rounds = 2 * table_lds(i, 16, nc) <= kLdsPerBlockMax ? (load / 2) * c.pair + (load & 1) : (float)load;
    const int walk = 2 * ((twos + t.kg - 1) / t.kg);
    const float us = c.fixed + rounds * (c.round + walk * (c.step + c.crowded * fminf(1.f, blocks / 256.f)) + c.table * nc / 4096.f);
    if (us < best.us) best = {i, us};
  }
  return best;
}

static int& last_table_tile() {
  static thread_local int tile = -1;
  return tile;
}

int launch_table_gemm(const VqCall& c, float other_us) {
  last_table_tile() = -1;
  if (c.packed_r || c.vl != 8 || c.cb_dtype != c.act || c.ldx >= NPAMD_TILE_MAX_STRIDE || (c.bits != 8 && c.bits != 12 && c.bits != 16)) return 1;
  const TablePlan p = plan_table_gemm(c.M, c.N, c.K, c.nc);
  if (p.tile < 0 || (tuning().table_tile == 0 && p.us >= other_us)) return 1;
  last_table_tile() = p.tile;
  return c.act == NPAMD_BF16 ? launch_table<NPAMD_BF16>(c, p.tile) : launch_table<NPAMD_F16>(c, p.tile);
}

}  // namespace npamd

extern "C" int npamd_diag_last_table_tile(void) { return npamd::last_table_tile(); }
extern "C" int npamd_diag_table_tile(int M, int N, int K, int rows) { return npamd::plan_table_gemm(M, N, K, rows).tile; }
