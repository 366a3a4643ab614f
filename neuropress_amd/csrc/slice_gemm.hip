// The slice GEMM (see slice_gemm.hpp): kernel, plan and launcher.
#include "slice_gemm.hpp"

#include <type_traits>
#include <utility>

namespace npamd {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

constexpr int kSliceRows = 8192;           // codebook rows per slice at most
constexpr int kSliceXBytes = 16 * 1024;    // a super-step's activations

// Loads that write LDS directly: lane l's 16 bytes land at dst + 16 l; dst is uniform over the wave.
__device__ __forceinline__ void slice_lds_load16(uint32_t dst, const void* from) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(from) : "memory");
}

template <int ACT>
__device__ __forceinline__ bool any_nonfinite(const u32x4& v) {
  constexpr uint32_t kExp = ACT == NPAMD_BF16 ? 0x7F80u : 0x7C00u;
  const auto mag = [](uint32_t d) { return __builtin_bit_cast(u16x2, d & 0x7FFF7FFFu); };
  const u16x2 m = __builtin_elementwise_max(__builtin_elementwise_max(mag(v.x), mag(v.y)),
                                            __builtin_elementwise_max(mag(v.z), mag(v.w)));
  return m.x >= kExp || m.y >= kExp;
}

template <int I>
using Int = std::integral_constant<int, I>;
template <int N, class Fn, int... I>
__device__ __forceinline__ void static_for_in(Fn&& fn, std::integer_sequence<int, I...>) {
  (fn(Int<I>{}), ...);
}
template <int N, class Fn>
__device__ __forceinline__ void static_for(Fn&& fn) {
  static_for_in<N>(fn, std::make_integer_sequence<int, N>{});
}

// A row of the slice by its LDS address.  Dynamic LDS starts where a kernel's static LDS ends, and this kernel has none.
typedef __attribute__((address_space(3))) u32x4 LdsRow;
__device__ __forceinline__ u32x4 lds_row(uint32_t at) { return *(const LdsRow*)at; }

// Half of a packed index difference (see the walk) as an LDS address: one instruction.
template <int HALF>
__device__ __forceinline__ uint32_t row_address(uint32_t rel) {
  uint32_t at;
  if constexpr (HALF)
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(at) : "v"(4), "v"(rel));
  else
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(at) : "v"(4), "v"(rel));
  return at;
}

// MT token tiles of 16; T row tiles per wave; CLAMP: indices may lie past the codebook, or the last super-step past K.
// Eight waves: two k groups x four row groups with one token tile, eight row groups with two.
template <int MT>
struct SliceShape {
  static constexpr int kWaves = 8, kKG = MT == 1 ? 2 : 1, kRG = kWaves / kKG;
};
template <int ACT, int MT, int T, bool CLAMP>
__global__ void __launch_bounds__((SliceShape<MT>::kWaves * 64))
slice_gemm_kernel(const SliceArgs a) {
  constexpr int KG = SliceShape<MT>::kKG, RG = SliceShape<MT>::kRG, kThreads = SliceShape<MT>::kWaves * 64;
  constexpr int kTokens = 16 * MT, kUnits = kTokens * KG * 32 / kThreads;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // slice, zero row, activations, flag
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, q = lane >> 4;
  const int kg = wave % KG, rg = wave / KG;

  // Blocks go to the dies in turn; the slices of a cell stay on one die.
  const int die = blockIdx.x & 7, turn = blockIdx.x >> 3;
  const int slice = turn % a.slices, cell = (turn / a.slices) * 8 + die;
  if (cell >= a.row_blocks * a.parts) return;
  const int part = cell % a.parts, row_block = cell / a.parts;
  const int ss_begin = part * a.part_super;
  const int ss_all = (a.chunks + 4 * KG - 1) / (4 * KG);
  const int ss_end = min(ss_begin + a.part_super, ss_all);
  const int row0 = row_block * (16 * RG * T) + rg * (16 * T);
  const int base = slice * a.slice_rows;
  const int rows = min(a.slice_rows, a.nc - base);  // of this slice
  const uint32_t xs_at = (uint32_t)(a.slice_rows + 1) * 16u;
  uint8_t* const xs = lds + xs_at;
  int* const flag = reinterpret_cast<int*>(lds + xs_at + kSliceXBytes);

  // ---- requests of the first super-step, then the slice -----------------------------------------------------------
  // A thread's 16-byte units of a super-step's activations.
  u32x4 xr[kUnits];
  int xw[kUnits];
  const uint16_t* xp[kUnits];
  int xchunk[kUnits];
#pragma unroll
  for (int i = 0; i < kUnits; ++i) {
    const int u = (int)threadIdx.x + kThreads * i;
    const int token = u / (32 * KG), within = u % (32 * KG), g = within / 32, unit = within % 32;
    xw[i] = ((g * kTokens + token) * 32 + (unit ^ (token & 7))) * 16;
    xchunk[i] = g * 4 + unit / 8;
    xp[i] = reinterpret_cast<const uint16_t*>(a.x) + (int64_t)min(token, a.M - 1) * a.ldx + (unit % 8) * 8;
  }
  const auto load_x = [&](int ss) {
#pragma unroll
    for (int i = 0; i < kUnits; ++i)
      xr[i] = *reinterpret_cast<const u32x4*>(xp[i] + (int64_t)min(ss * (4 * KG) + xchunk[i], a.chunks - 1) * 64);
  };
  u32x4 raw[2][T];  // of this super-step and the next
  uint32_t rp[T];  // byte offsets of the lane's rows (the stream is shorter than 4 GiB)
#pragma unroll
  for (int r = 0; r < T; ++r) rp[r] = (uint32_t)min(row0 + 16 * r + c, a.N - 1) * (uint32_t)a.chunks * 16u;
  const auto chunk_of = [&](int ss) { return ss * (4 * KG) + kg * 4 + q; };
  load_x(ss_begin);
  const auto load_raw = [&](u32x4(&to)[T], int ss) {
    const uint32_t kc = (uint32_t)min(chunk_of(min(ss, ss_end - 1)), a.chunks - 1) * 16u;
#pragma unroll
    for (int r = 0; r < T; ++r) to[r] = *reinterpret_cast<const u32x4*>(a.packed + (rp[r] + kc));
  };
  load_raw(raw[0], ss_begin);
  {
    const uint32_t dst0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const u32x4* const src = reinterpret_cast<const u32x4*>(a.cb) + base;
    for (int k = wave; k * 64 < rows; k += kThreads / 64)
      slice_lds_load16(dst0 + (uint32_t)k * 1024u, src + min(k * 64 + lane, rows - 1));
  }
  const auto store_x = [&] {
#pragma unroll
    for (int i = 0; i < kUnits; ++i) *reinterpret_cast<u32x4*>(xs + xw[i]) = xr[i];
  };
  if (threadIdx.x == 0) *flag = 0;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x < 4) reinterpret_cast<uint32_t*>(lds + (uint32_t)rows * 16u)[threadIdx.x] = 0u;  // the zero row
  store_x();
  __syncthreads();

  f32x4 acc[T][MT];
#pragma unroll
  for (int r = 0; r < T; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  constexpr int P = T >= 2 ? 2 : 1;  // row tiles looked up together
  constexpr int D = P == 2 ? 3 : 7;  // operands looked up ahead
  constexpr int kStages = T / P * 8, kMid = kStages / 2;
  constexpr int kPieces = (8 * MT + kMid - 1) / kMid;  // of the activations, read per stage of the second half
  static_assert(kStages % (D + 1) == 0, "the ring of looked-up operands goes on from one super-step to the next");
  u32x4 xa[2][MT][8], b[D + 1][P];
  uint32_t rel[P], last2, base2, kc_after;
  const uint32_t rows2 = (uint32_t)rows * 0x10001u;
  const auto clamped = [&](int ss) { return min(ss, ss_end - 1); };
  // Lanes past K look up zeros whatever they read: 0 - 1 is past every slice.
  const auto start = [&](int ss) {
    const bool kvalid = !CLAMP || chunk_of(ss) < a.chunks;
    base2 = kvalid ? (uint32_t)base * 0x10001u : 0x10001u;
    if constexpr (CLAMP) {
      last2 = kvalid ? (uint32_t)(a.nc - 1) * 0x10001u : 0u;
      asm volatile("" : "+v"(last2), "+v"(base2));
    }
    kc_after = (uint32_t)min(chunk_of(clamped(ss + 2)), a.chunks - 1) * 16u;
  };
  const auto look = [&](auto buf, auto stage) {
    constexpr int s = decltype(stage)::value, j = s % 8, BUF = decltype(buf)::value;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      constexpr int r0 = s / 8 * P;
      if constexpr (j % 2 == 0) {
        const uint32_t two = raw[BUF][r0 + p][j / 2];
        u16x2 v = __builtin_bit_cast(u16x2, two);
        if constexpr (CLAMP) v = __builtin_elementwise_min(v, __builtin_bit_cast(u16x2, last2));
        v -= __builtin_bit_cast(u16x2, base2);
        rel[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(v, __builtin_bit_cast(u16x2, rows2)));
      }
      b[s % (D + 1)][p] = lds_row(row_address<j % 2>(rel[p]));
      if constexpr (j == 7) raw[BUF][r0 + p] = *reinterpret_cast<const u32x4*>(a.packed + (rp[r0 + p] + kc_after));
    }
  };
  const auto read_x = [&](auto buf, auto piece) {
    constexpr int t = decltype(piece)::value / 8, j = decltype(piece)::value % 8;
    xa[decltype(buf)::value][t][j] =
        *reinterpret_cast<const u32x4*>(xs + ((kg * kTokens + t * 16 + c) * 32 + ((q * 8 + j) ^ (c & 7))) * 16);
  };
  // One super-step, its activations in xa[BUF].  Everything is asked for ahead of its use: the lookups of D operands, across
  // the end of the super-step; the activations of the next one go to LDS at the start, and to registers in the second half,
  // between two barriers that a wave reaches with half a super-step of work behind it.
  const auto super_step = [&](auto buf, int ss, auto last) {
    constexpr int BUF = decltype(buf)::value;
    constexpr bool LAST = decltype(last)::value;  // nothing is asked for past the end
    static_for<kStages>([&](auto stage) {
      constexpr int s = decltype(stage)::value;
      if constexpr (s == kStages - D && !LAST) start(ss + 1);
      if constexpr (s >= kMid && !LAST)
        static_for<kPieces>([&](auto i) {
          constexpr int piece = (s - kMid) * kPieces + decltype(i)::value;
          if constexpr (piece < 8 * MT) read_x(Int<1 - BUF>{}, Int<piece>{});
        });
      if constexpr (s + D < kStages || !LAST) look(Int<s + D < kStages ? BUF : 1 - BUF>{}, Int<(s + D) % kStages>{});
      if constexpr (s == 0 && !LAST) {
        block_sync_lds_keep<P>();  // everybody has read this super-step's activations (their lookups may still be under way)
        store_x();
        load_x(clamped(ss + 2));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[s / 8 * P + p][t] = mfma16<ACT>(b[s % (D + 1)][p], xa[BUF][t][s % 8], acc[s / 8 * P + p][t]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s == kMid - 1 && !LAST) block_sync_lds_keep<(P * D < (kMid - 1) * P ? P * D : (kMid - 1) * P)>();
    });
  };
  static_for<8 * MT>([&](auto i) { read_x(Int<0>{}, i); });
  load_x(clamped(ss_begin + 1));
  __builtin_amdgcn_sched_barrier(0);
  load_raw(raw[1], ss_begin + 1);  // behind the activations, as in the loop: nothing waits for the younger of the two
  __builtin_amdgcn_sched_barrier(0);
  start(ss_begin);
  static_for<D>([&](auto s) { look(Int<0>{}, s); });
  int ss = ss_begin;
  for (; ss + 1 < ss_end; ss += 2) {
    super_step(Int<0>{}, ss, std::false_type{});
    super_step(Int<1>{}, ss + 1, std::false_type{});
  }
  if (ss < ss_end) super_step(Int<0>{}, ss, std::true_type{});

  // An index outside the slice multiplies its activations by zeros, which is not nothing where they are infinite or NaN: then
  // every sum comes out as neither.  So only where a sum does is the part's x looked over, and with such a value in it -- all
  // slices of the cell find the same -- the part is done again, every slice's workgroup taking whole super-steps in turn with its lookups in memory.
  bool odd = false;
#pragma unroll
  for (int r = 0; r < T; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) odd |= !(fabsf(acc[r][t][i]) <= 3.4028234e38f);
  if (odd) *flag = 1;
  __syncthreads();  // everybody is done with the slice, too
  if (*flag) {
    const int k8_begin = ss_begin * (32 * KG), k8s = min(ss_end * (32 * KG), a.chunks * 8) - k8_begin;
    const uint16_t* const x = reinterpret_cast<const uint16_t*>(a.x);
    bool found = false;
    for (int m = 0; m < a.M; ++m)
      for (int k8 = threadIdx.x; k8 < k8s; k8 += kThreads)
        found |= any_nonfinite<ACT>(*reinterpret_cast<const u32x4*>(x + m * a.ldx + (int64_t)(k8_begin + k8) * 8));
    if (found) *flag = 2;
    __syncthreads();
    if (*flag == 2) {
#pragma unroll
      for (int r = 0; r < T; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (ss = ss_begin; ss < ss_end; ++ss) {
        if (ss % a.slices != slice) continue;
        const bool kvalid = chunk_of(ss) < a.chunks;
        const int64_t k8 = (int64_t)min(chunk_of(ss), a.chunks - 1) * 8;
        for (int j = 0; j < 8; ++j) {
          u32x4 xo[MT];
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            xo[t] = *reinterpret_cast<const u32x4*>(x + min(16 * t + c, a.M - 1) * a.ldx + (k8 + j) * 8);
            xo[t] = kvalid && 16 * t + c < a.M ? xo[t] : u32x4{0u, 0u, 0u, 0u};
          }
#pragma unroll
          for (int r = 0; r < T; ++r) {
            const uint32_t id = *reinterpret_cast<const uint16_t*>(a.packed + (rp[r] + (uint32_t)(k8 + j) * 2u));
            u32x4 w = reinterpret_cast<const u32x4*>(a.cb)[min(id, (uint32_t)a.nc - 1u)];
            w = kvalid ? w : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[r][t] = mfma16<ACT>(w, xo[t], acc[r][t]);
          }
        }
      }
    }
  }
  // D[weight 4q + i][token c].  The k groups' sums meet in LDS (over the slice).
  if constexpr (KG == 2) {
    f32x4* const meet = reinterpret_cast<f32x4*>(lds) + (rg * T) * 64 + lane;
    if (kg == 1) {
#pragma unroll
      for (int r = 0; r < T; ++r) meet[r * 64] = acc[r][0];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int r = 0; r < T; ++r) acc[r][0] += meet[r * 64];
  }
  float* const out = a.partials + (int64_t)(part * a.slices + slice) * a.M * a.N;
#pragma unroll
  for (int r = 0; r < T; ++r) {
    const int n = row0 + 16 * r + 4 * q;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = 16 * t + c;
      if (m >= a.M || n >= a.N) continue;
      float* const p = out + (int64_t)m * a.N + n;
      if (a.N % 4 == 0) {
        *reinterpret_cast<f32x4*>(p) = acc[r][t];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < a.N) p[i] = acc[r][t][i];
      }
    }
  }
}

// Microseconds of a plan: a fit (5 % r.m.s.) to 120 calls of 3 to 32 tokens on layers of 0.5 to 8.4 M indices with codebooks of
// 5000 to 65536 rows.  Per round of workgroups the fill and the super-steps (lanes of a lookup that hit conflict in LDS: the
// fewer slices the more of them), then the partial sums, written and read again.
static double slice_us(const SlicePlan& p, int M, int N) {
  const int mt = M > 16 ? 2 : 1;
  const int rounds = ((p.row_blocks * p.parts + 7) / 8 * p.slices + 31) / 32;
  const double step = 0.17 + p.tiles * (0.164 + 0.052 * mt + 0.445 / p.slices);
  return 4.8 + rounds * (1.6 * p.slice_rows / kSliceRows + p.part_super * step) + 0.786e-6 * (double)slice_partials_bytes(p, M, N);
}

// Of one, two and four row tiles per wave, with K in as many parts as one round of workgroups holds (32 compute units a
// die), half as many, or whole: the one that should be fastest.
static SlicePlan plan_slice(int M, int N, int chunks, int nc) {
  const int slices = (nc + kSliceRows - 1) / kSliceRows, slice_rows = ((nc + slices - 1) / slices + 63) / 64 * 64;
  const int mt = M > 16 ? 2 : 1, kg = mt == 1 ? 2 : 1, rg = 8 / kg;
  const int super = (chunks + 4 * kg - 1) / (4 * kg);
  SlicePlan best{};
  double best_us = 0;
  const int tiles_env = tuning().slice_tiles, parts_env = tuning().slice_parts;
  for (int t = 1; t <= 4; t *= 2) {
    if ((tiles_env == 1 || tiles_env == 2 || tiles_env == 4) && t != tiles_env) continue;
    SlicePlan p{slices, slice_rows, t, (N + 16 * rg * t - 1) / (16 * rg * t), 1, super};
    const int most = 32 / slices * 8 / p.row_blocks;
    for (int parts : {most, most / 2, 1}) {
      if (parts_env > 0) parts = parts_env < super ? parts_env : super;
      if (parts < 1) continue;
      p.part_super = (super + parts - 1) / parts;
      p.parts = (super + p.part_super - 1) / p.part_super;
      const double us = slice_us(p, M, N);
      if (!best.tiles || us < best_us) {
        best = p;
        best_us = us;
      }
    }
  }
  return best;
}

bool slice_takes(int M, int N, int K, int nc) {
  return M >= 1 && M <= kSliceMaxTokens && N >= 1 && K >= 64 && K % 64 == 0 && nc > 4096 && nc <= 65536 &&
         (int64_t)N * (K / 64) * 16 < ((int64_t)1 << 32);
}

int64_t slice_workspace_bytes(int M, int N, int chunks, int nc) {
  return slice_partials_bytes(plan_slice(M, N, chunks, nc), M, N);
}

double slice_estimate_ns(int M, int N, int chunks, int nc) {
  const double ns = 1e3 * slice_us(plan_slice(M, N, chunks, nc), M, N);
  return ns < 2e9 ? ns : 2e9;
}

template <int ACT, int MT, int T, bool CLAMP>
static int launch_slice_t(const SliceArgs& a, hipStream_t st, const char* what) {
  const int lds = (a.slice_rows + 1) * 16 + kSliceXBytes + 16;
  static LdsLatch latch;
  const hipError_t e = enable_dynamic_lds(latch, reinterpret_cast<const void*>(&slice_gemm_kernel<ACT, MT, T, CLAMP>), lds);
  if (e != hipSuccess) return fail(NPAMD_ERR_LAUNCH, "%s: cannot reserve %d bytes of LDS: %s", what, lds, hipGetErrorString(e));
  const int cells = a.row_blocks * a.parts;
  launch(slice_gemm_kernel<ACT, MT, T, CLAMP>, (unsigned)((cells + 7) / 8 * 8 * a.slices), SliceShape<MT>::kWaves * 64, lds, st, a);
  return NPAMD_OK;
}

template <int ACT, int MT, bool CLAMP>
static int launch_slice_mt(int tiles, const SliceArgs& a, hipStream_t st, const char* what) {
  switch (tiles) {
    case 1: return launch_slice_t<ACT, MT, 1, CLAMP>(a, st, what);
    case 2: return launch_slice_t<ACT, MT, 2, CLAMP>(a, st, what);
    default: return launch_slice_t<ACT, MT, 4, CLAMP>(a, st, what);
  }
}

template <int ACT>
static int launch_slice_act(const GemmShape& s, const SlicePlan& p, const SliceArgs& a, hipStream_t st, const char* what) {
  const bool clamp = a.nc < 65536 || a.chunks % (s.M <= 16 ? 8 : 4);
  const int rc = s.M <= 16 ? (clamp ? launch_slice_mt<ACT, 1, true>(p.tiles, a, st, what) : launch_slice_mt<ACT, 1, false>(p.tiles, a, st, what))
                           : (clamp ? launch_slice_mt<ACT, 2, true>(p.tiles, a, st, what) : launch_slice_mt<ACT, 2, false>(p.tiles, a, st, what));
  if (rc != NPAMD_OK) return rc;
  launch_splitk_reduce<ACT>(a.partials, p.slices * p.parts, s.M, s.N, s.bias, s.y, s.ldy, st);
  return check_launch(what);
}

int launch_slice(int act, const GemmShape& s, const uint8_t* packed, const void* cb, int nc, hipStream_t st, const char* what,
                 void* workspace) {
  const SlicePlan p = plan_slice(s.M, s.N, s.chunks, nc);
  const SliceArgs a{s.x, s.ldx, packed, cb, (float*)workspace, s.M, s.N, s.chunks, nc,
                    p.slices, p.slice_rows, p.row_blocks, p.parts, p.part_super};
  return act == NPAMD_BF16 ? launch_slice_act<NPAMD_BF16>(s, p, a, st, what) : launch_slice_act<NPAMD_F16>(s, p, a, st, what);
}

}  // namespace npamd
