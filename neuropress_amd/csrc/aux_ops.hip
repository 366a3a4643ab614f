// Neighbours of the quantized linear on the decode step: fused RMSNorm and the
// embedding lookups of VQ- and int-quantized tables.  All three are bound by
// HBM traffic (or, at one token, by the launch); none of them has matrix work.
#include "common.hpp"
#include "gather_columns.hpp"

using namespace npamd;

namespace {

// Rows go to the dies in eighths while what a kernel writes may still be in the L2s when its reader runs (lookup + norm
// of 2048 tokens x 4096: 20.1 us in turn, 16.7 in eighths; of 4096 tokens 27.6 either way, and the norm alone 11.8 / 13.1).
constexpr int64_t kAuxDieBytes = (int64_t)24 << 20;

// How the lookups split a token's row of `vectors` pieces of eight values: pieces per thread (vpt, at most `most`), blocks
// per row (segments), and threads per row and block (lanes).  Short rows share a block of up to 256 threads.  A thread with
// one piece has the shortest chain, which is all that few tokens take (1 / 2 pieces, us: VQ lookup of 64 tokens x 4096 2.49 /
// 2.83, of 256 2.82 / 3.05); many tokens wait for fewer rounds of waves with several (int4 lookup of 4096 tokens x 4096 with
// 1 / 2 / 4 / 8 pieces 13.3 / 11.4 / 10.6 / 9.8, of 3000 10.0 / 8.7 / 7.6 / 7.7, of 2048 7.0 / 6.3 / 6.5 / 6.7; the VQ lookup, bound by
// the L2, 15.6 / 15.3 / 15.9 / 15.5).
struct TokenGrid {
  int vpt, segments;
  unsigned lanes, tokens, threads;
  TokenGrid(int vectors, int64_t n_ids, int most) {
    const int64_t pieces = n_ids * vectors;
    vpt = vectors <= 256 || pieces < 200000 ? 1 : pieces < 1300000 ? 2 : pieces < 1900000 ? 4 : 8;
    if (vpt > most) vpt = most;
    segments = (vectors + 256 * vpt - 1) / (256 * vpt);
    const unsigned need = (unsigned)((vectors + segments * vpt - 1) / (segments * vpt));
    lanes = need <= 128 ? need : (need + 63) / 64 * 64;
    tokens = segments == 1 && lanes <= 128 ? 256 / lanes : 1;
    threads = tokens == 1 ? (lanes + 63) / 64 * 64 : 256;
  }
};
// The block's token and column of a thread; false for the few threads behind the block's last whole token.
__device__ __forceinline__ bool token_of_thread(unsigned lanes, unsigned tokens, unsigned per_die, int64_t* t, int* col) {
  const unsigned sub = tokens == 1 ? 0u : threadIdx.x / lanes;
  *t = die_block(blockIdx.x, per_die) * tokens + sub;
  *col = (int)(threadIdx.x - sub * lanes);
  return sub < tokens && *col < (int)lanes;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int DT>
__device__ __forceinline__ void unpack8(const u32x4& v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = act_bits_to_f32<DT>(v[i] & 0xFFFFu);
    f[2 * i + 1] = act_bits_to_f32<DT>(v[i] >> 16);
  }
}

template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (DT == NPAMD_BF16) return f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
  else return f32_to_f16_bits(lo) | (f32_to_f16_bits(hi) << 16);
}

// ---------------------------------------------------------------------------
// RMSNorm: out[m, i] = round(x[m, i] * rsqrt(mean_i(x[m, i]^2) + eps) * w[i]),
// all arithmetic in f32, one rounding at the store.
//
// The row stays in registers between the sum of squares and the scaling (NV 16-byte vectors per
// lane), so x is read from memory once.  Many rows: one wave per row, four rows per block, bound by
// HBM, an eighth of the rows to each die as the lookups in front of a norm deal them.  Few rows, bound by
// the launch and one memory round trip: four waves per row (ROW_WAVES), which meet in LDS -- a quarter of
// the loads and conversions per lane.
// ---------------------------------------------------------------------------
template <int DT, int NV, int ROW_WAVES>
__global__ void __launch_bounds__(256)
rms_norm_wave_kernel(const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ w,
                     uint16_t* __restrict__ out, int64_t ldo, int M, int H, float eps, unsigned per_die) {
  constexpr int kLanes = 64 * ROW_WAVES;
  const int lane = threadIdx.x & (kLanes - 1);
  const int row = (int)die_block(blockIdx.x, per_die) * (4 / ROW_WAVES) + threadIdx.x / kLanes;
  if (row >= M) return;
  const int n_vec = H >> 3;
  const uint16_t* xr = x + (int64_t)row * ldx;
  u32x4 v[NV], wv[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int p = lane + kLanes * i;
    v[i] = p < n_vec ? *reinterpret_cast<const u32x4*>(xr + 8 * p) : u32x4{0, 0, 0, 0};
  }
  // the weight does not depend on the reduction: requested now, it arrives while the sum is formed
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int p = lane + kLanes * i;
    wv[i] = p < n_vec ? *reinterpret_cast<const u32x4*>(w + 8 * p) : u32x4{0, 0, 0, 0};
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[8];
    unpack8<DT>(v[i], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(f[e], f[e], ss);
  }
  ss = wave_reduce_sum(ss);
  if constexpr (ROW_WAVES > 1) {
    __shared__ float part[ROW_WAVES];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < ROW_WAVES; ++i) ss += part[i];
  }
  const float scale = 1.0f / __builtin_sqrtf(ss / (float)H + eps);
  uint16_t* orow = out + (int64_t)row * ldo;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int p = lane + kLanes * i;
    if (p >= n_vec) continue;
    float f[8], g[8];
    unpack8<DT>(v[i], f);
    unpack8<DT>(wv[i], g);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack2<DT>(f[2 * e] * scale * g[2 * e], f[2 * e + 1] * scale * g[2 * e + 1]);
    *reinterpret_cast<u32x4*>(orow + 8 * p) = o;
  }
}

// Any H, any alignment: one block per row, x read twice.
template <int DT>
__global__ void __launch_bounds__(256)
rms_norm_block_kernel(const void* __restrict__ x, int64_t ldx, const void* __restrict__ w,
                      void* __restrict__ out, int64_t ldo, int H, float eps) {
  __shared__ float part[4];
  const int64_t row = blockIdx.x;
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += 256) {
    const float f = load_as_f32<DT>(x, row * ldx + i);
    ss = __builtin_fmaf(f, f, ss);
  }
  ss = wave_reduce_sum(ss);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float scale = 1.0f / __builtin_sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)H + eps);
  for (int i = threadIdx.x; i < H; i += 256)
    store_from_f32<DT>(out, row * ldo + i, load_as_f32<DT>(x, row * ldx + i) * scale * load_as_f32<DT>(w, i));
}

constexpr int kRmsFewRows = 1024;
template <int DT>
int launch_rms_norm(const void* x, int64_t ldx, const void* w, void* out, int64_t ldo, int M, int H, float eps,
                    hipStream_t st) {
  const bool vec = DT != NPAMD_F32 && H % 8 == 0 && ldx % 8 == 0 && ldo % 8 == 0 && aligned16(x) && aligned16(w) &&
                   aligned16(out) && H <= 8 * 64 * 16;
  if constexpr (DT != NPAMD_F32) {
    if (vec) {
      auto xs = (const uint16_t*)x;
      auto ws = (const uint16_t*)w;
      auto os = (uint16_t*)out;
#define NPAMD_RMS(NV, RW) \
  launch(rms_norm_wave_kernel<DT, NV, RW>, grid.blocks, 256, 0, st, xs, ldx, ws, os, ldo, M, H, eps, grid.per_die)
      if (M <= kRmsFewRows && H > 512) {
        const DieGrid grid(M, (int64_t)M * H * 2, kAuxDieBytes);
        const int nv = (H / 8 + 255) / 256;
        if (nv <= 1) NPAMD_RMS(1, 4);
        else if (nv <= 2) NPAMD_RMS(2, 4);
        else NPAMD_RMS(4, 4);
      } else {
        const DieGrid grid((M + 3) / 4, (int64_t)M * H * 2, kAuxDieBytes);
        const int nv = (H / 8 + 63) / 64;
        if (nv <= 1) NPAMD_RMS(1, 1);
        else if (nv <= 2) NPAMD_RMS(2, 1);
        else if (nv <= 4) NPAMD_RMS(4, 1);
        else if (nv <= 8) NPAMD_RMS(8, 1);
        else NPAMD_RMS(16, 1);
      }
#undef NPAMD_RMS
      return check_launch("npamd_rms_norm");
    }
  }
  launch(rms_norm_block_kernel<DT>, M, 256, 0, st, x, ldx, w, out, ldo, H, eps);
  return check_launch("npamd_rms_norm");
}

// ---------------------------------------------------------------------------
// VQ embedding lookup:
//   row[t, g*VL + v] = C[idx[ids[t], g], v]                       (fp16)
//   out[t, j] = cast(f16(row[t, inv_perm[j]] * scale))            (scale applied when != 1)
// idx is the pre-unpacked [vocab, groups] table of 16-bit indices.
// ---------------------------------------------------------------------------
template <int OUT>
__device__ __forceinline__ void store_embedding8(void* out, int64_t at, const uint32_t (&h)[8], float scale,
                                                  bool scaled) {
  uint32_t r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = scaled ? f32_to_f16_bits(f16_bits_to_f32(h[e]) * scale) : h[e];
  if constexpr (OUT == NPAMD_F16) {
    *reinterpret_cast<u32x4*>((uint16_t*)out + at) =
        u32x4{r[0] | (r[1] << 16), r[2] | (r[3] << 16), r[4] | (r[5] << 16), r[6] | (r[7] << 16)};
  } else if constexpr (OUT == NPAMD_BF16) {
    uint32_t b[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = f32_to_bf16_bits(f16_bits_to_f32(r[e]));
    *reinterpret_cast<u32x4*>((uint16_t*)out + at) =
        u32x4{b[0] | (b[1] << 16), b[2] | (b[3] << 16), b[4] | (b[5] << 16), b[6] | (b[7] << 16)};
  } else {
    float* o = (float*)out + at;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f16_bits_to_f32(r[e]);
  }
}

// VL = 8: a block takes one token's columns (blockIdx.y: VPT vectors of eight per thread; short rows share a
// block), so no thread divides 64-bit numbers; a thread's VPT table indices are asked for together, then its codebook rows.  Bound, with a
// codebook larger than L1, by the L2's requests and the chain id -> index row -> codebook row (4096 tokens x 4096, 65536
// rows: 15.5-17 us, 11 of them the requests; waves wait 71 % of their time), else by the output stream.  An eighth of the tokens to each die: whoever
// reads the rows next (a norm deals them the same way) finds them in its own L2.
template <int OUT, bool PERM, int VPT>
__global__ void __launch_bounds__(256)
vq_embedding_vl8_kernel(const int64_t* __restrict__ ids, int64_t n_ids, const uint16_t* __restrict__ idx,
                        int64_t vocab, int groups, const uint16_t* __restrict__ cb, uint32_t nc_minus_1,
                        const int32_t* __restrict__ inv_perm, float scale, bool scaled, void* __restrict__ out, unsigned lanes,
                        unsigned tokens, unsigned per_die) {
  int64_t t;
  int col;
  if (!token_of_thread(lanes, tokens, per_die, &t, &col) || t >= n_ids) return;
  int64_t tok = ids[t];
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);  // ids are clamped, never followed out of the table
  const uint16_t* trow = idx + tok * groups;
  const int step = (int)lanes, g0 = blockIdx.y * step * VPT + col;
  if constexpr (PERM) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const int g8 = g0 + step * j;
      if (g8 >= groups) return;
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int src = inv_perm[g8 * 8 + e];
        const uint32_t c = min((uint32_t)trow[src >> 3], nc_minus_1);
        h[e] = cb[(int64_t)c * 8 + (src & 7)];
      }
      store_embedding8<OUT>(out, (t * groups + g8) * 8, h, scale, scaled);
    }
  } else {
    u32x4 v[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j)  // columns past the end look up the last one and are not stored
      v[j] = *reinterpret_cast<const u32x4*>(cb + (int64_t)min((uint32_t)trow[min(g0 + step * j, groups - 1)], nc_minus_1) * 8);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (g0 + step * j >= groups) return;
      uint32_t h[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        h[2 * e] = v[j][e] & 0xFFFFu;
        h[2 * e + 1] = v[j][e] >> 16;
      }
      store_embedding8<OUT>(out, (t * groups + g0 + step * j) * 8, h, scale, scaled);
    }
  }
}

// Any vector length: one thread per output element.
template <int OUT>
__global__ void __launch_bounds__(256)
vq_embedding_generic_kernel(const int64_t* __restrict__ ids, int64_t n_ids, const uint16_t* __restrict__ idx,
                            int64_t vocab, int groups, int vl, const uint16_t* __restrict__ cb, uint32_t nc_minus_1,
                            const int32_t* __restrict__ inv_perm, float scale, bool scaled, void* __restrict__ out) {
  const int dim = groups * vl;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_ids * dim) return;
  const int64_t t = i / dim;
  const int j = (int)(i - t * dim);
  int64_t tok = ids[t];
  tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  const int src = inv_perm ? inv_perm[j] : j;
  const uint32_t c = min((uint32_t)idx[tok * groups + src / vl], nc_minus_1);
  uint32_t h = cb[(int64_t)c * vl + src % vl];
  if (scaled) h = f32_to_f16_bits(f16_bits_to_f32(h) * scale);
  store_from_f16_bits<OUT>(out, i, h);
}

template <int OUT>
int launch_vq_embedding(const int64_t* ids, int64_t n_ids, const uint16_t* idx, int64_t vocab, int groups,
                        const uint16_t* cb, int nc, int vl, const int32_t* inv_perm, float scale, void* out,
                        hipStream_t st) {
  const bool scaled = scale != 1.0f;
  if (vl == 8 && aligned16(cb) && aligned16(out) && n_ids <= 0x7FFFFFF0 && groups <= 256 * 65535) {
    const TokenGrid tg(groups, n_ids, 2);
    const DieGrid rows((n_ids + tg.tokens - 1) / tg.tokens, n_ids * groups * 16, kAuxDieBytes);
    const dim3 grid(rows.blocks, (unsigned)tg.segments);
#define NPAMD_VQ_EMB(PERM, VPT)                                                                                      \
  launch(vq_embedding_vl8_kernel<OUT, PERM, VPT>, grid, tg.threads, 0, st, ids, n_ids, idx, vocab, groups, cb, (uint32_t)nc - 1u, \
                                                                inv_perm, scale, scaled, out, tg.lanes, tg.tokens, rows.per_die)
    if (inv_perm) {
      if (tg.vpt == 2) NPAMD_VQ_EMB(true, 2);
      else NPAMD_VQ_EMB(true, 1);
    } else {
      if (tg.vpt == 2) NPAMD_VQ_EMB(false, 2);
      else NPAMD_VQ_EMB(false, 1);
    }
#undef NPAMD_VQ_EMB
  } else {
    const int64_t n = n_ids * groups * vl;
    launch(vq_embedding_generic_kernel<OUT>, (unsigned)((n + 255) / 256), 256, 0, st,
        ids, n_ids, idx, vocab, groups, vl, cb, (uint32_t)nc - 1u, inv_perm, scale, scaled, out);
  }
  return check_launch("npamd_vq_embedding");
}

// ---------------------------------------------------------------------------
// Group-affine n-bit embedding lookup (n in {1, 2, 4, 8}):
//   v16 = f16((q - zp) * s)          f32 arithmetic, zp = 2^(n-1) without a zero-point tensor
//   v16 = 0 on the padding row
//   out = round_out(cast_out(v16) * embed_scale)   (the multiply only when embed_scale != 1)
// ---------------------------------------------------------------------------
template <int OUT>
__device__ __forceinline__ void store_q_embedding(void* out, int64_t at, float v, float embed_scale, bool scaled) {
  const uint32_t h = f32_to_f16_bits(v);
  if (!scaled) {
    store_from_f16_bits<OUT>(out, at, h);
    return;
  }
  if constexpr (OUT == NPAMD_F16) store_from_f32<OUT>(out, at, f16_bits_to_f32(h) * embed_scale);
  else if constexpr (OUT == NPAMD_BF16)
    store_from_f32<OUT>(out, at, bf16_bits_to_f32(f32_to_bf16_bits(f16_bits_to_f32(h))) * embed_scale);
  else store_from_f32<OUT>(out, at, f16_bits_to_f32(h) * embed_scale);
}

// Eight 4-bit codes without a zero point -> eight fp16 values (q - 8) * s, natural order: byte i of the codes (elements 2 i and
// 2 i + 1) under both halves of a pair, whose exponents read it as (1024 + q, 64 + q); the product of a 4-bit and an
// 11-bit number is rounded once, as the f32 form rounds it.
__device__ __forceinline__ void q4_values8(uint32_t codes, uint32_t s2, uint32_t (&h)[4]) {
#pragma clang fp contract(off)
  const uint32_t spread[4] = {__builtin_amdgcn_perm(0u, codes, 0x0c000c00u), __builtin_amdgcn_perm(0u, codes, 0x0c010c01u),
                              __builtin_amdgcn_perm(0u, codes, 0x0c020c02u), __builtin_amdgcn_perm(0u, codes, 0x0c030c03u)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t pair = (spread[i] & 0x00F0000Fu) | 0x54006400u;
    const f16x2 q = __builtin_bit_cast(f16x2, pair) - __builtin_bit_cast(f16x2, 0x54806408u);
    h[i] = __builtin_bit_cast(uint32_t, q * __builtin_bit_cast(f16x2, s2));
  }
}

// 4-bit codes, group size a multiple of 8: eight elements (one 32-bit load of codes) at a time, VPT of them per thread;
// blocks and dies as for the VQ lookup.  Was bound by its vector instructions (19 per element, 92 % of all issue slots at 4096
// tokens x 4096: 11.6 us): converted two at a time in fp16 where there is no zero point, and the group found by a shift where
// its size allows (group_shift; -1: by a division), 14.0 -> 9.8 us with the pieces per thread of TokenGrid (3.4 TB/s written).
template <int OUT, int VPT, bool ZP>
__global__ void __launch_bounds__(256)
q4_embedding_kernel(const int64_t* __restrict__ ids, int64_t n_ids, const uint8_t* __restrict__ w_pack,
                    const uint16_t* __restrict__ scale, const uint16_t* __restrict__ zp, int octets_per_group, int group_shift,
                    int groups, int64_t vocab, int dim, int64_t padding_idx, float embed_scale, bool scaled,
                    void* __restrict__ out, unsigned lanes, unsigned tokens, unsigned per_die) {
  int64_t t;
  int col;
  if (!token_of_thread(lanes, tokens, per_die, &t, &col) || t >= n_ids) return;
  const int per_row = dim >> 3;
  const int64_t raw = ids[t];
  const int64_t tok = raw < 0 ? 0 : (raw >= vocab ? vocab - 1 : raw);
  const uint32_t* const wrow = reinterpret_cast<const uint32_t*>(w_pack + tok * (dim >> 1));
  const uint16_t* const srow = scale + tok * groups;
  const uint16_t* const zrow = ZP ? zp + tok * groups : nullptr;
  const bool pad = raw == padding_idx;
  uint32_t codes[VPT], s[VPT], z[VPT];
  const int step = (int)lanes, o0 = blockIdx.y * step * VPT + col;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {  // columns past the end repeat the last one and are not stored
    const int o = min(o0 + step * j, per_row - 1);
    const int grp = group_shift >= 0 ? o >> group_shift : o / octets_per_group;
    codes[j] = wrow[o];
    s[j] = srow[grp];
    if constexpr (ZP) z[j] = zrow[grp];
  }
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (o0 + step * j >= per_row) return;
    const int64_t i = t * per_row + o0 + step * j;
    uint32_t h[4];
    if constexpr (ZP) {
      const float sf = f16_bits_to_f32(s[j]), zf = f16_bits_to_f32(z[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = (float)((codes[j] >> (8 * e)) & 0xFu), hi = (float)((codes[j] >> (8 * e + 4)) & 0xFu);
        h[e] = pack2<NPAMD_F16>((lo - zf) * sf, (hi - zf) * sf);
      }
    } else {
      q4_values8(codes[j], s[j] * 0x10001u, h);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = pad ? 0u : h[e];
    if constexpr (OUT == NPAMD_F32) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        store_q_embedding<OUT>(out, i * 8 + e, f16_bits_to_f32(e % 2 ? h[e / 2] >> 16 : h[e / 2] & 0xFFFFu), embed_scale, scaled);
    } else {
      // eight 16-bit results leave as one 16-byte store; same roundings as store_q_embedding
      u32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[e] = OUT == NPAMD_F16 ? h[e] : f16x2_to_bf16x2(h[e]);
        if (scaled) r[e] = pack2<OUT>(act_bits_to_f32<OUT>(r[e] & 0xFFFFu) * embed_scale, act_bits_to_f32<OUT>(r[e] >> 16) * embed_scale);
      }
      *reinterpret_cast<u32x4*>((uint16_t*)out + i * 8) = r;
    }
  }
}

template <int OUT>
__global__ void __launch_bounds__(256)
q_embedding_generic_kernel(const int64_t* __restrict__ ids, int64_t n_ids, const uint8_t* __restrict__ w_pack,
                           const uint16_t* __restrict__ scale, const uint16_t* __restrict__ zp, int nbits,
                           int group_size, int64_t vocab, int dim, int64_t padding_idx, float embed_scale,
                           bool scaled, void* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_ids * dim) return;
  const int64_t t = i / dim;
  const int j = (int)(i - t * dim);
  const int64_t raw = ids[t];
  const int64_t tok = raw < 0 ? 0 : (raw >= vocab ? vocab - 1 : raw);
  const int vpb = 8 / nbits;
  const uint32_t byte = w_pack[tok * (dim / vpb) + j / vpb];
  const float q = (float)((byte >> ((j % vpb) * nbits)) & ((1u << nbits) - 1u));
  const int64_t grp = tok * (dim / group_size) + j / group_size;
  const float z = zp ? f16_bits_to_f32(zp[grp]) : (float)(1 << (nbits - 1));
  const float v = raw == padding_idx ? 0.f : (q - z) * f16_bits_to_f32(scale[grp]);
  store_q_embedding<OUT>(out, i, v, embed_scale, scaled);
}

template <int OUT>
int launch_q_embedding(const int64_t* ids, int64_t n_ids, const uint8_t* w_pack, const uint16_t* scale,
                       const uint16_t* zp, int nbits, int group_size, int64_t vocab, int dim, int64_t padding_idx,
                       float embed_scale, void* out, hipStream_t st) {
  const bool scaled = embed_scale != 1.0f;
  if (nbits == 4 && group_size % 8 == 0 && dim % 8 == 0 && (reinterpret_cast<uintptr_t>(w_pack) & 3) == 0 &&
      aligned16(out) && n_ids <= 0x7FFFFFF0) {
    const TokenGrid tg(dim / 8, n_ids, zp ? 2 : 8);
    const DieGrid rows((n_ids + tg.tokens - 1) / tg.tokens, n_ids * dim * 2, kAuxDieBytes);
    const dim3 grid(rows.blocks, (unsigned)tg.segments);
    const int octets = group_size / 8, shift = (octets & (octets - 1)) == 0 ? __builtin_ctz((unsigned)octets) : -1;
#define NPAMD_Q4_EMB(VPT, ZP)                                                                                            \
  launch(q4_embedding_kernel<OUT, VPT, ZP>, grid, tg.threads, 0, st, ids, n_ids, w_pack, scale, zp, octets, shift, dim / group_size, \
         vocab, dim, padding_idx, embed_scale, scaled, out, tg.lanes, tg.tokens, rows.per_die)
    if (zp) {
      if (tg.vpt == 2) NPAMD_Q4_EMB(2, true);
      else NPAMD_Q4_EMB(1, true);
    } else {
      if (tg.vpt == 8) NPAMD_Q4_EMB(8, false);
      else if (tg.vpt == 4) NPAMD_Q4_EMB(4, false);
      else if (tg.vpt == 2) NPAMD_Q4_EMB(2, false);
      else NPAMD_Q4_EMB(1, false);
    }
#undef NPAMD_Q4_EMB
  } else {
    const int64_t n = n_ids * dim;
    launch(q_embedding_generic_kernel<OUT>, (unsigned)((n + 255) / 256), 256, 0, st,
        ids, n_ids, w_pack, scale, zp, nbits, group_size, vocab, dim, padding_idx, embed_scale, scaled, out);
  }
  return check_launch("npamd_q_embedding");
}

// The gather of gather_columns.hpp, one block's share per block.
template <bool PERM, bool LDS, int ROWS>
__global__ void __launch_bounds__(256)
gather_columns_kernel(const uint16_t* __restrict__ x, int64_t ldx, const int32_t* __restrict__ perm,
                      uint16_t* __restrict__ out, int64_t ldo, int M, int K, bool vec, bool perm_vec) {
  extern __shared__ __attribute__((aligned(16))) uint16_t row_lds[];
  gather_columns_block<PERM, LDS, ROWS>(x, ldx, perm, out, ldo, M, K, vec, perm_vec, blockIdx.x, gridDim.x, blockIdx.y, row_lds);
}

}  // namespace

extern "C" int npamd_gather_columns(const void* x, int64_t ldx, const int32_t* perm, void* out, int64_t ldo, int M, int K,
                                    void* stream) {
  NPAMD_REQUIRE(M >= 0 && K >= 0 && ldx >= K && ldo >= K, "npamd_gather_columns: bad shape [%d, %d]", M, K);
  NPAMD_REQUIRE(ldo % 8 == 0 && ldo <= 0x7FFFFFFF - 2048, "npamd_gather_columns: output row stride must be a multiple of 8");
  if (M == 0 || ldo == 0) return NPAMD_OK;
  NPAMD_REQUIRE(x && out && aligned16(out), "npamd_gather_columns: null or unaligned pointer");
  hipStream_t st = (hipStream_t)stream;
  const bool vec = aligned16(x) && ldx % 8 == 0;
  auto xs = (const uint16_t*)x;
  auto os = (uint16_t*)out;
  const bool pv = aligned16(perm);
  for (int m0 = 0; m0 < M; m0 += 65534) {
    const int rows = M - m0 < 65534 ? M - m0 : 65534;
    GatherPlan plan(perm != nullptr, ldo, M, K);
    const dim3 grid(plan.segments, (unsigned)(plan.pair ? (rows + 1) / 2 : rows));
    const uint16_t* xm = xs + (int64_t)m0 * ldx;
    uint16_t* om = os + (int64_t)m0 * ldo;
    const auto go = [&](auto kernel) { launch(kernel, grid, 256, plan.lds_bytes, st, xm, ldx, perm, om, ldo, rows, K, vec, pv); };
    if (!perm) go(gather_columns_kernel<false, false, 1>);
    else if (plan.pair) go(gather_columns_kernel<true, true, 2>);
    else if (plan.lds) go(gather_columns_kernel<true, true, 1>);
    else go(gather_columns_kernel<true, false, 1>);
  }
  return check_launch("npamd_gather_columns");
}

extern "C" int npamd_rms_norm(const void* x, int64_t ldx, const void* weight, void* out, int64_t ldo, int M, int H,
                              float eps, int dtype, void* stream) {
  NPAMD_REQUIRE(dtype == NPAMD_F16 || dtype == NPAMD_BF16 || dtype == NPAMD_F32, "npamd_rms_norm: bad dtype code %d",
                dtype);
  NPAMD_REQUIRE(M >= 0 && H >= 1, "npamd_rms_norm: bad shape [%d, %d]", M, H);
  NPAMD_REQUIRE(ldx >= H && ldo >= H, "npamd_rms_norm: row stride smaller than the row");
  if (M == 0) return NPAMD_OK;
  NPAMD_REQUIRE(x && weight && out, "npamd_rms_norm: null pointer");
  hipStream_t st = (hipStream_t)stream;
  if (dtype == NPAMD_F16) return launch_rms_norm<NPAMD_F16>(x, ldx, weight, out, ldo, M, H, eps, st);
  if (dtype == NPAMD_BF16) return launch_rms_norm<NPAMD_BF16>(x, ldx, weight, out, ldo, M, H, eps, st);
  return launch_rms_norm<NPAMD_F32>(x, ldx, weight, out, ldo, M, H, eps, st);
}

extern "C" int npamd_vq_embedding(const int64_t* ids, int64_t n_ids, const int16_t* indices, int64_t vocab, int groups,
                                  const void* codebook_f16, int nc, int vl, const int32_t* inv_perm, float scale,
                                  void* out, int out_dtype, void* stream) {
  NPAMD_REQUIRE(out_dtype == NPAMD_F16 || out_dtype == NPAMD_BF16 || out_dtype == NPAMD_F32,
                "npamd_vq_embedding: bad dtype code %d", out_dtype);
  NPAMD_REQUIRE(n_ids >= 0 && vocab >= 1 && groups >= 1 && nc >= 1 && vl >= 1, "npamd_vq_embedding: bad shape");
  NPAMD_REQUIRE(nc <= 65536, "npamd_vq_embedding: the index table holds 16-bit indices, codebook has %d rows", nc);
  if (n_ids == 0) return NPAMD_OK;
  NPAMD_REQUIRE(ids && indices && codebook_f16 && out, "npamd_vq_embedding: null pointer");
  hipStream_t st = (hipStream_t)stream;
  auto idx = (const uint16_t*)indices;
  auto cb = (const uint16_t*)codebook_f16;
  if (out_dtype == NPAMD_F16)
    return launch_vq_embedding<NPAMD_F16>(ids, n_ids, idx, vocab, groups, cb, nc, vl, inv_perm, scale, out, st);
  if (out_dtype == NPAMD_BF16)
    return launch_vq_embedding<NPAMD_BF16>(ids, n_ids, idx, vocab, groups, cb, nc, vl, inv_perm, scale, out, st);
  return launch_vq_embedding<NPAMD_F32>(ids, n_ids, idx, vocab, groups, cb, nc, vl, inv_perm, scale, out, st);
}

extern "C" int npamd_q_embedding(const int64_t* ids, int64_t n_ids, const uint8_t* w_pack, const void* scale_f16,
                                 const void* zero_point_f16, int nbits, int group_size, int64_t vocab, int dim,
                                 int64_t padding_idx, float embed_scale, void* out, int out_dtype, void* stream) {
  NPAMD_REQUIRE(out_dtype == NPAMD_F16 || out_dtype == NPAMD_BF16 || out_dtype == NPAMD_F32,
                "npamd_q_embedding: bad dtype code %d", out_dtype);
  NPAMD_REQUIRE(nbits == 1 || nbits == 2 || nbits == 4 || nbits == 8, "npamd_q_embedding: nbits must be 1, 2, 4 or 8");
  NPAMD_REQUIRE(n_ids >= 0 && vocab >= 1 && dim >= 1 && group_size >= 1 && dim % group_size == 0 &&
                    dim % (8 / nbits) == 0,
                "npamd_q_embedding: bad shape (dim %d, group size %d)", dim, group_size);
  if (n_ids == 0) return NPAMD_OK;
  NPAMD_REQUIRE(ids && w_pack && scale_f16 && out, "npamd_q_embedding: null pointer");
  hipStream_t st = (hipStream_t)stream;
  auto sc = (const uint16_t*)scale_f16;
  auto zp = (const uint16_t*)zero_point_f16;
  if (out_dtype == NPAMD_F16)
    return launch_q_embedding<NPAMD_F16>(ids, n_ids, w_pack, sc, zp, nbits, group_size, vocab, dim, padding_idx,
                                         embed_scale, out, st);
  if (out_dtype == NPAMD_BF16)
    return launch_q_embedding<NPAMD_BF16>(ids, n_ids, w_pack, sc, zp, nbits, group_size, vocab, dim, padding_idx,
                                          embed_scale, out, st);
  return launch_q_embedding<NPAMD_F32>(ids, n_ids, w_pack, sc, zp, nbits, group_size, vocab, dim, padding_idx,
                                       embed_scale, out, st);
}
