// One-pass VQ decode kernels: packed index stream + fp16 codebook -> dense weight.
//
//   out.flat[v*VL + j] = cast(codebook[idx(v), j])
//
// HBM-bound byte work: one thread per vector, coalesced index reads (2 B/lane
// at 16 bits), one 16-byte codebook gather (L2-resident table), one vector
// store.  Traffic = index stream + output; the codebook is read from cache.
#include "common.hpp"
#include "gather_columns.hpp"
#include "../../include/npamd_diag.h"

namespace npamd {

#pragma clang fp contract(off)

// Index of vector v.  BITS is 8 or 16 for the byte-aligned widths, 12 for one two-byte read, 0 for the bounds-checked window
// reader, whose three byte reads show where nothing else is slow (12-bit indices into a table in LDS, 4096 x 4096: 11.7 -> 10.2 us).
template <int BITS>
__device__ __forceinline__ uint32_t vec_index(const uint8_t* __restrict__ packed, int64_t n_bytes,
                                              int64_t v, int bits) {
  if constexpr (BITS == 16) return reinterpret_cast<const uint16_t*>(packed)[v];
  else if constexpr (BITS == 8) return packed[v];
  else if constexpr (BITS == 12) {  // an index lies within two bytes, which need not be aligned
    const int64_t bit = v * 12;
    uint16_t w;
    __builtin_memcpy(&w, packed + (bit >> 3), 2);
    return ((uint32_t)w >> (bit & 7)) & 0xFFFu;
  }
  else return read_index(packed, n_bytes, v, bits);
}

template <int OUT>
__device__ __forceinline__ void store8(void* out, int64_t v, u32x4 c) {
  if constexpr (OUT == NPAMD_F16) {
    reinterpret_cast<u32x4*>(out)[v] = c;
  } else if constexpr (OUT == NPAMD_BF16) {
    reinterpret_cast<u32x4*>(out)[v] = cb_to_act<NPAMD_BF16>(c);
  } else {
    f32x4 lo, hi;
    lo.x = f16_bits_to_f32(c.x & 0xFFFFu); lo.y = f16_bits_to_f32(c.x >> 16);
    lo.z = f16_bits_to_f32(c.y & 0xFFFFu); lo.w = f16_bits_to_f32(c.y >> 16);
    hi.x = f16_bits_to_f32(c.z & 0xFFFFu); hi.y = f16_bits_to_f32(c.z >> 16);
    hi.z = f16_bits_to_f32(c.w & 0xFFFFu); hi.w = f16_bits_to_f32(c.w >> 16);
    reinterpret_cast<f32x4*>(out)[2 * v] = lo;
    reinterpret_cast<f32x4*>(out)[2 * v + 1] = hi;
  }
}

// VL = 8: one 16-byte gather and one vector store per thread.
template <int BITS, int OUT>
__global__ void __launch_bounds__(256)
vq_dequant_vl8_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                      const u32x4* __restrict__ codebook, uint32_t nc, void* __restrict__ out,
                      int64_t n_vectors, unsigned per_die) {
  const int64_t v = die_block(blockIdx.x, per_die) * 256 + threadIdx.x;
  if (v >= n_vectors) return;
  // An index past the codebook is clamped to the last row so a corrupt stream
  // cannot read outside the table.
  const uint32_t idx = min(vec_index<BITS>(packed, n_bytes, v, bits), nc - 1u);
  store8<OUT>(out, v, codebook[idx]);
}

// The same decode and, in the blocks in front of it, the gather of the activations its product reads (gather_columns.hpp):
// both are short and wait for memory most of their time, and neither needs the other (77 x 2184 permuted and 3003 x 2240
// decoded: 2.7 + 5.1 us one behind the other).
template <int BITS, int OUT, bool PERM>
__global__ void __launch_bounds__(256)
vq_dequant_gather_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                         const u32x4* __restrict__ codebook, uint32_t nc, void* __restrict__ out,
                         int64_t n_vectors, unsigned per_die, const uint16_t* __restrict__ x, int64_t ldx,
                         const int32_t* __restrict__ perm, uint16_t* __restrict__ xo, int64_t ldo, int M, int K, bool vec,
                         bool perm_vec, unsigned segments, unsigned gather_blocks) {
  extern __shared__ __attribute__((aligned(16))) uint16_t row_lds[];
  if (blockIdx.x < gather_blocks) {
    const unsigned row = blockIdx.x / segments;
    if (row < (unsigned)M)
      gather_columns_block<PERM, PERM, 1>(x, ldx, perm, xo, ldo, M, K, vec, perm_vec, blockIdx.x % segments, segments, row, row_lds);
    return;
  }
  const int64_t v = die_block(blockIdx.x - gather_blocks, per_die) * 256 + threadIdx.x;
  if (v >= n_vectors) return;
  store8<OUT>(out, v, codebook[min(vec_index<BITS>(packed, n_bytes, v, bits), nc - 1u)]);
}

// VL = 4: two vectors per thread -- two 8-byte gathers, one 16-byte (f32: 32-byte) store.
template <int OUT>
__device__ __forceinline__ void store4x2(void* out, int64_t v0, u32x2 c0, u32x2 c1, bool both) {
  if (both) {
    store8<OUT>(out, v0 >> 1, u32x4{c0.x, c0.y, c1.x, c1.y});  // v0 is even: 8 values = one store8 unit
  } else if constexpr (OUT == NPAMD_F16) {
    reinterpret_cast<u32x2*>(out)[v0] = c0;
  } else if constexpr (OUT == NPAMD_BF16) {
    reinterpret_cast<u32x2*>(out)[v0] = u32x2{f16x2_to_bf16x2(c0.x), f16x2_to_bf16x2(c0.y)};
  } else {
    reinterpret_cast<f32x4*>(out)[v0] = f32x4{f16_bits_to_f32(c0.x & 0xFFFFu), f16_bits_to_f32(c0.x >> 16),
                                              f16_bits_to_f32(c0.y & 0xFFFFu), f16_bits_to_f32(c0.y >> 16)};
  }
}

template <int BITS, int OUT>
__global__ void __launch_bounds__(256)
vq_dequant_vl4_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                      const u32x2* __restrict__ codebook, uint32_t nc, void* __restrict__ out,
                      int64_t n_vectors, unsigned per_die) {
  const int64_t v0 = (die_block(blockIdx.x, per_die) * 256 + threadIdx.x) * 2;
  if (v0 >= n_vectors) return;
  const bool both = v0 + 1 < n_vectors;
  const u32x2 c0 = codebook[min(vec_index<BITS>(packed, n_bytes, v0, bits), nc - 1u)];
  const u32x2 c1 = codebook[min(vec_index<BITS>(packed, n_bytes, both ? v0 + 1 : v0, bits), nc - 1u)];
  store4x2<OUT>(out, v0, c0, c1, both);
}

// VL = 8 or 4, a table of 16 to 64 KiB copied into LDS first.  Such a table overflows or fills
// the 32 KiB vector L1, so gathers from memory run at the L1-miss rate (36 us for a
// 14336 x 4096 layer with 4096 rows of 16 bytes, the same as a 65536-row table); from LDS the
// kernel is bound by the store stream.  Two blocks of 1024 threads per compute unit, each
// decoding a contiguous run of vectors.
template <int BITS, int OUT, int VL>
__global__ void __launch_bounds__(1024)
vq_dequant_lds_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                      const u32x4* __restrict__ codebook, uint32_t nc, void* __restrict__ out,
                      int64_t n_vectors, int64_t vectors_per_block, unsigned per_die) {
  extern __shared__ __attribute__((aligned(16))) u32x4 cb_lds[];
  const uint32_t vec16 = VL == 8 ? nc : (nc + 1) / 2;  // the allocation behind an odd VL = 4 table is not read past:
  for (uint32_t i = threadIdx.x; i < vec16; i += 1024) {  // its last half-filled unit is fetched as 8 bytes
    if (VL == 4 && (nc & 1) && i == vec16 - 1) {
      const u32x2 t = reinterpret_cast<const u32x2*>(codebook)[nc - 1];
      cb_lds[i] = u32x4{t.x, t.y, 0u, 0u};
    } else {
      cb_lds[i] = codebook[i];
    }
  }
  __syncthreads();
  const int64_t begin = die_block(blockIdx.x, per_die) * vectors_per_block;
  const int64_t end = min(begin + vectors_per_block, n_vectors);
  if constexpr (VL == 8) {
    for (int64_t v = begin + threadIdx.x; v < end; v += 1024) {
      const uint32_t idx = min(vec_index<BITS>(packed, n_bytes, v, bits), nc - 1u);
      store8<OUT>(out, v, cb_lds[idx]);
    }
  } else {
    // two vectors per thread (a run starts at an even vector: vectors_per_block is a multiple of 1024)
    const u32x2* cb2 = reinterpret_cast<const u32x2*>(cb_lds);
    for (int64_t v0 = begin + 2 * threadIdx.x; v0 < end; v0 += 2048) {
      const bool both = v0 + 1 < end;
      const u32x2 c0 = cb2[min(vec_index<BITS>(packed, n_bytes, v0, bits), nc - 1u)];
      const u32x2 c1 = cb2[min(vec_index<BITS>(packed, n_bytes, both ? v0 + 1 : v0, bits), nc - 1u)];
      store4x2<OUT>(out, v0, c0, c1, both);
    }
  }
}

// Any VL: scalar copy of the codebook row.
template <int OUT>
__global__ void __launch_bounds__(256)
vq_dequant_generic_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                          const uint16_t* __restrict__ codebook, uint32_t nc,
                          void* __restrict__ out, int64_t n_vectors, int vl) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= n_vectors) return;
  const uint32_t idx = min(read_index(packed, n_bytes, v, bits), nc - 1u);
  const uint16_t* c = codebook + (int64_t)idx * vl;
  for (int j = 0; j < vl; ++j) store_from_f16_bits<OUT>(out, v * vl + j, c[j]);
}

__global__ void __launch_bounds__(256)
vq_widen_u16_kernel(const uint8_t* __restrict__ packed, int64_t n_bytes, int bits,
                    int64_t n_indices, uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_indices) return;
  out[i] = (uint16_t)read_index(packed, n_bytes, i, bits);
}

// Residual VQ: three separately rounded fp16 operations per element.
__device__ __forceinline__ uint32_t rvq_elem(uint32_t cm, uint32_t cr, bool has_s, _Float16 s,
                                             bool has_b, _Float16 b) {
  _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)cm) + __builtin_bit_cast(_Float16, (uint16_t)cr);
  if (has_s) h = h * s;
  if (has_b) h = h + b;
  return (uint32_t)__builtin_bit_cast(uint16_t, h);
}

template <int OUT>
__global__ void __launch_bounds__(256)
rvq_dequant_kernel(const uint8_t* __restrict__ pm, int64_t nbm, int bits_m,
                   const uint8_t* __restrict__ pr, int64_t nbr, int bits_r,
                   const uint16_t* __restrict__ cbm, uint32_t ncm,
                   const uint16_t* __restrict__ cbr, uint32_t ncr,
                   const uint16_t* __restrict__ row_scale, const uint16_t* __restrict__ row_bias,
                   int vl, int64_t groups, int64_t n_vectors, void* __restrict__ out) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= n_vectors) return;
  const uint32_t im = min(read_index(pm, nbm, v, bits_m), ncm - 1u);
  const uint32_t ir = min(read_index(pr, nbr, v, bits_r), ncr - 1u);
  const int64_t n = v / groups;
  const bool has_s = row_scale != nullptr, has_b = row_bias != nullptr;
  const _Float16 s = has_s ? __builtin_bit_cast(_Float16, row_scale[n]) : (_Float16)1.0f;
  const _Float16 b = has_b ? __builtin_bit_cast(_Float16, row_bias[n]) : (_Float16)0.0f;
  const uint16_t* cm = cbm + (int64_t)im * vl;
  const uint16_t* cr = cbr + (int64_t)ir * vl;
  for (int j = 0; j < vl; ++j)
    store_from_f16_bits<OUT>(out, v * vl + j, rvq_elem(cm[j], cr[j], has_s, s, has_b, b));
}

// VL = 8: two 16-byte gathers, packed fp16 arithmetic (each operation rounds per element, like
// the scalar form), one vector store, VPT of them per thread.  Grid = (row, 256 VPT groups of the row): no division.  Two
// vectors per thread keep more lookups on their way where there are many (14336 x 4096 33.5 -> 30.0 us, 4096 x 4096 12.8 -> 11.7; 3003 x
// 2240 7.4 -> 7.8; four 34.5 and 13.9).
__device__ __forceinline__ u32x4 rvq_combine8(const u32x4& a, const u32x4& r, bool has_s, uint32_t s2, bool has_b, uint32_t b2) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t am = a[i], rr = r[i];
    f16x2 h = __builtin_bit_cast(f16x2, am) + __builtin_bit_cast(f16x2, rr);
    if (has_s) h = h * __builtin_bit_cast(f16x2, s2);
    if (has_b) h = h + __builtin_bit_cast(f16x2, b2);
    o[i] = __builtin_bit_cast(uint32_t, h);
  }
  return o;
}

template <int BITS_M, int BITS_R, int OUT, int VPT>
__global__ void __launch_bounds__(256)
rvq_dequant_vl8_kernel(const uint8_t* __restrict__ pm, int64_t nbm, int bits_m,
                       const uint8_t* __restrict__ pr, int64_t nbr, int bits_r,
                       const u32x4* __restrict__ cbm, uint32_t ncm, const u32x4* __restrict__ cbr, uint32_t ncr,
                       const uint16_t* __restrict__ row_scale, const uint16_t* __restrict__ row_bias,
                       int rows, int groups, unsigned per_die, void* __restrict__ out) {
  const int n = (int)die_block(blockIdx.x, per_die);
  const int g0 = blockIdx.y * (256 * VPT) + threadIdx.x;
  if (n >= rows || g0 >= groups) return;
  const int64_t row = (int64_t)n * groups;
  uint32_t im[VPT], ir[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {  // columns past the end look up the last one and are not stored
    const int64_t v = row + min(g0 + 256 * j, groups - 1);
    im[j] = min(vec_index<BITS_M>(pm, nbm, v, bits_m), ncm - 1u);
    ir[j] = min(vec_index<BITS_R>(pr, nbr, v, bits_r), ncr - 1u);
  }
  u32x4 a[VPT], r[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    a[j] = cbm[im[j]];
    r[j] = cbr[ir[j]];
  }
  const bool has_s = row_scale != nullptr, has_b = row_bias != nullptr;
  const uint32_t s2 = has_s ? (uint32_t)row_scale[n] * 0x10001u : 0u;
  const uint32_t b2 = has_b ? (uint32_t)row_bias[n] * 0x10001u : 0u;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (g0 + 256 * j < groups) store8<OUT>(out, row + g0 + 256 * j, rvq_combine8(a[j], r[j], has_s, s2, has_b, b2));
}

// The same on large layers whose main table (16 to 64 KiB) and residual table (up to 16 KiB) fit LDS, copied there first: a
// lookup costs the vector memory path about a cycle per lane whether it hits or not.  Two blocks of 1024 threads per compute
// unit, each a contiguous run of vectors, two per thread at a time; the row of a vector moves on without a division.  4096
// rows, 12-bit indices read in one piece, from memory / from LDS: 14336 x 4096 31.8 / 26.1 us (45.7 with the window reader),
// 4096 x 4096 12.7 / 12.2 (17.1).  The residual table alone in LDS, beside a main table in memory: 33.2 / 30.1 with Zipf indices,
// 41.8 / 43.4 with uniform ones: not taken.
template <int BITS_M, int BITS_R, int OUT>
__global__ void __launch_bounds__(1024)
rvq_dequant_vl8_lds_kernel(const uint8_t* __restrict__ pm, int64_t nbm, int bits_m,
                           const uint8_t* __restrict__ pr, int64_t nbr, int bits_r,
                           const u32x4* __restrict__ cbm, uint32_t ncm, const u32x4* __restrict__ cbr, uint32_t ncr,
                           const uint16_t* __restrict__ row_scale, const uint16_t* __restrict__ row_bias,
                           uint32_t groups, uint32_t n_vectors, uint32_t vectors_per_block, unsigned per_die,
                           void* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) u32x4 cb_lds[];
  u32x4* const main_lds = cb_lds + ncr;
  for (uint32_t i = threadIdx.x; i < ncr; i += 1024) cb_lds[i] = cbr[i];
  for (uint32_t i = threadIdx.x; i < ncm; i += 1024) main_lds[i] = cbm[i];
  __syncthreads();
  const int64_t begin = die_block(blockIdx.x, per_die) * vectors_per_block;
  if (begin >= n_vectors) return;
  const uint32_t end = (uint32_t)min(begin + vectors_per_block, (int64_t)n_vectors);
  const bool has_s = row_scale != nullptr, has_b = row_bias != nullptr;
  const uint32_t q = 1024u / groups, rest = 1024u % groups;  // what 1024 vectors further on means in rows and groups
  uint32_t v = (uint32_t)begin + threadIdx.x, n = v / groups, g = v % groups;
  const auto advance = [&] {
    v += 1024u;
    n += q;
    g += rest;
    if (g >= groups) {
      g -= groups;
      ++n;
    }
  };
  while (v < end) {
    uint32_t im[2], ir[2], s2[2], b2[2], at[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      at[j] = v;
      const bool in = v < end;
      const uint32_t vv = in ? v : end - 1, nn = in ? n : (end - 1) / groups;
      im[j] = min(vec_index<BITS_M>(pm, nbm, vv, bits_m), ncm - 1u);
      ir[j] = min(vec_index<BITS_R>(pr, nbr, vv, bits_r), ncr - 1u);
      s2[j] = has_s ? (uint32_t)row_scale[nn] * 0x10001u : 0u;
      b2[j] = has_b ? (uint32_t)row_bias[nn] * 0x10001u : 0u;
      advance();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (at[j] < end) store8<OUT>(out, at[j], rvq_combine8(main_lds[im[j]], cb_lds[ir[j]], has_s, s2[j], has_b, b2[j]));
  }
}

template <int OUT>
static int launch_vq_dequant(const uint8_t* packed, int64_t n_bytes, int bits, const void* cb,
                             uint32_t nc, int vl, int64_t n_vectors, void* out, hipStream_t st) {
  const unsigned blocks = (unsigned)((n_vectors + 255) / 256);
  const int64_t bytes = n_vectors * vl * (OUT == NPAMD_F32 ? 4 : 2);
  const DieGrid grid(blocks, bytes);
  const bool cb_aligned = (reinterpret_cast<uintptr_t>(cb) % 16) == 0;
  const bool out_aligned = (reinterpret_cast<uintptr_t>(out) % 16) == 0;
  // Tables of 16 to 64 KiB on layers large enough to pay for one copy per block.
  const int64_t table_bytes = (int64_t)nc * vl * 2;
  if ((vl == 8 || vl == 4) && cb_aligned && out_aligned && table_bytes > 16 * 1024 && table_bytes <= 64 * 1024 &&
      n_vectors >= (1 << 20)) {
    const u32x4* c = reinterpret_cast<const u32x4*>(cb);
    const int lds = (int)((table_bytes + 15) / 16 * 16);
    const int64_t per_block = ((n_vectors + 511) / 512 + 1023) / 1024 * 1024;
    const DieGrid grid((n_vectors + per_block - 1) / per_block, bytes);
    const bool b16 = bits == 16 && (reinterpret_cast<uintptr_t>(packed) % 2) == 0;
#define NPAMD_VQ_LDS(B, V) \
  launch(vq_dequant_lds_kernel<B, OUT, V>, grid.blocks, 1024, lds, st, packed, n_bytes, bits, c, nc, out, n_vectors, per_block, grid.per_die)
    if (vl == 8) {
      if (b16) NPAMD_VQ_LDS(16, 8);
      else if (bits == 12) NPAMD_VQ_LDS(12, 8);
      else NPAMD_VQ_LDS(0, 8);
    } else {
      if (b16) NPAMD_VQ_LDS(16, 4);
      else NPAMD_VQ_LDS(0, 4);
    }
#undef NPAMD_VQ_LDS
    return check_launch("npamd_vq_dequant");
  }
  if (vl == 8 && cb_aligned && out_aligned) {
    const u32x4* c = reinterpret_cast<const u32x4*>(cb);
    if (bits == 16 && (reinterpret_cast<uintptr_t>(packed) % 2) == 0)
      launch(vq_dequant_vl8_kernel<16, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
    else if (bits == 8)
      launch(vq_dequant_vl8_kernel<8, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
    else
      launch(vq_dequant_vl8_kernel<0, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
  } else if (vl == 4 && (reinterpret_cast<uintptr_t>(cb) % 8) == 0 && out_aligned) {
    const u32x2* c = reinterpret_cast<const u32x2*>(cb);
    const DieGrid grid(((n_vectors + 1) / 2 + 255) / 256, bytes);  // two vectors per thread
    if (bits == 16 && (reinterpret_cast<uintptr_t>(packed) % 2) == 0)
      launch(vq_dequant_vl4_kernel<16, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
    else if (bits == 8)
      launch(vq_dequant_vl4_kernel<8, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
    else
      launch(vq_dequant_vl4_kernel<0, OUT>, grid.blocks, 256, 0, st, packed, n_bytes, bits, c, nc, out, n_vectors, grid.per_die);
  } else {
    launch(vq_dequant_generic_kernel<OUT>, blocks, 256, 0, st,
        packed, n_bytes, bits, reinterpret_cast<const uint16_t*>(cb), nc, out, n_vectors, vl);
  }
  return check_launch("npamd_vq_dequant");
}

// LUT gather: y[m, j] = sum over groups g of lut[m, g, idx(j, g)], float32.
// One wave per output row j: lane l takes groups l, l + 64, ... (consecutive indices of the
// stream), the 64 partial sums are added pairwise across the wave in a fixed order.
// blockIdx.y = token.
__global__ void __launch_bounds__(256) vq_lut_gather_kernel(const float* __restrict__ lut,
                                                             const uint8_t* __restrict__ packed, int64_t n_bytes,
                                                             int bits, float* __restrict__ y, int N, int groups,
                                                             int nc) {
  const int lane = threadIdx.x & 63;
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (j >= N) return;
  const float* lut_m = lut + (int64_t)blockIdx.y * groups * nc;
  float acc = 0.f;
  for (int g = lane; g < groups; g += 64) {
    uint32_t c = read_index(packed, n_bytes, (int64_t)j * groups + g, bits);
    if (c > (uint32_t)nc - 1u) c = (uint32_t)nc - 1u;  // same clamp as the decode kernels
    acc += lut_m[(int64_t)g * nc + c];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if (lane == 0) y[(int64_t)blockIdx.y * N + j] = acc;
}

}  // namespace npamd

using namespace npamd;

extern "C" int npamd_vq_dequant(const uint8_t* packed, int64_t n_bytes, int bits,
                                const void* codebook_f16, int nc, int vl, int64_t n_vectors,
                                void* out, int out_dtype, void* stream) {
  NPAMD_REQUIRE(bits >= 4 && bits <= 20, "npamd_vq_dequant: bits must be in [4, 20], got %d", bits);
  NPAMD_REQUIRE(vl >= 1 && nc >= 1, "npamd_vq_dequant: bad codebook shape [%d, %d]", nc, vl);
  NPAMD_REQUIRE(n_vectors >= 0, "npamd_vq_dequant: negative n_vectors");
  NPAMD_REQUIRE((n_vectors * bits + 7) / 8 <= n_bytes,
                "npamd_vq_dequant: packed buffer too short for %lld indices of %d bits",
                (long long)n_vectors, bits);
  if (n_vectors == 0) return NPAMD_OK;
  NPAMD_REQUIRE(packed && codebook_f16 && out, "npamd_vq_dequant: null pointer");
  NPAMD_REQUIRE(n_vectors <= (int64_t)0x7FFFFFFF * 256, "npamd_vq_dequant: too many vectors");
  hipStream_t st = (hipStream_t)stream;
  switch (out_dtype) {
    case NPAMD_F16: return launch_vq_dequant<NPAMD_F16>(packed, n_bytes, bits, codebook_f16, (uint32_t)nc, vl, n_vectors, out, st);
    case NPAMD_BF16: return launch_vq_dequant<NPAMD_BF16>(packed, n_bytes, bits, codebook_f16, (uint32_t)nc, vl, n_vectors, out, st);
    case NPAMD_F32: return launch_vq_dequant<NPAMD_F32>(packed, n_bytes, bits, codebook_f16, (uint32_t)nc, vl, n_vectors, out, st);
  }
  return fail(NPAMD_ERR_INVALID, "npamd_vq_dequant: out_dtype must be f16, bf16 or f32");
}

// The whole launch has the LDS of a block that gathers: K elements where columns are permuted.  Up to 10240 of them eight blocks,
// all their waves, still fit a compute unit; past that the decoding blocks, which wait for memory, are fewer, and the larger the
// layer the sooner that costs more than a launch.  us with 60 rows, one launch / two: 8-bit indices 4096 x 10240 17.0 / 19.5,
// 4096 x 12288 21.7 / 22.4, 4096 x 14336 27.1 / 25.2, 1024 x 16384 12.2 / 13.2, 4096 x 16384 35.2 / 27.8, 11008 x 16384 125.6 / 105.8;
// 16-bit 4096 x 14336 39.1 / 39.9, 11008 x 12288 134.8 / 134.7, 4096 x 16384 48.6 / 44.8, 11008 x 16384 182.4 / 176.9.
static bool gather_fits_decode(int bits, int64_t n_vectors, int K, bool perm) {
  if (!perm || K <= 10240) return true;
  const int over = K > 12288 ? (K - 12288 + 2047) / 2048 : 0;
  return K <= 16384 && n_vectors <= ((int64_t)(bits == 16 ? 16 : 8) << 20) >> over;
}

extern "C" int npamd_diag_gather_fits_decode(int bits, int64_t n_vectors, int K, int permuted) {
  return gather_fits_decode(bits, n_vectors, K, permuted != 0) ? 1 : 0;
}

extern "C" int npamd_gather_columns(const void* x, int64_t ldx, const int32_t* perm, void* out, int64_t ldo, int M, int K, void* stream);

extern "C" int npamd_vq_dequant_gather(const uint8_t* packed, int64_t n_bytes, int bits, const void* codebook_f16, int nc, int vl,
                                       int64_t n_vectors, void* out, int out_dtype, const void* x, int64_t ldx,
                                       const int32_t* perm, void* x_out, int64_t ldo, int M, int K, void* stream) {
  const auto al = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
  const int64_t table_bytes = (int64_t)nc * vl * 2;
  // Few rows, a decode without a table in LDS: one launch.  Anything else, and whatever has to be refused: the two calls.
  const bool fits = vl == 8 && (out_dtype == NPAMD_F16 || out_dtype == NPAMD_BF16) && (bits == 8 || bits == 12 || bits == 16) &&
                    !(table_bytes > 16 * 1024 && table_bytes <= 64 * 1024 && n_vectors >= (1 << 20)) && n_vectors > 0 &&
                    n_vectors <= (int64_t)1 << 30 && nc >= 1 && (n_vectors * bits + 7) / 8 <= n_bytes && packed && codebook_f16 && out &&
                    al(packed, 2) && al(codebook_f16, 16) && al(out, 16) && x && x_out && al(x_out, 16) && M >= 1 &&
                    M < kGatherPairRows && K >= 1 && K <= 16384 && gather_fits_decode(bits, n_vectors, K, perm != nullptr) && ldx >= K && ldo >= K && ldo % 8 == 0 && ldo <= 32768;
  if (!fits) {
    const int rc = npamd_gather_columns(x, ldx, perm, x_out, ldo, M, K, stream);
    return rc != NPAMD_OK ? rc : npamd_vq_dequant(packed, n_bytes, bits, codebook_f16, nc, vl, n_vectors, out, out_dtype, stream);
  }
  hipStream_t st = (hipStream_t)stream;
  const GatherPlan plan(perm != nullptr, ldo, M, K);
  const unsigned gather_blocks = (plan.segments * plan.row_blocks + 7) / 8 * 8;  // a decoding block stays on its die
  const DieGrid grid((n_vectors + 255) / 256, n_vectors * 16);
  const bool vec = al(x, 16) && ldx % 8 == 0, perm_vec = al(perm, 16);
#define NPAMD_VQ_GATHER(B, OUT, PERM)                                                                                          \
  launch(vq_dequant_gather_kernel<B, OUT, PERM>, gather_blocks + grid.blocks, 256, plan.lds_bytes, st, packed, n_bytes, bits,   \
         (const u32x4*)codebook_f16, (uint32_t)nc, out, n_vectors, grid.per_die, (const uint16_t*)x, ldx, perm, (uint16_t*)x_out, \
         ldo, M, K, vec, perm_vec, plan.segments, gather_blocks)
#define NPAMD_VQ_GATHER_PERM(B, OUT)            \
  do {                                          \
    if (perm) NPAMD_VQ_GATHER(B, OUT, true);    \
    else NPAMD_VQ_GATHER(B, OUT, false);        \
  } while (0)
#define NPAMD_VQ_GATHER_BITS(OUT)                        \
  do {                                                   \
    if (bits == 16) NPAMD_VQ_GATHER_PERM(16, OUT);       \
    else if (bits == 12) NPAMD_VQ_GATHER_PERM(12, OUT);  \
    else NPAMD_VQ_GATHER_PERM(8, OUT);                   \
  } while (0)
  if (out_dtype == NPAMD_F16) NPAMD_VQ_GATHER_BITS(NPAMD_F16);
  else NPAMD_VQ_GATHER_BITS(NPAMD_BF16);
#undef NPAMD_VQ_GATHER_BITS
#undef NPAMD_VQ_GATHER_PERM
#undef NPAMD_VQ_GATHER
  return check_launch("npamd_vq_dequant_gather");
}

extern "C" int npamd_vq_widen_u16(const uint8_t* packed, int64_t n_bytes, int bits,
                                  int64_t n_indices, uint16_t* out, void* stream) {
  NPAMD_REQUIRE(bits >= 4 && bits <= 16, "npamd_vq_widen_u16: bits must be in [4, 16], got %d", bits);
  NPAMD_REQUIRE(n_indices >= 0 && (n_indices * bits + 7) / 8 <= n_bytes,
                "npamd_vq_widen_u16: packed buffer too short");
  if (n_indices == 0) return NPAMD_OK;
  NPAMD_REQUIRE(packed && out, "npamd_vq_widen_u16: null pointer");
  const unsigned blocks = (unsigned)((n_indices + 255) / 256);
  launch(vq_widen_u16_kernel, blocks, 256, 0, (hipStream_t)stream, packed, n_bytes, bits, n_indices, out);
  return check_launch("npamd_vq_widen_u16");
}

extern "C" int npamd_vq_lut_gather(const float* lut, const uint8_t* packed, int64_t n_bytes, int bits,
                                   float* y, int M, int N, int groups, int nc, void* stream) {
  const char* what = "npamd_vq_lut_gather";
  NPAMD_REQUIRE(bits >= 4 && bits <= 20, "%s: bits must be in [4, 20], got %d", what, bits);
  NPAMD_REQUIRE(M >= 0 && N >= 0 && groups >= 1 && nc >= 1, "%s: bad shape M=%d N=%d groups=%d NC=%d", what, M, N,
                groups, nc);
  NPAMD_REQUIRE(((int64_t)N * groups * bits + 7) / 8 <= n_bytes, "%s: packed buffer too short", what);
  NPAMD_REQUIRE(M <= 65535, "%s: at most 65535 tokens per call (got %d)", what, M);
  if (M == 0 || N == 0) return NPAMD_OK;
  NPAMD_REQUIRE(lut && packed && y, "%s: null pointer", what);
  const dim3 grid((unsigned)((N + 3) / 4), (unsigned)M);
  launch(vq_lut_gather_kernel, grid, 256, 0, (hipStream_t)stream, lut, packed, n_bytes, bits, y, N, groups, nc);
  return check_launch(what);
}

extern "C" int npamd_rvq_dequant(const uint8_t* packed_main, int64_t n_bytes_main, int bits_main,
                                 const uint8_t* packed_res, int64_t n_bytes_res, int bits_res,
                                 const void* cb_main_f16, int nc_main, const void* cb_res_f16,
                                 int nc_res, const void* row_scale_f16, const void* row_bias_f16,
                                 int vl, int N, int K, void* out, int out_dtype, void* stream) {
  NPAMD_REQUIRE(bits_main >= 4 && bits_main <= 20 && bits_res >= 4 && bits_res <= 20,
                "npamd_rvq_dequant: bits must be in [4, 20]");
  NPAMD_REQUIRE(vl >= 1 && nc_main >= 1 && nc_res >= 1, "npamd_rvq_dequant: bad codebook shape");
  NPAMD_REQUIRE(N >= 0 && K >= 0 && K % vl == 0, "npamd_rvq_dequant: K=%d not divisible by VL=%d", K, vl);
  const int64_t groups = K / vl, n_vectors = (int64_t)N * groups;
  NPAMD_REQUIRE((n_vectors * bits_main + 7) / 8 <= n_bytes_main &&
                    (n_vectors * bits_res + 7) / 8 <= n_bytes_res,
                "npamd_rvq_dequant: packed buffer too short");
  if (n_vectors == 0) return NPAMD_OK;
  NPAMD_REQUIRE(packed_main && packed_res && cb_main_f16 && cb_res_f16 && out,
                "npamd_rvq_dequant: null pointer");
  const unsigned blocks = (unsigned)((n_vectors + 255) / 256);
  hipStream_t st = (hipStream_t)stream;
  const bool aligned16 = ((reinterpret_cast<uintptr_t>(cb_main_f16) | reinterpret_cast<uintptr_t>(cb_res_f16) |
                           reinterpret_cast<uintptr_t>(out)) % 16) == 0;
  if (vl == 8 && aligned16 && (groups + 255) / 256 <= 65535) {
    const DieGrid rows(N, n_vectors * 8 * (out_dtype == NPAMD_F32 ? 4 : 2));
    const int vpt = n_vectors >= 3 << 19 && groups > 256 ? 2 : 1;
    const dim3 grid(rows.blocks, (unsigned)((groups + 256 * vpt - 1) / (256 * vpt)));
    const bool m16 = bits_main == 16 && (reinterpret_cast<uintptr_t>(packed_main) % 2) == 0;
    const bool r8 = bits_res == 8;
    const int64_t main_bytes = (int64_t)nc_main * 16, res_bytes = (int64_t)nc_res * 16;
    if (r8 && (m16 || bits_main == 12) && main_bytes > 16 * 1024 && main_bytes <= 64 * 1024 && res_bytes <= 16 * 1024 &&
        n_vectors >= (1 << 20) && n_vectors < (1 << 30)) {
      const int lds = (int)(main_bytes + res_bytes);
      const int64_t per_block = ((n_vectors + 511) / 512 + 1023) / 1024 * 1024;
      const DieGrid runs((n_vectors + per_block - 1) / per_block, n_vectors * 8 * (out_dtype == NPAMD_F32 ? 4 : 2));
#define NPAMD_RVQ8_LDS(BM, OUT)                                                                                             \
  do {                                                                                                                      \
    static LdsLatch latch;                                                                                                  \
    if (lds > 64 * 1024) {                                                                                                  \
      const hipError_t e = enable_dynamic_lds(latch, reinterpret_cast<const void*>(&rvq_dequant_vl8_lds_kernel<BM, 8, OUT>), lds); \
      if (e != hipSuccess) return fail(NPAMD_ERR_LAUNCH, "npamd_rvq_dequant: %s", hipGetErrorString(e));                     \
    }                                                                                                                       \
    launch(rvq_dequant_vl8_lds_kernel<BM, 8, OUT>, runs.blocks, 1024, lds, st, packed_main, n_bytes_main, bits_main,         \
           packed_res, n_bytes_res, bits_res, (const u32x4*)cb_main_f16, (uint32_t)nc_main, (const u32x4*)cb_res_f16,        \
           (uint32_t)nc_res, (const uint16_t*)row_scale_f16, (const uint16_t*)row_bias_f16, (uint32_t)groups,                \
           (uint32_t)n_vectors, (uint32_t)per_block, runs.per_die, out);                                                     \
  } while (0)
#define NPAMD_RVQ8_LDS_BITS(OUT)           \
  do {                                     \
    if (m16) NPAMD_RVQ8_LDS(16, OUT);      \
    else NPAMD_RVQ8_LDS(12, OUT);          \
  } while (0)
      switch (out_dtype) {
        case NPAMD_F16: NPAMD_RVQ8_LDS_BITS(NPAMD_F16); break;
        case NPAMD_BF16: NPAMD_RVQ8_LDS_BITS(NPAMD_BF16); break;
        case NPAMD_F32: NPAMD_RVQ8_LDS_BITS(NPAMD_F32); break;
        default: return fail(NPAMD_ERR_INVALID, "npamd_rvq_dequant: out_dtype must be f16, bf16 or f32");
      }
#undef NPAMD_RVQ8_LDS_BITS
#undef NPAMD_RVQ8_LDS
      return check_launch("npamd_rvq_dequant");
    }
#define NPAMD_RVQ8_LAUNCH(BM, BR, OUT)              \
  do {                                               \
    if (vpt == 2) NPAMD_RVQ8_VPT(BM, BR, OUT, 2);    \
    else NPAMD_RVQ8_VPT(BM, BR, OUT, 1);             \
  } while (0)
#define NPAMD_RVQ8_VPT(BM, BR, OUT, VPT)                                                               \
  launch(rvq_dequant_vl8_kernel<BM, BR, OUT, VPT>, grid, 256, 0, st,                                          \
      packed_main, n_bytes_main, bits_main, packed_res, n_bytes_res, bits_res, (const u32x4*)cb_main_f16, \
      (uint32_t)nc_main, (const u32x4*)cb_res_f16, (uint32_t)nc_res, (const uint16_t*)row_scale_f16,  \
      (const uint16_t*)row_bias_f16, N, (int)groups, rows.per_die, out)
#define NPAMD_RVQ8_BITS(OUT)                                \
  do {                                                      \
    if (m16 && r8) NPAMD_RVQ8_LAUNCH(16, 8, OUT);           \
    else if (bits_main == 12 && r8) NPAMD_RVQ8_LAUNCH(12, 8, OUT); \
    else if (m16) NPAMD_RVQ8_LAUNCH(16, 0, OUT);            \
    else NPAMD_RVQ8_LAUNCH(0, 0, OUT);                      \
  } while (0)
    switch (out_dtype) {
      case NPAMD_F16: NPAMD_RVQ8_BITS(NPAMD_F16); break;
      case NPAMD_BF16: NPAMD_RVQ8_BITS(NPAMD_BF16); break;
      case NPAMD_F32: NPAMD_RVQ8_BITS(NPAMD_F32); break;
      default: return fail(NPAMD_ERR_INVALID, "npamd_rvq_dequant: out_dtype must be f16, bf16 or f32");
    }
#undef NPAMD_RVQ8_BITS
#undef NPAMD_RVQ8_LAUNCH
#undef NPAMD_RVQ8_VPT
    return check_launch("npamd_rvq_dequant");
  }
#define NPAMD_RVQ_LAUNCH(OUT)                                                                   \
  launch(rvq_dequant_kernel<OUT>, blocks, 256, 0, st,                                               \
      packed_main, n_bytes_main, bits_main, packed_res, n_bytes_res, bits_res,                  \
      (const uint16_t*)cb_main_f16, (uint32_t)nc_main, (const uint16_t*)cb_res_f16,             \
      (uint32_t)nc_res, (const uint16_t*)row_scale_f16, \
      (const uint16_t*)row_bias_f16, vl, groups, n_vectors, out)
  switch (out_dtype) {
    case NPAMD_F16: NPAMD_RVQ_LAUNCH(NPAMD_F16); break;
    case NPAMD_BF16: NPAMD_RVQ_LAUNCH(NPAMD_BF16); break;
    case NPAMD_F32: NPAMD_RVQ_LAUNCH(NPAMD_F32); break;
    default: return fail(NPAMD_ERR_INVALID, "npamd_rvq_dequant: out_dtype must be f16, bf16 or f32");
  }
#undef NPAMD_RVQ_LAUNCH
  return check_launch("npamd_rvq_dequant");
}
