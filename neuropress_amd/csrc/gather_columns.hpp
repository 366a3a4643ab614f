#pragma once

#include "common.hpp"

namespace npamd {

// ---------------------------------------------------------------------------
// Activations as the MFMA kernels read them: columns permuted and / or rows padded with zeros to a
// whole number of 64-column chunks, 16-bit elements:
//   out[m, k] = x[m, perm ? perm[k] : k] for k < K, 0 for K <= k < ldo and for column numbers that x does not have.
//
// Bound by the launch at the token counts of a decode step and by HBM beyond.  With a permutation a block first
// copies whole rows into LDS (one contiguous read) and gathers there with 2-byte reads: through the vector memory path
// an element gather costs a lane one cycle and a cache line each (77 x 2184: 2.3 us where torch's gather takes 4.2).
// Few rows: a block takes 2048 output columns of one, and a row is copied once per block.  Past kGatherBlocks blocks of
// those a row has only as many as make up that number, which stride over its columns (220 x 13968 10.4 -> 5.8 us), one
// from 1024 rows on, of two rows at a time then, which share the reads of the permutation.  A row copied by every
// block of 2048 columns / like this, us: 300 x 13968 20.2 / 7.0, 600 x 4096
// 7.6 / 4.3, 1200 x 13968 65.0 / 23.5, 4096 x 3456 39.3 / 11.4, 4096 x 14336 195.6 / 54.4 (4.3 TB/s).
// ---------------------------------------------------------------------------
constexpr int kGatherRowMax = 32768;  // elements of the rows held in LDS (64 KiB)
constexpr int kGatherBlocks = 1024, kGatherPairRows = 1024;
// One block of 256 threads: its `segment` of `segments` of ROWS rows from row ROWS * `rows` on; row_lds: the rows in LDS.
template <bool PERM, bool LDS, int ROWS>
__device__ __forceinline__ void gather_columns_block(const uint16_t* __restrict__ x, int64_t ldx, const int32_t* __restrict__ perm,
                                                     uint16_t* __restrict__ out, int64_t ldo, int M, int K, bool vec, bool perm_vec,
                                                     unsigned segment, unsigned segments, unsigned rows, uint16_t* row_lds) {
  const int row0 = (int)rows * ROWS;
  const int stride = (K + 7) & ~7;  // elements between the rows in LDS
  const uint16_t* xr[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) xr[r] = x + (int64_t)min(row0 + r, M - 1) * ldx;
  if constexpr (PERM && LDS) {
    const int whole = vec ? K >> 3 : 0;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      uint16_t* const mine = row_lds + r * stride;
#pragma unroll 4
      for (int i = threadIdx.x; i < whole; i += 256)
        reinterpret_cast<u32x4*>(mine)[i] = reinterpret_cast<const u32x4*>(xr[r])[i];
      for (int i = whole * 8 + threadIdx.x; i < K; i += 256) mine[i] = xr[r][i];
      xr[r] = mine;
    }
    __syncthreads();
  }
  for (int64_t c0 = (int64_t)(segment * 256 + threadIdx.x) * 8; c0 < ldo; c0 += (int64_t)segments * 2048) {
    const int k0 = (int)c0;
    int at[8];
    if (PERM && perm_vec && k0 + 8 <= K) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(perm + k0), hi = *reinterpret_cast<const u32x4*>(perm + k0 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        at[e] = (int)lo[e];
        at[4 + e] = (int)hi[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) at[e] = k0 + e < K ? (PERM ? perm[k0 + e] : k0 + e) : -1;
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      if (row0 + r >= M) break;
      uint16_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (unsigned)at[e] < (unsigned)K ? xr[r][at[e]] : (uint16_t)0;
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (uint32_t)v[2 * e] | ((uint32_t)v[2 * e + 1] << 16);
      *reinterpret_cast<u32x4*>(out + (int64_t)(row0 + r) * ldo + k0) = o;
    }
  }
}

// How a call of M rows of K columns, ldo columns of output, is dealt to blocks.
struct GatherPlan {
  bool lds, pair;
  unsigned segments, row_blocks;
  int lds_bytes;
  GatherPlan(bool perm, int64_t ldo, int M, int K) {
    const unsigned whole = (unsigned)((ldo + 2047) / 2048);
    lds = perm && K <= kGatherRowMax;
    pair = lds && M >= kGatherPairRows && 2 * ((K + 7) & ~7) <= kGatherRowMax;
    lds_bytes = lds ? ((K + 7) & ~7) * 2 * (pair ? 2 : 1) : 0;
    const unsigned per_row = lds ? (unsigned)(M < kGatherBlocks ? kGatherBlocks / M : 1) : whole;
    segments = per_row < whole ? per_row : whole;
    row_blocks = (unsigned)(pair ? (M + 1) / 2 : M);
  }
};

}  // namespace npamd
