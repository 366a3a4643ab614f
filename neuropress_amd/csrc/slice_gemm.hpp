// Slice GEMM: y = x @ W^T (+ bias) for a few tokens (up to 32) and 16-bit VQ indices into a codebook of more than 4096
// rows of eight, read from the packed stream as it lies in memory.
//
// What bounds the kernels that look such codebooks up in memory is the L2: one request per index, 236 G/s at most,
// 31 us for the 7.3 M indices of a 14336 x 4096 layer whatever else they do.  Here a workgroup keeps one slice of the
// codebook (up to 8192 rows, 128 KiB) in LDS and walks the indices of its rows as the fused GEMV does -- a looked-up
// row is an MFMA operand -- except that an index outside the slice reads a row of zeros.  The slices' workgroups
// each contribute a partial sum and splitk_reduce_kernel adds them.  A 65536-row codebook is eight slices, so every
// index is walked eight times: 8 x (1.5 vector instructions + one LDS read + one MFMA) per index, the LDS reads being
// what paces it (7/8 of the lanes of a read ask for the same zeros: about 5 cycles per read, not 12).
//
// Measured (bf16, streams rotating, us at 16 tokens; the GEMV over memory / this): 4096 x 14336 with 65536 rows 39 / 27.5
// (through the module 36.9 / 24.4), 14336 x 4096 39 / 32, 8192 x 8192 43 / 28; with 16384 rows 37 / 16.6, 37 / 16.6 and 41 / 17;
// with 8192 rows 34 / 14.8, 34 / 14.9 and 37 / 13.2.  Where it goes at 4096 x 14336 with 65536 rows (kernel 21.5): 8.5 for the
// launch, the fill and the end, 0.93 per super-step of 256 rows -- LDS reads 0.6 of it, the rest mostly waiting for
// activations and indices -- and the reduction, 6 of the 27.5 and 3 of the 24.4.  LDS is active in 84 % of the walk's cycles
// (50 % of the launch), matrix pipes 30 % and vector instructions 32 % of the launch.  What did not pay: checks for infinities on the way to LDS
// (0.15 per super-step; now only where a sum shows one), sixteen waves of half the registers, all activations read behind
// one barrier (a third of the time in waits), eight row tiles per wave, a reduction by four waves per row.
//
// Work split: a cell is (row block, part of K); the workgroups of a cell's slices run on one die, whose L2 then serves the
// cell's indices to all but the first of them.  Block = 8 waves, KG k groups x RG row groups; a wave owns T row tiles
// of 16.  A super-step is 256 * KG k: the lane's 16-byte index load is one 64-k chunk of one row, as in the fused GEMV.
// The super-step's activations go through LDS once per workgroup (16 KiB).
#pragma once

#include "gemm_tile.hpp"

namespace npamd {

constexpr int kSliceMaxTokens = 32;

struct SliceArgs {
  const void* x;
  int64_t ldx;
  const uint8_t* packed;  // 16-bit indices, [N][K / 8]
  const void* cb;         // [nc][8] in the activation dtype
  float* partials;        // [slices * parts][M][N]
  int M, N, chunks, nc;
  int slices, slice_rows;           // slice s: rows [s * slice_rows, ...)
  int row_blocks, parts, part_super;  // cells = row_blocks * parts, part_super super-steps each
};

struct SlicePlan {
  int slices, slice_rows, tiles, row_blocks, parts, part_super;
};
inline int64_t slice_partials_bytes(const SlicePlan& p, int M, int N) { return (int64_t)p.slices * p.parts * M * N * 4; }

bool slice_takes(int M, int N, int K, int nc);
int64_t slice_workspace_bytes(int M, int N, int chunks, int nc);
double slice_estimate_ns(int M, int N, int chunks, int nc);
// act: NPAMD_F16 or NPAMD_BF16 (activations, codebook and output); workspace: slice_workspace_bytes of it.
int launch_slice(int act, const GemmShape& s, const uint8_t* packed, const void* cb, int nc, hipStream_t st, const char* what,
                 void* workspace);

}  // namespace npamd
