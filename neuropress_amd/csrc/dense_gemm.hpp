// The arguments of the dense product's kernels (dense_gemm.hip, wide_gemm.hpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace npamd {

struct DenseShape {
  const void* x;
  const void* w;
  const float* bias;
  void* y;
  int64_t ldx, ldw, ldy;
  int M, N, steps;   // 64-k steps of a row
  int row_tiles, col_tiles, splits, units_per_die;  // unit: a part of K of one tile
  float* partials;   // splits > 1: [splits][M][N]
  int pieces;        // 16-byte pieces of a row: K / 8
  int group;         // row tiles of a group (wide tiles)
};

// The product on wide tile `tile` of the plan's list; splits > 1: its parts, without their sum.
int launch_wide(const DenseShape& s, int act, int tile, hipStream_t st);

}  // namespace npamd
