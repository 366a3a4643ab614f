// The wide tiles of the dense product (wide_gemm.hpp), and which number of the plan's list (dense_gemm.hip) is which.
#include "wide_gemm.hpp"

namespace npamd {

namespace {

template <int ACT>
int launch_wide_act(const DenseShape& s, int tile, hipStream_t st) {
  switch (tile) {
    case 1: return launch_wide_tile<ACT, WideTile<2, 2, 2, 2, 6, 4>>(s, st);    // 64 x 64
    case 2: return launch_wide_tile<ACT, WideTile<2, 2, 2, 4, 5, 12>>(s, st);   // 64 x 128
    case 3: return launch_wide_tile<ACT, WideTile<2, 2, 4, 4, 4, 24>>(s, st);   // 128 x 128
    case 4: return launch_wide_tile<ACT, WideTile<2, 2, 5, 4, 4, 24>>(s, st);   // 160 x 128
    case 5: return launch_wide_tile<ACT, WideTile<4, 2, 4, 4, 3, 24>>(s, st);   // 256 x 128
    case 6: return launch_wide_tile<ACT, WideTile<4, 2, 3, 4, 3, 20>>(s, st);   // 192 x 128
    case 7: return launch_wide_tile<ACT, WideTile<2, 2, 3, 4, 4, 20>>(s, st);   // 96 x 128
    case 8: return launch_wide_tile<ACT, WideTile<2, 4, 5, 4, 3, 24>>(s, st);   // 160 x 256
    case 9: return launch_wide_tile<ACT, WideTile<2, 4, 6, 4, 2, 20>>(s, st);   // 192 x 256
    case 10: return launch_wide_tile<ACT, WideTile<4, 2, 4, 7, 2, 24>>(s, st);  // 256 x 224
    case 11: return launch_wide_tile<ACT, WideTile<2, 4, 8, 4, 2, 24>>(s, st);  // 256 x 256
    case 12: return launch_wide_tile<ACT, WideTile<2, 2, 3, 2, 6, 6>>(s, st);   // 96 x 64
    default: return launch_wide_tile<ACT, WideTile<2, 4, 6, 3, 3, 24>>(s, st);  // 192 x 192
  }
}

}  // namespace

int launch_wide(const DenseShape& s, int act, int tile, hipStream_t st) {
  return act == NPAMD_BF16 ? launch_wide_act<NPAMD_BF16>(s, tile, st) : launch_wide_act<NPAMD_F16>(s, tile, st);
}

}  // namespace npamd
