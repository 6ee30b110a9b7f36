// FP64 GEMM on 64 x 192 C tiles, four waves of 64 x 48 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_64x192(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg64x192, 64, 192, 64, 48>(g, s); }
