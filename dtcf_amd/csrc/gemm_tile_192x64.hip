// FP64 GEMM on 192 x 64 C tiles, four waves of 48 x 64 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_192x64(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg192x64, 192, 64, 48, 64>(g, s); }
