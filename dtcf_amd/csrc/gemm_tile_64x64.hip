// FP64 GEMM on 64 x 64 C tiles, four waves of 32 x 32 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_64x64(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg64x64, 64, 64, 32, 32>(g, s); }

int dtcf::gemm_group_tile_64x64(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    return launch_group_tile<kCfg64x64, 64, 64, 32, 32>(ga, amode, bmode, s);
}
