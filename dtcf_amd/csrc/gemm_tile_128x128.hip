// FP64 GEMM on 128 x 128 C tiles, four waves of 64 x 64 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_128x128(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg128x128, 128, 128, 64, 64>(g, s); }

int dtcf::gemm_group_tile_128x128(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    return launch_group_tile<kCfg128x128, 128, 128, 64, 64>(ga, amode, bmode, s);
}
