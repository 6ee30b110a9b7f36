// FP64 GEMM on 192 x 96 C tiles, four waves of 96 x 48 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_192x96(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg192x96, 192, 96, 96, 48>(g, s); }

int dtcf::gemm_group_tile_192x96(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    return launch_group_tile<kCfg192x96, 192, 96, 96, 48>(ga, amode, bmode, s);
}
