// FP64 GEMM on 96 x 192 C tiles, four waves of 48 x 96 (gemm_tile.hpp).
#include "gemm_tile.hpp"

int dtcf::gemm_tile_96x192(const GemmArgs &g, hipStream_t s) { return launch_tile<kCfg96x192, 96, 192, 48, 96>(g, s); }

int dtcf::gemm_group_tile_96x192(const GemmGroupArgs &ga, int amode, int bmode, hipStream_t s)
{
    return launch_group_tile<kCfg96x192, 96, 192, 48, 96>(ga, amode, bmode, s);
}
