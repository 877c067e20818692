// Instantiations of matmul_tile for Q4_0 and Q4_1 (units of their own so that the formats compile in parallel).
#include "matmul_tile.hpp"

namespace slhip {

int launch_tile_part2(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_0: return launch_tile_fmt<SLHIP_FMT_Q4_0>(a, dual, st);
    case SLHIP_FMT_Q4_1: return launch_tile_fmt<SLHIP_FMT_Q4_1>(a, dual, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
