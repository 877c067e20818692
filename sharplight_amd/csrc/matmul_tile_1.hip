// Instantiations of matmul_tile for Q6_K and Q8_0 (units of their own so that the formats compile in parallel).
#include "matmul_tile.hpp"

namespace slhip {

int launch_tile_part1(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q6_K: return launch_tile_fmt<SLHIP_FMT_Q6_K>(a, dual, st);
    case SLHIP_FMT_Q8_0: return launch_tile_fmt<SLHIP_FMT_Q8_0>(a, dual, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
