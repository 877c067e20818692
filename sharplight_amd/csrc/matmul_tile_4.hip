// Instantiations of matmul_tile for Q2_K and Q3_K (units of their own so that the formats compile in parallel).
#include "matmul_tile.hpp"

namespace slhip {

int launch_tile_part4(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q2_K: return launch_tile_fmt<SLHIP_FMT_Q2_K>(a, dual, st);
    case SLHIP_FMT_Q3_K: return launch_tile_fmt<SLHIP_FMT_Q3_K>(a, dual, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
