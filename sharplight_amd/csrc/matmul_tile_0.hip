// Instantiations of matmul_tile for Q4_K and Q5_K (units of their own so that the formats compile in parallel).
#include "matmul_tile.hpp"

namespace slhip {

int launch_tile_part0(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_K: return launch_tile_fmt<SLHIP_FMT_Q4_K>(a, dual, st);
    case SLHIP_FMT_Q5_K: return launch_tile_fmt<SLHIP_FMT_Q5_K>(a, dual, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
