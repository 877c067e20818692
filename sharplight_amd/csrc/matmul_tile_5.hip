// Instantiations of matmul_tile for bf16 and f16 weights (units of their own so that the formats compile in parallel).
#include "matmul_tile.hpp"

namespace slhip {

int launch_tile_part5(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_BF16: return launch_tile_fmt<SLHIP_FMT_BF16>(a, dual, st);
    case SLHIP_FMT_F16: return launch_tile_fmt<SLHIP_FMT_F16>(a, dual, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
