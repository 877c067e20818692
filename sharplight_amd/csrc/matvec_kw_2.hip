// Instantiations of matvec_kw for Q4_0 and Q4_1 (units of their own so that the formats compile in parallel).
#include "matvec_kw.hpp"

namespace slhip {

int launch_kw_part2(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_0: return launch_kw_fmt<SLHIP_FMT_Q4_0>(a, dual, mt, tn, st);
    case SLHIP_FMT_Q4_1: return launch_kw_fmt<SLHIP_FMT_Q4_1>(a, dual, mt, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
