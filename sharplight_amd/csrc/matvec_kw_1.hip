// Instantiations of matvec_kw for Q6_K and Q8_0 (units of their own so that the formats compile in parallel).
#include "matvec_kw.hpp"

namespace slhip {

int launch_kw_part1(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q6_K: return launch_kw_fmt<SLHIP_FMT_Q6_K>(a, dual, mt, tn, st);
    case SLHIP_FMT_Q8_0: return launch_kw_fmt<SLHIP_FMT_Q8_0>(a, dual, mt, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
