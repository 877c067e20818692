// Instantiations of matvec_kw8 for Q6_K and Q8_0 (units of their own so that the formats compile in parallel).
#include "matvec_kw8.hpp"

namespace slhip {

int launch_kw8_part1(int fmt, const I8Args& a, bool dual, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q6_K: return launch_kw8_fmt<SLHIP_FMT_Q6_K>(a, dual, tn, st);
    case SLHIP_FMT_Q8_0: return launch_kw8_fmt<SLHIP_FMT_Q8_0>(a, dual, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
