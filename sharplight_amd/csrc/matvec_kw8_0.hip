// Instantiations of matvec_kw8 for Q4_K and Q5_K (units of their own so that the formats compile in parallel).
#include "matvec_kw8.hpp"

namespace slhip {

int launch_kw8_part0(int fmt, const I8Args& a, bool dual, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_K: return launch_kw8_fmt<SLHIP_FMT_Q4_K>(a, dual, tn, st);
    case SLHIP_FMT_Q5_K: return launch_kw8_fmt<SLHIP_FMT_Q5_K>(a, dual, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
