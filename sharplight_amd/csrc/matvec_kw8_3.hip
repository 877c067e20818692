// Instantiations of matvec_kw8 for Q5_0, Q5_1 and IQ4_NL (units of their own so that the formats compile in parallel).
#include "matvec_kw8.hpp"

namespace slhip {

int launch_kw8_part3(int fmt, const I8Args& a, bool dual, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q5_0: return launch_kw8_fmt<SLHIP_FMT_Q5_0>(a, dual, tn, st);
    case SLHIP_FMT_Q5_1: return launch_kw8_fmt<SLHIP_FMT_Q5_1>(a, dual, tn, st);
    case SLHIP_FMT_IQ4_NL: return launch_kw8_fmt<SLHIP_FMT_IQ4_NL>(a, dual, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
