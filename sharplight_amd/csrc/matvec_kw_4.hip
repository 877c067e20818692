// Instantiations of matvec_kw for Q2_K and Q3_K (units of their own so that the formats compile in parallel).
#include "matvec_kw.hpp"

namespace slhip {

int launch_kw_part4(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q2_K: return launch_kw_fmt<SLHIP_FMT_Q2_K>(a, dual, mt, tn, st);
    case SLHIP_FMT_Q3_K: return launch_kw_fmt<SLHIP_FMT_Q3_K>(a, dual, mt, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
