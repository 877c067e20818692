// Instantiations of matvec_kw for Q4_K and Q5_K (units of their own so that the formats compile in parallel).
#include "matvec_kw.hpp"

namespace slhip {

int launch_kw_part0(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_K: return launch_kw_fmt<SLHIP_FMT_Q4_K>(a, dual, mt, tn, st);
    case SLHIP_FMT_Q5_K: return launch_kw_fmt<SLHIP_FMT_Q5_K>(a, dual, mt, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
