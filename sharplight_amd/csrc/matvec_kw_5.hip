// Instantiations of matvec_kw for bf16 and f16 weights (units of their own so that the formats compile in parallel).
#include "matvec_kw.hpp"

namespace slhip {

int launch_kw_part5(int fmt, const MatvecArgs& a, bool dual, int mt, int tn, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_BF16: return launch_kw_fmt<SLHIP_FMT_BF16>(a, dual, mt, tn, st);
    case SLHIP_FMT_F16: return launch_kw_fmt<SLHIP_FMT_F16>(a, dual, mt, tn, st);
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
