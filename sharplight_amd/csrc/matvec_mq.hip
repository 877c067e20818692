// Instantiations of matvec_mq2 (a unit of its own so that it compiles in parallel with the other kernels).
#include "matvec_mq.hpp"

namespace slhip {

int run_mq2_any(int fmt, const MatvecArgs& a, bool dual, hipStream_t st)
{
    switch (fmt) {
    case SLHIP_FMT_Q4_0: return mq2_fits<SLHIP_FMT_Q4_0>(a) ? run_mq2<SLHIP_FMT_Q4_0>(a, dual, st) : SLHIP_ERR_UNSUPPORTED;
    case SLHIP_FMT_Q8_0: return mq2_fits<SLHIP_FMT_Q8_0>(a) ? run_mq2<SLHIP_FMT_Q8_0>(a, dual, st) : SLHIP_ERR_UNSUPPORTED;
    case SLHIP_FMT_Q4_1: return mq2_fits<SLHIP_FMT_Q4_1>(a) ? run_mq2<SLHIP_FMT_Q4_1>(a, dual, st) : SLHIP_ERR_UNSUPPORTED;
    case SLHIP_FMT_Q5_0: return mq2_fits<SLHIP_FMT_Q5_0>(a) ? run_mq2<SLHIP_FMT_Q5_0>(a, dual, st) : SLHIP_ERR_UNSUPPORTED;
    case SLHIP_FMT_Q5_1: return mq2_fits<SLHIP_FMT_Q5_1>(a) ? run_mq2<SLHIP_FMT_Q5_1>(a, dual, st) : SLHIP_ERR_UNSUPPORTED;
    default: return SLHIP_ERR_UNSUPPORTED;
    }
}

}  // namespace slhip
