// Backward for f16 head dims between the compiled ones up to 128 (p.head_cols
// columns, BwdParamsCols), without bias or dropout (see fa_fwd_cols_f16.hip).
#include "fa_bwd.hpp"

namespace fa {

template <>
hipError_t launch_bwd_cols<f16>(const BwdParams& p, int D, bool causal, int stage, hipStream_t s) {
    BwdParamsCols pc;
    static_cast<BwdParams&>(pc) = p;
    const int DK = D == 128 && p.head_cols <= 96 ? 96 : D;
#define FA_COLS_CASE(DD)                                                          \
    if (DK == DD) return causal ? launch_bwd_t<f16, DD, true, 0, void>(pc, stage, s) \
                                : launch_bwd_t<f16, DD, false, 0, void>(pc, stage, s);
    FA_COLS_CASE(64)
    FA_COLS_CASE(96)
    FA_COLS_CASE(128)
#undef FA_COLS_CASE
    return hipErrorInvalidValue;
}

}  // namespace fa
