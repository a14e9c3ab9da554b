// Forward for bf16 head dims between the compiled ones (p.head_cols columns,
// FwdParamsCols), without bias or dropout: units of their own, so that those of
// the compiled head dims compile the same code as without them.  Head dims up
// to 96 run kernels of 96 columns: 3/4 of the products and tile bytes of 128.
// Bound as the kernels of the compiled head dims are; what this saves is the
// padded copies (five in, four out per step, each about a copy of its tensor)
// and the padding's products.  Measured (bf16, 4 x 1025 tokens, 16 heads of 80,
// forward + backward): 353 -> 191 us.
#include "fa_fwd.hpp"

namespace fa {

template <>
hipError_t launch_fwd_cols<bf16>(const FwdParams& p, int D, bool causal, hipStream_t s) {
    FwdParamsCols pc;
    static_cast<FwdParams&>(pc) = p;
    const int DK = D == 128 && p.head_cols <= 96 ? 96 : D;
#define FA_COLS_CASE(DD) \
    if (DK == DD) return causal ? launch_fwd_t<bf16, DD, true, 0, void>(pc, s) : launch_fwd_t<bf16, DD, false, 0, void>(pc, s);
    FA_COLS_CASE(64)
    FA_COLS_CASE(96)
    FA_COLS_CASE(128)
    FA_COLS_CASE(256)
#undef FA_COLS_CASE
    return hipErrorInvalidValue;
}

}  // namespace fa
