// Backward for bf16 head dims between 128 and 256 (p.head_cols columns,
// BwdParamsCols), without bias or dropout: a unit of its own for its compiler
// flags (accumulators in AGPRs, as fa_bwd_d256_bf16.hip).
#include "fa_bwd.hpp"

namespace fa {

template <>
hipError_t launch_bwd_cols256<bf16>(const BwdParams& p, bool causal, int stage, hipStream_t s) {
    BwdParamsCols pc;
    static_cast<BwdParams&>(pc) = p;
    return causal ? launch_bwd_t<bf16, 256, true, 0, void>(pc, stage, s) : launch_bwd_t<bf16, 256, false, 0, void>(pc, stage, s);
}

}  // namespace fa
