// Few-row forward (fa_fwd_decode.hpp) for 16-bit inputs, D in {32, 64, 128}:
// a translation unit of its own, so that the units of the other forwards
// compile the same code as without it.
#include "fa_fwd_decode.hpp"

namespace fa {

template hipError_t launch_fwd_decode<bf16>(const FwdParams&, int, bool, hipStream_t);
template hipError_t launch_fwd_decode<f16>(const FwdParams&, int, bool, hipStream_t);

}  // namespace fa
