// Instantiations of the 17-to-64-row fused argmax kernel for f16_t base logits (one
// translation unit per base dtype keeps the build parallel).
#include "fused_argmax_rows.h"

namespace dels {

hipError_t launch_rows_f16(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s) {
    return launch_rows_for_base<f16_t>(ka, packed, prior_kind, vec, s);
}

}  // namespace dels
