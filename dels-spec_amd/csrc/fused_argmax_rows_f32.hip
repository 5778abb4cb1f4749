// Instantiations of the 17-to-64-row fused argmax kernel for fp32 base logits (one
// translation unit per base dtype keeps the build parallel).
#include "fused_argmax_rows.h"

namespace dels {

hipError_t launch_rows_f32(const ArgmaxKArgs& ka, bool packed, int prior_kind, bool vec, hipStream_t s) {
    return launch_rows_for_base<float>(ka, packed, prior_kind, vec, s);
}

}  // namespace dels
