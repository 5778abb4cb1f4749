// Instantiations of the 17-to-64-row e4m3 fused argmax kernel for bf16_t base logits (one
// translation unit per base dtype keeps the build parallel).
#include "fused_argmax_rows8.h"

namespace dels {

hipError_t launch_rows8_bf16(const ArgmaxKArgs& ka, int prior_kind, bool vec, hipStream_t s) {
    return launch_rows8_for_base<bf16_t>(ka, prior_kind, vec, s);
}

}  // namespace dels
