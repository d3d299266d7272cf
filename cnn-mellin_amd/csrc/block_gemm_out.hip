// The channel-blocked matrix kernel with a blocked output: a layer whose reader is another such layer.
#include "block_gemm_kernel.hpp"

namespace mellin {

hipError_t launch_out_blocked(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  return launch_shape<OUT_BLOCKED>(pl, a, stream);
}

}  // namespace mellin
