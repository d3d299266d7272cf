// The channel-blocked matrix kernel as the input gradient of a layer behind a ReLU, as it lies.
#include "block_gemm_kernel.hpp"

namespace mellin {

hipError_t launch_grad_plain(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  return launch_shape<GRAD_PLAIN>(pl, a, stream);
}

}  // namespace mellin
