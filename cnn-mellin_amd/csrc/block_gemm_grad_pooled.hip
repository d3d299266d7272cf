// The channel-blocked matrix kernel as the input gradient of a layer behind frequency pooling, stored as that of the values in front of it.
#include "block_gemm_kernel.hpp"

namespace mellin {

hipError_t launch_grad_pooled(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  return launch_shape<GRAD_POOLED>(pl, a, stream);
}

}  // namespace mellin
