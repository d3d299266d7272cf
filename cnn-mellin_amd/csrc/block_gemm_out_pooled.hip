// The channel-blocked matrix kernel that stores the maxima of pairs of columns, blocked: a layer in front of frequency pooling.
#include "block_gemm_kernel.hpp"

namespace mellin {

hipError_t launch_out_pooled(const BlockPlan &pl, const BlockGemmArgs &a, hipStream_t stream) {
  return launch_shape<OUT_POOLED>(pl, a, stream);
}

}  // namespace mellin
