// The products of some activation rows with 4-bit weights (gemm_split.hpp).
#include "gemm_split.hpp"

namespace qa {
int split_launch_w4(const GemvParams& p, int shape, const GemvConv* conv, hipStream_t stream) { return split::launch_shape<4>(p, shape, conv, stream); }
}  // namespace qa
