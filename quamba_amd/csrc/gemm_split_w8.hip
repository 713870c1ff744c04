// The products of some activation rows with int8 weights (gemm_split.hpp).
#include "gemm_split.hpp"

namespace qa {
int split_launch_w8(const GemvParams& p, int shape, const GemvConv* conv, hipStream_t stream) { return split::launch_shape<8>(p, shape, conv, stream); }
}  // namespace qa
