// What the assembled mixers (mixer.hip) use of the other files beyond the C ABI.
#pragma once

#include "qa_common.hpp"

namespace qa {

// sscan.hip: bytes of scratch qa_sscan_fwd can use for these sizes with token-major inputs (0: none)
int64_t sscan_token_major_workspace(const QaSScanParams& p);

// conv2.hip: the channel-contiguous forward conv.  Without x_out_scales every channel is an x channel with the one
// output scale `x_out_scale` (the Mamba1 conv); with conv_state the last inputs of every channel are left there.
int conv_channel_last_fwd(const QaConv2Params& p, hipStream_t stream);

}  // namespace qa
