// What the assembled mixers (mixer.hip) use of the other files beyond the C ABI.
#pragma once

#include "qa_common.hpp"

namespace qa {

// hadamard.hip: whether norm_hadamard_quant takes rows of `dim` columns in norm groups of `group`, and
// qa_rmsnorm_gated_hadamard_quant itself, which as an entry point of its own leaves rows of 4096 columns in one group to the
// two kernels (`in_layer` false)
bool norm_hadamard_fuses(int dim, int group);
int norm_hadamard_quant(const QaNormGatedParams* n, const QaHadamardParams* h, bool in_layer, void* stream);

// sscan_tm.hip: qa_sscan_fwd for token-major inputs.  With `dt` the step size codes are not read but made in the scan:
// dt_proj's product of x (x_proj's rows, x_l_stride apart) with w (d_inner rows of `rank` codes, a multiple of 16 up to 192),
// scaled col * (row * acc) and rounded as the int8 product does it.  seqlen * x_l_stride below 2^30.
struct SscanDtProj {
    const int8_t *w, *x;
    int64_t x_batch_stride, x_l_stride;
    const float *row_scale, *col_scale;
    int rank, col_numel;
};
constexpr int kSscanDtRank = 192;
int sscan_token_major_check(const QaSScanParams& p, const SscanDtProj* dt);       // what it refuses, without a launch
int sscan_token_major_fwd(const QaSScanParams& p, const SscanDtProj* dt, hipStream_t stream);
// bytes of scratch it can use for these sizes (0: none)
int64_t sscan_token_major_workspace(const QaSScanParams& p);

// sscan_step.hip: the single-token state update of a Mamba1 layer with dt_proj in front of it (p.dt is not read): the step size
// code of channel d is the projection of `x` (16 * pieces codes a batch entry, x_batch_stride apart) with row d of `w`
// (contiguous rows), scaled and rounded as the int8 product does it.  QA_ERR_UNSUPPORTED where the layout is not the one it
// takes (contiguous channels and states, whole waves of sixteen channels).
struct SsmDtProj {
    const int8_t *w, *x;
    int64_t x_batch_stride;
    const float *row_scale, *col_scale;
    int pieces, col_numel, use_alpha;
    float alpha;
};
constexpr int kSsmDtPieces = 12;       // up to 192 inputs
int mamba1_step(const QaSsmUpdateParams& p, const SsmDtProj& dt, hipStream_t stream);
// what qa_ssm_state_update refuses, without a launch
int ssm_update_check(const QaSsmUpdateParams& p);

// ssd.hip: what qa_ssd_chunk_scan_fwd refuses about sizes and tensors, without a launch
int ssd_check(const QaSsdParams& p);

// normgated.hip: columns of the widest group
constexpr int kNormGroup = 32768;

// conv2.hip: the channel-contiguous forward conv.  Without x_out_scales every channel is an x channel with the one
// output scale `x_out_scale` (the Mamba1 conv); with conv_state the last inputs of every channel are left there.
int conv_channel_last_fwd(const QaConv2Params& p, hipStream_t stream);
// the single-step update in the same terms
int conv_single_update(const QaConv2Params& p, hipStream_t stream);

}  // namespace qa
