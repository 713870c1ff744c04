// sscan_waves.hip: the token-major Mamba1 scan with the time cut over the waves of a workgroup.
#pragma once
#include "mixer_common.hpp"

namespace qa {

constexpr int kScanWavesMax = 16;          // waves of a workgroup
// lanes of a QaSScanParams.mapping that name this kernel: with the lanes and waves of scan_waves_plan, and with four lanes a
// channel (32 more: eight) and one wave (w more: w + 1)
constexpr int kScanWavesMapping = 16, kScanWavesNamed = 64;

// Lanes per channel and waves per workgroup for these sizes, and the estimated time (kScanWavesNever: better left to another
// kernel, one pass of eight lanes).
constexpr int64_t kScanWavesNever = 1LL << 62;
struct ScanWavesPlan {
    int lanes, waves;
    int64_t ns;
};
ScanWavesPlan scan_waves_plan(const QaSScanParams& p, int cus);

// for arguments that sscan_token_major_check accepts
int sscan_waves_fwd(const QaSScanParams& p, const SscanDtProj* dt, int lanes, int waves, hipStream_t stream);

}  // namespace qa
