// Packed deltas of many matrices in one launch (gemm_deltas.hip)
#pragma once
#include "gemm_epilogue.h"

namespace gemmk
{
// one packed delta [gradDim][srcDim] = alpha * *alphaPtr * grad^T src of a batch of them, both operands row-major as they lie
struct DeltaJob {
    const uint8_t *grad, *src;
    uint8_t *delta;
    float *tileScale;
    const float *alphaPtr, *kTileScale; // kTileScale (i8): [gradDim / kTileScaleRows][k-tiles]; kTileScaleRows 0 = one set
    float alpha;
    int ldGrad, ldSrc, ldDelta; // bytes
    int ldTileScale;            // floats
    int gradDim, srcDim, kTileScaleRows;
    int first; // first workgroup (set by the launch)
};
constexpr int DELTA_JOBS = 32;
struct DeltaBatchP {
    DeltaJob job[DELTA_JOBS];
    int count, kBytes, kLive, kTileBytes, kGroup; // kGroup (i8): k-tiles that are summed apart
};
// any number of deltas over the same rows, 32 to a launch (T_I8 with k-tile scales, T_FP8)
bool DeltaBatchCanRun(const DeltaJob &d, int type, int kBytes, int kLive, int kTileBytes);
int RunDeltaBatch(const DeltaJob *jobs, int count, int type, int kBytes, int kLive, int kTileBytes, hipStream_t stream);
} // namespace gemmk
