// The kernel for products with few output tiles (gemm_slice.hip)
#pragma once
#include "gemm_epilogue.h"

namespace gemmk
{
struct SliceP {
    GemmP g;
    int ct, epi;                 // C_*, TS2_EPI_STORE / TS2_EPI_ADD
    int kLive;                   // K-major operands: contraction rows that count (none if 0); later rows read as zeros
    int kTileScaleRows;          // kTileScale: > 0 = every so many rows of C have a set of scales of their own (sets one after the other)
    // > 1: blockIdx.z picks one of several products of one shape that share A and are stored separately (C_BF16NORM; of p, b, c, tileScale,
    // alphaPtr, normalize and rope's use are each product's own)
    int jobs, jobNormalize, jobRope; // the latter two: bit per product
    const uint8_t *jobB[4];
    uint8_t *jobC[4];
    float *jobTileScale[4];
    const float *jobAlphaPtr[4];
};
bool SliceCanRun(const SliceP &sp, int type, bool tn);
int RunSlice(const SliceP &sp, int type, bool tn, hipStream_t stream);
// up to four i8 products with row scales of their own summed into one stored fp32 result on the 128x128 tile (gemm.hip)
int RunSumI8(const GemmP &p, hipStream_t stream);
} // namespace gemmk
