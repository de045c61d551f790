// The kernel for products with few output tiles (gemm_slice.hip)
#pragma once
#include "gemm_epilogue.h"

namespace gemmk
{
struct SliceP {
    GemmP g;
    int ct, epi;                 // C_*, TS2_EPI_STORE / TS2_EPI_ADD
    int kLive;                   // K-major operands: contraction rows that count (0 = all); later rows read as zeros
    const float *segRowScale[3]; // i8: row scales of the further products
    int kTileScaleRows;          // kTileScale: > 0 = every so many rows of C have a set of scales of their own (sets one after the other)
};
bool SliceCanRun(const SliceP &sp, int type, bool tn);
int RunSlice(const SliceP &sp, int type, bool tn, hipStream_t stream);
} // namespace gemmk
