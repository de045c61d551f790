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
};
bool SliceCanRun(const SliceP &sp, int type, bool tn);
int RunSlice(const SliceP &sp, int type, bool tn, hipStream_t stream);
// g.jobs products that share A, each normalised (or not) and stored: the 128x128 (T_FP8) and 256x128 (T_I8) kernels (gemm.hip, gemm_tall.hip)
bool PreferJobs(const GemmP &g, int type);
int RunJobs(const GemmP &g, int type, hipStream_t stream);
// up to four i8 products with row scales of their own summed into one stored fp32 result on the 128x128 tile (gemm.hip)
int RunSumI8(const GemmP &p, hipStream_t stream);
} // namespace gemmk
