// Products whose 64x128 tiles leave CUs idle, on 64x64 tiles (gemm_square.hip)
#pragma once
#include "gemm_epilogue.h"

namespace gemmk
{
// stored and accumulated products (C_F32, C_BF16) of T_I8 / T_FP8; T_FP8: also sums of up to four
bool PreferSquare(const GemmP &p);
bool SquareCanRun(const GemmP &p, int type, int ct, int epi);
int RunSquare(const GemmP &p, int type, int ct, int epi, hipStream_t stream);
} // namespace gemmk
