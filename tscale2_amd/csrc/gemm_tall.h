// Products of medium size on a 256x128 tile (gemm_tall.hip)
#pragma once
#include "gemm_epilogue.h"

namespace gemmk
{
// stored (C_F32, C_BF16, C_BF16NORM) and accumulated (C_F32) products of T_I8 / T_FP8; T_I8: also sums of up to four with row scales of their own
bool PreferTall(const GemmP &p, int type, int ct, int epi);
bool TallCanRun(const GemmP &p, int type, int ct, int epi);
int RunTall(const GemmP &p, int type, int ct, int epi, hipStream_t stream);
} // namespace gemmk
