// 8-bit products on 64x64 tiles: results whose 64x128 tiles (gemm_slice.hip) are fewer than the CUs.  What bounds those is the path from L2 to a
// CU's LDS, about 32 bytes per clock: a tile of 64x128 fetches 192 bytes per byte of K on half of the chip or less, one of 64x64 fetches 128 on
// twice as many CUs.
//
// A workgroup of eight waves owns 64 x 64 of C and cuts the contraction four ways, as the kernel for few tiles does: a step is 256 bytes of K,
// and the wave pair `kg` (a wave per 32 columns, 64x32 accumulators) multiplies bytes kg*64 .. kg*64+63 of it.  Four stages of 32 KB, one workgroup
// per CU: three steps are under way while one is multiplied, four loads per wave and step.  The partial tiles are added through LDS in the order of
// that kernel, so the results are its results, bit by bit.  Row tiles without a live row load and multiply nothing.
#include "gemm_square.h"

using namespace gemmk;

namespace
{
constexpr int QT = 64, QK = 256;              // tile (rows and columns), bytes of K per step
constexpr int QA = QT * QK, QSTAGE = 2 * QA;  // bytes
constexpr int QSTAGES = 4, QPART = QT * QT * 4;

typedef __attribute__((address_space(3))) uint8_t *TLds3;

// CT: C_F32 or C_BF16; ADD: accumulate; SEG (fp8): p.nSeg products in one set of accumulators, brought to the next product's factor at each seam
template <int TYPE, int CT, bool ADD, bool SEG> __global__ void __launch_bounds__(512, 2) GemmSquare(GemmP p)
{
    typedef typename AccT<TYPE>::type TAcc;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[QSTAGES * QSTAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, kg = wave >> 1, half = lane >> 5, l32 = lane & 31;
    const unsigned ldsBase = (unsigned)(uintptr_t)(TLds3)lds;

    int tm, tn;
    MapTile(blockIdx.x, p.tilesM * p.tilesN, p.tilesM, p.tilesN, &tm, &tn, 8);
    const int rowBase = tm * QT, colBase = tn * QT;
    const int mLive = p.mLive > 0 ? p.mLive : p.m;
    const int kUnits = rowBase < mLive ? p.kBytes / BKB : 0; // of 128 bytes
    const int nSteps = (kUnits + 1) / 2;
    const bool oddTail = kUnits & 1; // the last step holds 128 bytes of K only

    // thread -> row er, 8 columns in two chunks of four: 16-byte stores of fp32 are chunks of neighbouring lanes
    const int er = tid >> 3, eu = tid & 7, row = rowBase + er;
    const bool live = row < mLive;
    auto chunkOf = [&](int c) { return CT == C_F32 ? c * 8 + eu : eu * 2 + c; };
    uint8_t *const cRow = p.c + (int64_t)row * p.ldc;
    float out[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (ADD && live) { // (under way before the first operands)
        if constexpr (CT == C_F32) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float4 o = *(const float4 *)(cRow + (int64_t)(colBase + chunkOf(c) * 4) * 4);
                out[c * 4 + 0] = o.x;
                out[c * 4 + 1] = o.y;
                out[c * 4 + 2] = o.z;
                out[c * 4 + 3] = o.w;
            }
        } else {
            const uint4 o = *(const uint4 *)(cRow + (int64_t)(colBase + eu * 8) * 2);
            const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                out[2 * k] = __uint_as_float(w[k] << 16);
                out[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
            }
        }
    }
    const float rowScale = p.rowScale ? p.rowScale[row] : 1.f;

    // ---- loader: 32 wave-level loads of 1 KB (4 tile rows of 256 bytes) per step, four per wave; the slot of a lane holds chunk slot ^ (row % 16)
    const int lda = (int)p.lda, ldb = (int)p.ldb;
    int aOff[2], bOff[2], back[2]; // back: bytes from the upper to the lower half of a step for lanes that hold the upper
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int rr = (wave + 8 * i) * 4 + (lane >> 4), ch = (lane & 15) ^ (rr & 15);
        aOff[i] = rr * lda + ch * 16;
        bOff[i] = rr * ldb + ch * 16;
        back[i] = (ch >> 3) * 128;
    }
    auto aOf = [&](int seg) { return !SEG || seg == 0 ? p.a : seg == 1 ? p.segA[0] : seg == 2 ? p.segA[1] : p.segA[2]; };
    auto bOf = [&](int seg) { return !SEG || seg == 0 ? p.b : seg == 1 ? p.segB[0] : seg == 2 ? p.segB[1] : p.segB[2]; };
    auto factorOf = [&](int seg) -> float {
        float f = !SEG || seg == 0 ? p.alpha : seg == 1 ? p.segAlpha[0] : seg == 2 ? p.segAlpha[1] : p.segAlpha[2];
        const float *q = !SEG || seg == 0 ? p.alphaPtr : seg == 1 ? p.segAlphaPtr[0] : seg == 2 ? p.segAlphaPtr[1] : p.segAlphaPtr[2];
        return q ? f * *q : f;
    };
    // the products that count, two bits each (a factor of zero, the scale of an all-zero matrix, has no units to convert into)
    unsigned list = 0;
    int count = 1;
    float units = factorOf(0);
    if constexpr (SEG) {
        count = 0;
        for (int seg = p.nSeg - 1; seg >= 0; --seg) {
            const float f = factorOf(seg);
            if (f != 0) {
                list = (list << 2) | seg;
                ++count;
                units = f;
            }
        }
    }
    const int total = count * nSteps;
    unsigned loadList = list;
    int loadStepNo = 0, loadStage = 0;
    auto loadNext = [&]() {
        const int seg = loadList & 3;
        const int64_t k0 = (int64_t)loadStepNo * QK;
        const v4i ra = BufferRsrc(aOf(seg) + (int64_t)rowBase * p.lda + k0), rb = BufferRsrc(bOf(seg) + (int64_t)colBase * p.ldb + k0);
        const unsigned st = ldsBase + loadStage * QSTAGE;
        // the upper half of a 128-byte last step is not multiplied: its lanes fetch the lower half again
        const bool cut = oddTail && loadStepNo == nSteps - 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            TS2_LOAD_LDS16(st + (wave + 8 * i) * 1024, aOff[i] - (cut ? back[i] : 0), ra);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            TS2_LOAD_LDS16(st + QA + (wave + 8 * i) * 1024, bOff[i] - (cut ? back[i] : 0), rb);
        }
        loadStage = loadStage == QSTAGES - 1 ? 0 : loadStage + 1;
        if (++loadStepNo == nSteps) {
            loadStepNo = 0;
            loadList >>= 2;
        }
    };

    // ---- operand fragments of this wave's 64 bytes of K.  fp8: chunks kg*4 + half*2 + {0, 1}; i8: chunks kg*4 + half + {0, 2} feed two MFMAs
    constexpr int CSTEP = TYPE == T_FP8 ? 1 : 2;
    const int c0 = kg * 4 + (TYPE == T_FP8 ? half * 2 : half);
    const int ch0 = (c0 ^ (l32 & 15)) << 4, ch1 = ((c0 + CSTEP) ^ (l32 & 15)) << 4;
    TAcc acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            acc[i][e] = 0;
        }
    }
    auto multiply = [&](int step, int stage) {
        if (oddTail && step == nSteps - 1 && kg >= 2) { // (uniform over the wave)
            return;
        }
        const uint8_t *st = lds + stage * QSTAGE, *br = st + QA + (wn * 32 + l32) * QK;
        const v4i b0 = *(const v4i *)(br + ch0), b1 = *(const v4i *)(br + ch1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint8_t *ar = st + (i * 32 + l32) * QK;
            const v4i a0 = *(const v4i *)(ar + ch0), a1 = *(const v4i *)(ar + ch1);
            if constexpr (TYPE == T_FP8) {
                acc[i] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(__builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7),
                    __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7), acc[i], 0, 0, 0, 0, 0, 0);
            } else {
                acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b0, a0, acc[i], 0, 0, 0);
                acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b1, a1, acc[i], 0, 0, 0);
            }
        }
    };
#define SQUARE_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

#pragma unroll
    for (int t = 0; t < QSTAGES - 1; ++t) {
        if (t < total) {
            loadNext();
        }
    }
    int step = 0, stage = 0;
    for (int t = 0; t < total; ++t) {
        if (t + 2 < total) {
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        } else if (t + 1 < total) {
            asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        SQUARE_BARRIER(); // step t is in LDS, and every wave is done with the stage that step t+3 goes to
        if (t + QSTAGES - 1 < total) {
            loadNext();
        }
        multiply(step, stage);
        stage = stage == QSTAGES - 1 ? 0 : stage + 1;
        if (SEG && ++step == nSteps) {
            step = 0;
            list >>= 2;
            if constexpr (TYPE != T_I8) {
                if (t + 1 < total) { // the accumulators go on in the next product's units
                    const float nxt = factorOf(list & 3);
                    if (nxt != units) {
                        const float ratio = units / nxt;
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
#pragma unroll
                            for (int e = 0; e < 16; ++e) {
                                acc[i][e] *= ratio;
                            }
                        }
                        units = nxt;
                    }
                }
            }
        } else if (!SEG) {
            ++step;
        }
    }

    // ---- partial tiles of the four wave pairs -> LDS (a lane owns a row: operands swapped), sums of the thread's 8 columns back; 16-byte chunks
    // of a 256-byte row are swizzled by the row
    SQUARE_BARRIER(); // every wave has read its last operands
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = i * 32 + l32;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint8_t *d = lds + kg * QPART + r * (QT * 4) + (((wn * 8 + q * 2 + half) ^ (r & 15)) << 4);
            if constexpr (TYPE == T_I8) {
                *(int4 *)d = make_int4(acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]);
            } else {
                *(float4 *)d = make_float4(acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]);
            }
        }
    }
    __syncthreads();
    if (ADD && !live) {
        return;
    }
    float scale = units;
    if (p.rowScale) {
        scale *= rowScale;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        typedef typename std::conditional<TYPE == T_I8, v4i, v4f>::type TQuad;
        const uint8_t *s = lds + er * (QT * 4) + ((chunkOf(c) ^ (er & 15)) << 4);
        const TQuad q0 = *(const TQuad *)s, q1 = *(const TQuad *)(s + QPART), q2 = *(const TQuad *)(s + 2 * QPART), q3 = *(const TQuad *)(s + 3 * QPART);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = (float)((q0[e] + q1[e]) + (q2[e] + q3[e]));
            out[c * 4 + e] = live ? out[c * 4 + e] + v * scale : 0.f;
        }
    }
    if constexpr (CT == C_F32) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            *(float4 *)(cRow + (int64_t)(colBase + chunkOf(c) * 4) * 4) = make_float4(out[c * 4], out[c * 4 + 1], out[c * 4 + 2], out[c * 4 + 3]);
        }
    } else {
        *(uint4 *)(cRow + (int64_t)(colBase + eu * 8) * 2) =
            make_uint4(PackBf16x2(out[0], out[1]), PackBf16x2(out[2], out[3]), PackBf16x2(out[4], out[5]), PackBf16x2(out[6], out[7]));
    }
}

template <int TYPE> int Launch(const GemmP &p, int ct, int epi, hipStream_t stream)
{
    const dim3 grid(p.tilesM * p.tilesN);
#define SQUARE(CT, ADD, SEG) hipLaunchKernelGGL((GemmSquare<TYPE, CT, ADD, SEG>), grid, dim3(512), 0, stream, p)
#define SQUARE_EPI(CT, SEG)                                                                                                                \
    if (epi == TS2_EPI_ADD) {                                                                                                              \
        SQUARE(CT, true, SEG);                                                                                                             \
    } else {                                                                                                                               \
        SQUARE(CT, false, SEG);                                                                                                            \
    }
    if (p.nSeg > 1) {
        if constexpr (TYPE == T_FP8) {
            if (ct == C_F32) {
                SQUARE_EPI(C_F32, true)
            } else {
                SQUARE_EPI(C_BF16, true)
            }
        }
    } else if (ct == C_F32) {
        SQUARE_EPI(C_F32, false)
    } else {
        SQUARE_EPI(C_BF16, false)
    }
#undef SQUARE_EPI
#undef SQUARE
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}
} // namespace

namespace gemmk
{
// Up to one tile per CU.  Measured in a graph of 40 launches against the kernels that took these products before (gemm_slice.hip, 128x128 tiles), 4
// to 256 tiles, K 128 to 4096: stored fp32 0.60-0.75 of the time, accumulated 0.56-0.74, stored bf16 0.59-0.86 (i8 and e4m3; 1024x1024, accumulated:
// K 1024 7.9 -> 5.3 us, K 4096 15.9 -> 9.7; 512x256, K 256 5.2 -> 3.4).  A second round costs what the first did: 384 tiles 1.0-1.3.
bool PreferSquare(const GemmP &p)
{
    return (int64_t)(p.m / QT) * (p.n / QT) <= 256;
}

bool SquareCanRun(const GemmP &p, int type, int ct, int epi)
{
    if ((type != T_I8 && type != T_FP8) || p.m <= 0 || p.n <= 0 || p.kBytes <= 0 || (p.m % QT) || (p.n % QT) || (p.kBytes % BKB) || p.tileGroup ||
        p.groupOffsets || p.splits > 1 || p.splitK > 1 || p.kTileScale || p.kMajor || (ct != C_F32 && ct != C_BF16) ||
        (epi != TS2_EPI_STORE && epi != TS2_EPI_ADD) || (p.nSeg > 1 && type != T_FP8) || p.nSeg > 4) {
        return false;
    }
    for (int i = 0; i + 1 < p.nSeg; ++i) {
        if (!p.segA[i] || !p.segB[i] || (((uintptr_t)p.segA[i] | (uintptr_t)p.segB[i]) & 15)) {
            return false;
        }
    }
    if (((uintptr_t)p.a | (uintptr_t)p.lda | (uintptr_t)p.b | (uintptr_t)p.ldb | (uintptr_t)p.c | (uintptr_t)p.ldc) & 15) {
        return false;
    }
    // offsets inside a tile are 32-bit
    return p.lda < (1 << 24) && p.ldb < (1 << 24);
}

int RunSquare(const GemmP &in, int type, int ct, int epi, hipStream_t stream)
{
    if (!SquareCanRun(in, type, ct, epi)) {
        return TS2_ERR_UNSUPPORTED;
    }
    GemmP p = in;
    p.tilesM = p.m / QT;
    p.tilesN = p.n / QT;
    return type == T_I8 ? Launch<T_I8>(p, ct, epi, stream) : Launch<T_FP8>(p, ct, epi, stream);
}
} // namespace gemmk
