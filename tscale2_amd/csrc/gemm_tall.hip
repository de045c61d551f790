// Stored and accumulated 8-bit products of medium size on a 256x128 tile: results that fill the chip about once with it, contractions of a few
// steps.  The 128x128 kernel (gemm.hip) has one step of 32 KB under way per workgroup and waits for all of it at every step, so a step takes the
// latency of memory (1.4 us) whatever it multiplies, and further products of a sum start from nothing; the 256x256 ring needs four times the
// tiles.
//
// A workgroup of eight waves (64x64 accumulators each, one workgroup per CU) walks 128-byte steps of K through three stages of 48 KB, global ->
// LDS without registers, two steps under way while one is multiplied; the steps of several products (i8, row scales of their own) are one
// pipeline.  What bounds it then is the rate at which a CU fetches lines from L2, about 32 bytes per clock.  A lane owns a row of the result
// (operands swapped): the 16-bit epilogue is the row-owning one of gemm_epilogue.h, fp32 rows leave through 16 KB of LDS per wave as whole
// 256-byte runs, and what an accumulating product adds to is fetched behind the first two steps.
#include "gemm_tall.h"

using namespace gemmk;

namespace
{
constexpr int TBM = 256, TBN = 128;
constexpr int TA = TBM * BKB, TSTAGE = (TBM + TBN) * BKB, TSTAGES = 3;

typedef __attribute__((address_space(3))) uint8_t *TLds3;

// SEG (i8, fp32 result): p.nSeg products, each with row scales of its own, added in fp32 in their order
// JOBS: blockIdx.z picks one of several products (GemmP)
template <int TYPE, int CT, int EPI, bool SEG, bool JOBS = false> __global__ void __launch_bounds__(512, 2) GemmTall(GemmP p)
{
    if constexpr (JOBS) {
        PickJob(p);
    }
    typedef typename AccT<TYPE>::type TAcc;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[TSTAGES * TSTAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, half = lane >> 5, l32 = lane & 31;
    const unsigned ldsBase = (unsigned)(uintptr_t)(TLds3)lds;

    int tm, tn;
    MapTile(blockIdx.x, p.tilesM * p.tilesN, p.tilesM, p.tilesN, &tm, &tn, p.mapGroup ? p.mapGroup : 8);
    const int rowBase = tm * TBM, colBase = tn * TBN;
    const int kSteps = p.kBytes / BKB, total = SEG ? kSteps * p.nSeg : kSteps;

    // ---- loader: 48 wave-level loads of 1 KB (8 rows of 128 bytes) per step, six per wave; 16-byte chunks XOR-swizzled by the row
    const int lda = (int)p.lda, ldb = (int)p.ldb;
    int aOff[4], bOff[2];
    {
        const int r = lane >> 3, ch = (lane & 7) ^ (((wave & 1) << 2) + (lane >> 4));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            aOff[i] = ((wave + 8 * i) * 8 + r) * lda + ch * 16;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            bOff[i] = ((wave + 8 * i) * 8 + r) * ldb + ch * 16;
        }
    }
    const int64_t aTile = (int64_t)rowBase * p.lda, bTile = (int64_t)colBase * p.ldb;
    int loadStepNo = 0, loadSeg = 0, loadStage = 0, loaded = 0;
    auto loadNext = [&]() {
        const uint8_t *a = p.a, *b = p.b;
        if constexpr (SEG) {
            a = loadSeg == 0 ? p.a : loadSeg == 1 ? p.segA[0] : loadSeg == 2 ? p.segA[1] : p.segA[2];
            b = loadSeg == 0 ? p.b : loadSeg == 1 ? p.segB[0] : loadSeg == 2 ? p.segB[1] : p.segB[2];
        }
        const unsigned st = ldsBase + loadStage * TSTAGE;
        const v4i ra = BufferRsrc(a + aTile + (int64_t)loadStepNo * BKB), rb = BufferRsrc(b + bTile + (int64_t)loadStepNo * BKB);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            TS2_LOAD_LDS16(st + (wave + 8 * i) * 1024, aOff[i], ra);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            TS2_LOAD_LDS16(st + TA + (wave + 8 * i) * 1024, bOff[i], rb);
        }
        ++loaded;
        loadStage = loadStage == TSTAGES - 1 ? 0 : loadStage + 1;
        if (++loadStepNo == kSteps) {
            loadStepNo = 0;
            ++loadSeg;
        }
    };

    // ---- a step: two halves of 64 bytes of K
    TAcc acc[2][2];
    auto zeroAcc = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[i][n][e] = 0;
                }
            }
        }
    };
    constexpr int CSTEP = TYPE == T_FP8 ? 1 : 2;
    auto multiply = [&](int stage) {
        const uint8_t *st = lds + stage * TSTAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c0 = u * 4 + (TYPE == T_FP8 ? half * 2 : half);
            v8i fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ar = wm * 64 + i * 32 + l32, br = wn * 64 + i * 32 + l32;
                const v4i a0 = *(const v4i *)(st + SwizzleOffset(ar, c0)), a1 = *(const v4i *)(st + SwizzleOffset(ar, c0 + CSTEP));
                const v4i b0 = *(const v4i *)(st + TA + SwizzleOffset(br, c0)), b1 = *(const v4i *)(st + TA + SwizzleOffset(br, c0 + CSTEP));
                fa[i] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                fb[i] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    if constexpr (TYPE == T_FP8) {
                        acc[i][n] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[n], fa[i], acc[i][n], 0, 0, 0, 0, 0, 0);
                    } else {
                        const v4i a0 = __builtin_shufflevector(fa[i], fa[i], 0, 1, 2, 3), a1 = __builtin_shufflevector(fa[i], fa[i], 4, 5, 6, 7);
                        const v4i b0 = __builtin_shufflevector(fb[n], fb[n], 0, 1, 2, 3), b1 = __builtin_shufflevector(fb[n], fb[n], 4, 5, 6, 7);
                        acc[i][n] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b0, a0, acc[i][n], 0, 0, 0);
                        acc[i][n] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b1, a1, acc[i][n], 0, 0, 0);
                    }
                }
            }
        }
    };
#define TALL_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

    const int firstRow = rowBase + wm * 64;
    float segRow[SEG ? 4 : 1][2]; // row scales of the lane's two rows
    if constexpr (SEG) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float *rs = s == 0 ? p.rowScale : s == 1 ? p.segRowScale[0] : s == 2 ? p.segRowScale[1] : p.segRowScale[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                segRow[s][i] = s < p.nSeg ? rs[firstRow + i * 32 + l32] : 0.f;
            }
        }
    }
    zeroAcc();
    loadNext();
    if (total > 1) {
        loadNext();
    }
    // fp32 rows: lane -> 16-byte chunk cc of row it * 4 + cr, sixteen times
    const int cr = lane >> 4, cc = lane & 15;
    const int mLive = p.mLive > 0 ? p.mLive : p.m;
    uint8_t *const cWave = p.c + (int64_t)firstRow * p.ldc + (int64_t)(colBase + wn * 64) * 4;
    float4 old[EPI == TS2_EPI_ADD ? 16 : 1];
    if constexpr (EPI == TS2_EPI_ADD) {
#pragma unroll
        for (int it = 0; it < 16; ++it) { // (rows of the tile are rows of C: read all, use the live ones)
            old[it] = *(const float4 *)(cWave + (int64_t)(it * 4 + cr) * p.ldc + cc * 16);
        }
    }
    float facc[SEG ? 2 : 1][SEG ? 2 : 1][16];
    int stage = 0, inSeg = 0, seg = 0;
    for (int t = 0; t < total; ++t) {
        if (EPI == TS2_EPI_ADD && t < 2 && t + 1 < total) {
            asm volatile("s_waitcnt vmcnt(22)" ::: "memory"); // the sixteen loads of C lie behind steps 0 and 1
        } else if (t + 1 < total) {
            asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        TALL_BARRIER(); // step t is in LDS, and every wave is done with the stage that step t+2 goes to
        if (t + 2 < total) {
            loadNext();
        }
        multiply(stage);
        stage = stage == TSTAGES - 1 ? 0 : stage + 1;
        if constexpr (SEG) {
            if (++inSeg == kSteps) {
                inSeg = 0;
                float f = seg == 0 ? p.alpha : seg == 1 ? p.segAlpha[0] : seg == 2 ? p.segAlpha[1] : p.segAlpha[2];
                const float *fp = seg == 0 ? p.alphaPtr : seg == 1 ? p.segAlphaPtr[0] : seg == 2 ? p.segAlphaPtr[1] : p.segAlphaPtr[2];
                if (fp) {
                    f *= *fp;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float r = f * (seg == 0 ? segRow[0][i] : seg == 1 ? segRow[1][i] : seg == 2 ? segRow[2][i] : segRow[3][i]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            facc[i][n][e] = (seg == 0 ? 0.f : facc[i][n][e]) + (float)acc[i][n][e] * r;
                        }
                    }
                }
                zeroAcc();
                ++seg;
            }
        }
    }
    TALL_BARRIER(); // every wave has read its last operands

    if constexpr (CT == C_F32) {
        // ADD: the sums are scaled where the lane holds what they are added to, in one fused operation like in the other kernels (scaled before, the
        // product was rounded once more: 2.64e-8 from 64 bits instead of 2.50e-8)
        constexpr bool ADD = EPI == TS2_EPI_ADD;
        uint8_t *const mine = lds + wave * 16384;
        float *const rowFactor = (float *)(lds + 8 * 16384) + wave * 64;
        float scale = p.alpha;
        if (!SEG && p.alphaPtr) {
            scale *= *p.alphaPtr;
        }
        if constexpr (ADD) {
            rowFactor[lane] = p.rowScale ? scale * p.rowScale[firstRow + lane] : scale;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = i * 32 + l32;
            const float rs = SEG || ADD ? 1.f : p.rowScale ? scale * p.rowScale[firstRow + r] : scale;
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = SEG ? facc[i][n][q * 4 + e] : ADD ? (float)acc[i][n][q * 4 + e] : (float)acc[i][n][q * 4 + e] * rs;
                    }
                    *(float4 *)(mine + r * 256 + (((n * 8 + q * 2 + half) ^ (r & 15)) << 4)) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
        // (a wave reads what it wrote itself)
#pragma unroll
        for (int it = 0; it < 16; ++it) {
            const int r = it * 4 + cr;
            float4 v = *(const float4 *)(mine + r * 256 + ((cc ^ (r & 15)) << 4));
            const bool live = firstRow + r < mLive;
            uint8_t *q = cWave + (int64_t)r * p.ldc + cc * 16;
            if constexpr (ADD) {
                const float f = rowFactor[r];
                if (live) {
                    *(float4 *)q = make_float4(__builtin_fmaf(v.x, f, old[it].x), __builtin_fmaf(v.y, f, old[it].y), __builtin_fmaf(v.z, f, old[it].z),
                        __builtin_fmaf(v.w, f, old[it].w));
                }
            } else {
                *(float4 *)q = live ? v : make_float4(0, 0, 0, 0);
            }
        }
    } else {
        NormEpilogueRows<TYPE, CT == C_BF16NORM, CT == C_F16, 2, 2>(p, acc, lds + wave * 8192, (float *)(lds + 8 * 8192), rowBase, colBase, wm, wn, lane);
    }
}

template <int TYPE> int Launch(const GemmP &p, int ct, int epi, hipStream_t stream)
{
    const dim3 grid(p.tilesM * p.tilesN);
#define TALL(CT, EPI, SEG) hipLaunchKernelGGL((GemmTall<TYPE, CT, EPI, SEG>), grid, dim3(512), 0, stream, p)
    if (p.nSeg > 1) {
        if constexpr (TYPE == T_I8) {
            TALL(C_F32, TS2_EPI_STORE, true);
        }
    } else if (ct == C_F32) {
        if (epi == TS2_EPI_ADD) {
            TALL(C_F32, TS2_EPI_ADD, false);
        } else {
            TALL(C_F32, TS2_EPI_STORE, false);
        }
    } else if (ct == C_BF16NORM && p.jobs > 1) {
        if constexpr (TYPE == T_I8) {
            hipLaunchKernelGGL((GemmTall<TYPE, C_BF16NORM, TS2_EPI_STORE, false, true>), dim3(grid.x, 1, p.jobs), dim3(512), 0, stream, p);
        }
    } else if (ct == C_BF16NORM) {
        TALL(C_BF16NORM, TS2_EPI_STORE, false);
    } else {
        TALL(C_BF16, TS2_EPI_STORE, false);
    }
#undef TALL
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}
} // namespace

namespace gemmk
{
// Where this kernel takes over, by its tiles T (256 x 128 of C each, one per CU of the 256) and the bytes K of the contraction: short contractions, up
// to a round or two, and results that other kernels write badly.  Measured in a graph of 40 launches, others -> this one, us; ranges are over
// 30 to 70 shapes of 1024 to 32768 rows and 256 to 2048 columns in each interval.  Up to 64 tiles the kernel for few tiles is better (0.6 to 0.9
// of this one's time).
//   accumulating  4096x1024 (T = 128) K 512 i8 13.7 -> 11.9, e4m3 13.2 -> 12.0; 16384x512 (256) K 256 18.6 -> 14.2, 18.3 -> 14.0, K 2048 31.6 -> 26.2, 30.2 ->
//                 26.1; T 65 .. 128 i8 K 256 0.83-0.90, 512 0.89-0.99, 1024 0.89-1.13, 1536 0.99-1.14, 2048 0.98-1.22 (4096x640 15.3 -> 18.7), 3072 to T = 96 0.93-1.09,
//                 beyond 0.91-0.93, 4096 0.92-0.97, e4m3 K 256 0.85-0.97, 384 0.90-0.98, 512 0.91-1.03, 640 0.94-1.06, 768 0.97-1.09, 1024 0.96-1.11; 129 .. 256 0.71-0.93, e4m3 K 4096 0.94-1.05; 257 .. 448 0.72-0.99 to K 2048 (e4m3 3072 1.08); 449 .. 512
//                 0.72-0.95 to K 1024 (4096 1.16); 513 .. 640 i8 0.61-0.87 to K 2048, e4m3 0.79-0.90 to K 512
//   sums (i8)     two products 16384x512 K 512 25.9 -> 16.9, 16384x1024 53.2 -> 29.9 (two launches before), 8192x512 (128) K 1024 21.6 -> 22.0, 2048 31.8 -> 35.7;
//                 four 16384x512 K 384 35.2 -> 22.4, 16384x1024 (512) K 512 124.8 -> 48.9 (four launches), 32768x2048 (2048) K 2048 808 -> 632, 4096 1190 -> 1255
//   normalised    i8: 4096x1024 (128) K 512 13.4 -> 12.6, 16384x384 (192) 19.1 -> 13, 16384x512 (256), product and pass before, 27 -> 13.9; T 65 .. 128 0.89-1.00,
//                 129 .. 320 0.34-0.83 to K 2048, 321 .. 448 0.45-0.65 to K 1024 (2048 1.03), 449 .. 768 0.59-0.89 to K 512 (1024 1.06); where 256x256 tiles fill
//                 the chip (T from 384 on, whole ones) 384 .. 448 K 256 0.94-0.97, 512 1.00-1.03, 768 1.05-1.08, 1024 1.05-1.10, 449 .. 768 K 256 0.82-0.96, 512 0.86-0.99
//   stored fp32   T 65 .. 768 K 256, 512 i8 0.75-0.99, e4m3 0.84-1.02; K 1024 0.92-1.30, 0.99-1.40
//   stored bf16   i8: T 129 .. 256 0.90-1.01 to K 2048; 449 .. 768 K 256, 512 0.71-1.01; e4m3 (and others) equal or worse
bool PreferTall(const GemmP &p, int type, int ct, int epi)
{
    const long T = (long)(p.m / TBM) * (p.n / TBN);
    const int K = p.kBytes;
    const bool i8 = type == T_I8;
    if (T <= 64) {
        return false;
    }
    if (p.nSeg > 1) {
        return (p.nSeg > 2 || T > 128 || K <= 1024) && (K <= 2048 || (T > 128 && T <= 256));
    }
    if (epi == TS2_EPI_ADD) {
        if (T <= 128) {
            return K <= 512 || (i8 && K >= (T <= 96 ? 4096 : 3072) && K <= 4096);
        }
        return K <= (T <= 256 ? (i8 ? 4096 : 3072) : T <= 448 ? 2048 : T <= 512 ? 1024 : T <= 640 ? (i8 ? 2048 : 512) : 0);
    }
    if (ct == C_BF16NORM) {
        const bool large = T >= 384 && p.n % 256 == 0;
        return i8 && K <= (T <= 320 ? 2048 : T <= 448 ? (large ? 256 : 1024) : T <= 768 ? 512 : 0);
    }
    if (ct == C_F32) {
        return T <= 768 && K <= 512;
    }
    return ct == C_BF16 && i8 && (T <= 128 ? false : T <= 256 ? K <= 2048 : T > 448 && T <= 768 && K <= 512);
}

bool TallCanRun(const GemmP &p, int type, int ct, int epi)
{
    if ((type != T_I8 && type != T_FP8) || p.m <= 0 || p.n <= 0 || p.kBytes <= 0 || (p.m % TBM) || (p.n % TBN) || (p.kBytes % BKB) || p.tileGroup ||
        p.groupOffsets || p.splits > 1 || p.splitK > 1 || p.kTileScale || p.kMajor) {
        return false;
    }
    if (ct != C_F32 && ((ct != C_BF16 && ct != C_BF16NORM) || epi != TS2_EPI_STORE)) {
        return false;
    }
    if (p.nSeg > 1 && (type != T_I8 || ct != C_F32 || epi != TS2_EPI_STORE || p.nSeg > 4 || !p.rowScale)) {
        return false;
    }
    for (int i = 0; i + 1 < p.nSeg; ++i) {
        if (!p.segRowScale[i] || !p.segA[i] || !p.segB[i] || (((uintptr_t)p.segA[i] | (uintptr_t)p.segB[i]) & 15)) {
            return false;
        }
    }
    if (((uintptr_t)p.a | (uintptr_t)p.lda | (uintptr_t)p.b | (uintptr_t)p.ldb | (uintptr_t)p.c | (uintptr_t)p.ldc) & 15) {
        return false;
    }
    if (p.jobs > 1 && (type != T_I8 || ct != C_BF16NORM)) {
        return false;
    }
    if (ct == C_BF16NORM && ((p.normalize && !p.tileScale) || (p.rope && (((uintptr_t)p.rope & 15) || (p.ldRope & 3))))) {
        return false;
    }
    // offsets inside a tile are 32-bit
    return p.lda < (1 << 22) && p.ldb < (1 << 22) && p.ldc < (1 << 22);
}

int RunTall(const GemmP &in, int type, int ct, int epi, hipStream_t stream)
{
    if (!TallCanRun(in, type, ct, epi)) {
        return TS2_ERR_UNSUPPORTED;
    }
    GemmP p = in;
    p.tilesM = p.m / TBM;
    p.tilesN = p.n / TBN;
    return type == T_I8 ? Launch<T_I8>(p, ct, epi, stream) : Launch<T_FP8>(p, ct, epi, stream);
}
} // namespace gemmk
