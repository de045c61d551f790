// Products whose result has too few tiles to fill the chip with the 128x128 and 256x256 kernels (gemm.hip): short batches, narrow
// matrices, deltas.  There a workgroup's time is a chain - load latency, a few contraction steps, epilogue - and the matrix cores idle.
//
// A workgroup of eight waves owns 64 x 128 of C and cuts the contraction four ways inside itself: a step is 256 bytes of K, and the wave
// pair `kg` (one wave per 64 columns, 64x64 accumulators) multiplies bytes kg*64 .. kg*64+63 of it.  So one output tile keeps all four
// matrix cores of a CU busy, each with a wave tile whose LDS reads balance its MFMAs (8 KB per 4 MFMAs), and a contraction of 1024 bytes
// is four steps.  Three stages of 48 KB (144 KB of LDS, one workgroup per CU): two steps are in flight while one is multiplied.  Loads
// go global -> LDS without registers (buffer_load_dwordx4 .. lds); every wave issues exactly six per step, so "six outstanding" at the
// top of a step means its own part of the step has landed (loads complete in order), and the barrier makes that true of all waves.
// The four partial tiles are added through LDS in a fixed order (int32 for i8: exact), after which a thread holds 16 columns of one row
// and every epilogue is a few lines: eight lanes own a row of 128 columns, which is the tile of the normalising and packing epilogues.
//
// K-major operands (TN: A [k][m], B [k][n]) are read by the transposing LDS reads as in the ring kernel; contraction rows at and beyond
// kLive read as zeros (the descriptor of a step ends there), so ragged batches need no transposed or cleared copies.
// KT (i8): one scale per kTile contraction elements.  A workgroup takes the k-tiles of its slice, up to four, wave pair kg the whole of the
// kg-th (a step is 64 elements of each), so every pair holds one tile's exact int32 sum at the end and the reduction adds them scaled, in
// tile order.
// Several products into one result: fp8 / bf16 keep one set of accumulators, brought to the next product's factor at each seam; i8
// products carry row scales of their own and are added one after the other in fp32, in the order of separate accumulating launches.
#include "gemm_slice.h"

using namespace gemmk;

namespace
{
constexpr int SBM = 64, SBN = 128, SK = 256;           // tile, bytes of K per step
constexpr int SA = SBM * SK, STAGE = (SBM + SBN) * SK; // bytes
constexpr int NSTAGE = 3;

typedef __attribute__((address_space(3))) uint8_t *TLds3;

template <int TYPE, bool TN, bool KT = false> __global__ void __launch_bounds__(512, 2) GemmSlice(SliceP sp)
{
    typedef typename AccT<TYPE>::type TAcc;
    const GemmP &p = sp.g;
    constexpr int ESZ = TYPE == T_BF16 ? 2 : 1;
    constexpr int KR = SK / ESZ; // contraction elements of a step
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NSTAGE * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, kg = wave >> 1;
    const int half = lane >> 5, l32 = lane & 31;
    const unsigned ldsBase = (unsigned)(uintptr_t)(TLds3)lds;

    int tm, tn;
    MapTile(blockIdx.x, p.tilesM * p.tilesN, p.tilesM, p.tilesN, &tm, &tn, 8);
    const int rowBase = tm * SBM, colBase = tn * SBN;
    // slice or group of the contraction, in units of 128 bytes of K
    int kBeg = 0, kUnits = p.kBytes / BKB;
    uint8_t *cBase = p.c;
    float *tileScale = p.tileScale;
    const uint8_t *bBase = p.b;
    const float *alphaPtr = p.alphaPtr;
    bool normalize = p.normalize, rotate = p.rope != nullptr;
    if (p.jobs > 1) {
        const int j = blockIdx.z;
        bBase = p.jobB[j];
        cBase = p.jobC[j];
        tileScale = p.jobTileScale[j];
        alphaPtr = p.jobAlphaPtr[j];
        normalize = (p.jobNormalize >> j) & 1;
        rotate = (p.jobRope >> j) & 1;
    }
    int64_t bSlab = 0;
    if (p.tileGroup) {
        const int g = p.tileGroup[rowBase / TILE];
        if (g < 0) {
            return;
        }
        bSlab = (int64_t)g * p.bSlab;
    }
    if (p.groupOffsets) {
        const int g = blockIdx.y;
        kBeg = p.groupOffsets[g] * ESZ / BKB;
        kUnits = p.groupOffsets[g + 1] * ESZ / BKB - kBeg;
        cBase += (int64_t)g * p.cSlab;
        if (tileScale) {
            tileScale += (int64_t)g * p.tileScaleSlab;
        }
    } else if (p.splits > 1) {
        const int per = (kUnits + p.splits - 1) / p.splits;
        kBeg = blockIdx.y * per;
        kUnits = min(per, max(kUnits - kBeg, 0));
        cBase += (int64_t)blockIdx.y * p.splitSlab;
    }
    int nSteps = (kUnits + 1) / 2;
    const bool oddTail = !TN && !KT && (kUnits & 1); // NT: the last step holds 128 bytes of K only
    int kt0 = 0, ktCount = 0;                        // KT: first k-tile of the workgroup, number of its k-tiles
    if constexpr (KT) {
        const int all = p.kBytes / p.kTileBytes, per = p.splits > 1 ? (all + p.splits - 1) / p.splits : all;
        kt0 = blockIdx.y * per;
        ktCount = min(per, max(all - kt0, 0));
        nSteps = ktCount > 0 ? p.kTileBytes / 64 : 0;
    }

    // ---- what the epilogue reads is fetched while the first operands are under way.  Thread -> row er, 16 columns in four chunks of four
    const int er = tid >> 3, eu = tid & 7;
    const int row = rowBase + er;
    const int mLive = p.mLive > 0 ? p.mLive : p.m;
    const bool live = row < mLive;
    // chunk c of a thread: 16-byte stores of the result type are whole chunks of neighbouring lanes
    const int ct = sp.ct;
    auto chunkOf = [&](int c) { return (ct == C_F32 || ct == C_I32) ? c * 8 + eu : ct == C_I8PACK ? eu * 4 + c : (c >> 1) * 16 + eu * 2 + (c & 1); };
    float out[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        out[e] = 0;
    }
    uint8_t *cRow = cBase + (int64_t)row * p.ldc;
    if (sp.epi == TS2_EPI_ADD && live) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int col = colBase + chunkOf(c) * 4;
            if (ct == C_F32) {
                const float4 o = *(const float4 *)(cRow + (int64_t)col * 4);
                out[c * 4 + 0] = o.x;
                out[c * 4 + 1] = o.y;
                out[c * 4 + 2] = o.z;
                out[c * 4 + 3] = o.w;
            } else {
                const uint2 o = *(const uint2 *)(cRow + (int64_t)col * 2);
                out[c * 4 + 0] = __uint_as_float(o.x << 16);
                out[c * 4 + 1] = __uint_as_float(o.x & 0xffff0000u);
                out[c * 4 + 2] = __uint_as_float(o.y << 16);
                out[c * 4 + 3] = __uint_as_float(o.y & 0xffff0000u);
            }
        }
    }

    // ---- loader: 48 wave-level loads of 1 KB per step, six per wave (A blocks wave, wave + 8; B blocks wave, wave + 8, +16, +24).
    // NT: a block is 4 tile rows of 256 bytes; the slot of a lane holds chunk slot ^ (row % 16), so that eight consecutive rows read at
    // one chunk lie in different banks.  TN: a block is 1 KB of contraction rows (16 / 8 of A, 8 / 4 of B for 8-bit / bf16); the granules
    // of one MFMA block (32 tile rows) are XOR-swizzled so that what one transposing read touches covers all banks once.
    int aOff[2], bOff[4];
    const int lda = (int)p.lda, ldb = (int)p.ldb;
    if constexpr (!TN) {
        const int r = lane >> 4, slot = lane & 15;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int rr = (wave + 8 * i) * 4 + r;
            const int ch = slot ^ (rr & 15);
            aOff[i] = rr * lda + (KT ? ((ch >> 2) < ktCount ? (ch >> 2) : 0) * p.kTileBytes + (ch & 3) * 16 : ch << 4);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = (wave + 8 * i) * 4 + r;
            const int ch = slot ^ (rr & 15);
            bOff[i] = rr * ldb + (KT ? ((ch >> 2) < ktCount ? (ch >> 2) : 0) * p.kTileBytes + (ch & 3) * 16 : ch << 4);
        }
    } else if constexpr (ESZ == 1) {
        const int ra = lane >> 2, sa = lane & 3, rb = lane >> 3, sb = lane & 7;
        const int ca = (((sa >> 1) ^ ((ra >> 2) & 1)) << 5) + (sa & 1) * 16, cb = (((sb >> 1) ^ ((rb >> 1) & 3)) << 5) + (sb & 1) * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            // KT: rows kg * 64 .. + 63 of a stage are rows of the kg-th k-tile
            const int rr = (wave + 8 * i) * 16 + ra;
            aOff[i] = (KT ? ((rr >> 6) < ktCount ? (rr >> 6) : 0) * p.kTileBytes + (rr & 63) : rr) * lda + ca;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = (wave + 8 * i) * 8 + rb;
            bOff[i] = (KT ? ((rr >> 6) < ktCount ? (rr >> 6) : 0) * p.kTileBytes + (rr & 63) : rr) * ldb + cb;
        }
    } else {
        const int ra = lane >> 3, sa = lane & 7, rb = lane >> 4, sb = lane & 15;
        const int ca = (((sa >> 2) ^ ((ra >> 1) & 1)) << 6) + (sa & 3) * 16, cb = (((sb >> 2) ^ (rb & 3)) << 6) + (sb & 3) * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            aOff[i] = ((wave + 8 * i) * 8 + ra) * lda + ca;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bOff[i] = ((wave + 8 * i) * 4 + rb) * ldb + cb;
        }
    }
    const int kLive = sp.kLive;
    auto loadStep = [&](const uint8_t *a, const uint8_t *b, int step, int stage) {
        const unsigned st = ldsBase + stage * STAGE;
        v4i ra, rb;
        int cut = 0;
        if constexpr (KT) {
            const int64_t k0 = (int64_t)kt0 * p.kTileBytes + step * 64;
            ra = BufferRsrc(TN ? a + k0 * p.lda + rowBase : a + (int64_t)rowBase * p.lda + k0);
            rb = BufferRsrc(TN ? b + k0 * p.ldb + colBase : b + (int64_t)colBase * p.ldb + k0);
        } else if constexpr (TN) {
            const int k0 = kBeg * (BKB / ESZ) + step * KR;
            // rows of this step that belong to the slice and are live
            const int rows = min(min(kBeg * (BKB / ESZ) + kUnits * (BKB / ESZ), kLive) - k0, KR);
            ra = BufferRsrc(a + (int64_t)k0 * p.lda + rowBase * ESZ, rows > 0 ? (rows - 1) * lda + SBM * ESZ : 0);
            rb = BufferRsrc(b + (int64_t)k0 * p.ldb + colBase * ESZ, rows > 0 ? (rows - 1) * ldb + SBN * ESZ : 0);
        } else {
            const int64_t k0 = (int64_t)kBeg * BKB + (int64_t)step * SK;
            ra = BufferRsrc(a + (int64_t)rowBase * p.lda + k0);
            rb = BufferRsrc(b + (int64_t)colBase * p.ldb + k0);
            // the upper half of a 128-byte last step is not multiplied: its lanes fetch the lower half again
            cut = (oddTail && step == nSteps - 1) ? 1 : 0;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            int off = aOff[i];
            if (!TN && cut) {
                const int rr = (wave + 8 * i) * 4 + (lane >> 4);
                off -= ((((lane & 15) ^ (rr & 15)) >> 3) & 1) * 128;
            }
            TS2_LOAD_LDS16(st + (wave + 8 * i) * 1024, off, ra);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int off = bOff[i];
            if (!TN && cut) {
                const int rr = (wave + 8 * i) * 4 + (lane >> 4);
                off -= ((((lane & 15) ^ (rr & 15)) >> 3) & 1) * 128;
            }
            TS2_LOAD_LDS16(st + SA + (wave + 8 * i) * 1024, off, rb);
        }
    };

    // ---- operand fragments of this wave's 64 bytes of K
    TAcc acc[2][2];
    auto zeroAcc = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[i][j][e] = 0;
                }
            }
        }
    };
    auto mul8 = [&](const v8i &a, const v8i &b, TAcc c) -> TAcc { // 64 bytes of K; a lane owns a ROW of the block (operands swapped)
        if constexpr (TYPE == T_FP8) {
            return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b, a, c, 0, 0, 0, 0, 0, 0);
        } else {
            const v4i a0 = __builtin_shufflevector(a, a, 0, 1, 2, 3), a1 = __builtin_shufflevector(a, a, 4, 5, 6, 7);
            const v4i b0 = __builtin_shufflevector(b, b, 0, 1, 2, 3), b1 = __builtin_shufflevector(b, b, 4, 5, 6, 7);
            if constexpr (TYPE == T_I8) {
                c = __builtin_amdgcn_mfma_i32_32x32x32_i8(b0, a0, c, 0, 0, 0);
                return __builtin_amdgcn_mfma_i32_32x32x32_i8(b1, a1, c, 0, 0, 0);
            } else {
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, b0), __builtin_bit_cast(v8bf, a0), c, 0, 0, 0);
                return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, b1), __builtin_bit_cast(v8bf, a1), c, 0, 0, 0);
            }
        }
    };
    // NT, fp8: chunks kg*4 + half*2 + {0, 1} are 32 consecutive bytes of K; i8 / bf16: chunks kg*4 + half + {0, 2} feed two MFMAs
    constexpr int CSTEP = TYPE == T_FP8 ? 1 : 2;
    const int c0 = kg * 4 + (TYPE == T_FP8 ? half * 2 : half);
    const int ch0 = (c0 ^ (l32 & 15)) << 4, ch1 = ((c0 + CSTEP) ^ (l32 & 15)) << 4;
    // TN (see the ring kernel for what a transposing read hands to which lane)
    int tA[2], tB[2];
    constexpr int PA = SBM * ESZ, PB = SBN * ESZ; // bytes of a contraction row in the stage
    if constexpr (TN && ESZ == 1) {
        const int e8 = (lane & 15) >> 1, kr = kg * 64 + 32 * half + e8, part = 16 * ((lane >> 4) & 1) + 8 * (lane & 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            tA[i] = kr * PA + ((i ^ ((e8 >> 2) & 1)) << 5) + part;
            tB[i] = kr * PB + (((wn * 2 + i) ^ ((e8 >> 1) & 3)) << 5) + part;
        }
    } else if constexpr (TN) {
        const int e4 = (lane & 15) >> 2, kr = kg * 32 + 8 * half + e4, part = 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            tA[i] = kr * PA + ((i ^ ((e4 >> 1) & 1)) << 6) + part;
            tB[i] = kr * PB + (((wn * 2 + i) ^ (e4 & 3)) << 6) + part;
        }
    }
    typedef int v2i_t __attribute__((ext_vector_type(2)));
    auto fragT = [&](const uint8_t *base, int off, int pitch) -> v8i {
        const __attribute__((address_space(3))) uint8_t *q = (const __attribute__((address_space(3))) uint8_t *)TS2_LDS_PTR(base) + off;
        v2i_t r0, r1, r2, r3;
        if constexpr (ESZ == 1) {
            typedef __attribute__((address_space(3))) v2i_t *TTr8;
            r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q));
            r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 8 * pitch));
            r2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 16 * pitch));
            r3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 24 * pitch));
        } else {
            typedef short v4s_t __attribute__((ext_vector_type(4)));
            typedef __attribute__((address_space(3))) v4s_t *TTr16;
            r0 = __builtin_bit_cast(v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((TTr16)(q)));
            r1 = __builtin_bit_cast(v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((TTr16)(q + 4 * pitch)));
            r2 = __builtin_bit_cast(v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((TTr16)(q + 16 * pitch)));
            r3 = __builtin_bit_cast(v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((TTr16)(q + 20 * pitch)));
        }
        return v8i{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
    };
    auto multiply = [&](int step, int stage) {
        if (oddTail && step == nSteps - 1 && kg >= 2) { // (uniform over the wave)
            return;
        }
        const uint8_t *st = lds + stage * STAGE;
        v8i fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (TN) {
                fa[i] = fragT(st, tA[i], PA);
                fb[i] = fragT(st + SA, tB[i], PB);
            } else {
                const uint8_t *ar = st + (i * 32 + l32) * SK, *br = st + SA + (wn * 64 + i * 32 + l32) * SK;
                const v4i a0 = *(const v4i *)(ar + ch0), a1 = *(const v4i *)(ar + ch1);
                const v4i b0 = *(const v4i *)(br + ch0), b1 = *(const v4i *)(br + ch1);
                fa[i] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
                fb[i] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[i][j] = mul8(fa[i], fb[j], acc[i][j]);
            }
        }
    };
#define SLICE_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

    // ---- products
    auto factorOf = [&](int seg) -> float {
        float f = seg == 0 ? p.alpha : seg == 1 ? p.segAlpha[0] : seg == 2 ? p.segAlpha[1] : p.segAlpha[2];
        const float *q = seg == 0 ? alphaPtr : seg == 1 ? p.segAlphaPtr[0] : seg == 2 ? p.segAlphaPtr[1] : p.segAlphaPtr[2];
        return q ? f * *q : f;
    };
    auto aOf = [&](int seg) { return seg == 0 ? p.a : seg == 1 ? p.segA[0] : seg == 2 ? p.segA[1] : p.segA[2]; };
    auto bOf = [&](int seg) { return (seg == 0 ? bBase : seg == 1 ? p.segB[0] : seg == 2 ? p.segB[1] : p.segB[2]) + bSlab; };
    // partial tiles of the four wave pairs -> LDS, sums of the thread's 16 columns back.  16-byte chunks of a 512-byte row are swizzled
    // by the row like the stages.
    float val[16]; // KT: the scaled sum over the k-tiles; otherwise set from the sum
    auto partials = [&]() {
        SLICE_BARRIER(); // every wave has read its last operands
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = i * 32 + l32;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int cc = wn * 16 + j * 8 + q * 2 + half;
                    uint8_t *d = lds + kg * (SBM * SBN * 4) + r * 512 + ((cc ^ (r & 15)) << 4);
                    if constexpr (TYPE == T_I8) {
                        *(int4 *)d = make_int4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                    } else {
                        *(float4 *)d = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                    }
                }
            }
        }
        __syncthreads();
    };
    auto reduce = [&](TAcc &sum) {
        partials();
        if constexpr (KT) {
            const float *ts = p.kTileScale + (sp.kTileScaleRows ? (int64_t)(rowBase / sp.kTileScaleRows) * (p.kBytes / p.kTileBytes) : 0) + kt0;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                val[e] = 0;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (g < ktCount) {
                    const float sc = ts[g];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int4 v = *(const int4 *)(lds + g * (SBM * SBN * 4) + er * 512 + ((chunkOf(c) ^ (er & 15)) << 4));
                        val[c * 4 + 0] += sc * (float)v.x;
                        val[c * 4 + 1] += sc * (float)v.y;
                        val[c * 4 + 2] += sc * (float)v.z;
                        val[c * 4 + 3] += sc * (float)v.w;
                    }
                }
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint8_t *s = lds + er * 512 + ((chunkOf(c) ^ (er & 15)) << 4);
            typedef typename std::conditional<TYPE == T_I8, v4i, v4f>::type TQuad;
            const TQuad q0 = *(const TQuad *)s, q1 = *(const TQuad *)(s + SBM * SBN * 4), q2 = *(const TQuad *)(s + 2 * (SBM * SBN * 4)),
                        q3 = *(const TQuad *)(s + 3 * (SBM * SBN * 4));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[c * 4 + e] = (q0[e] + q1[e]) + (q2[e] + q3[e]);
            }
        }
    };
    // the steps of the products in `list` (two bits each, `count` of them) as one pipeline
    auto runProducts = [&](unsigned list, int count, float &units) {
        unsigned loadList = list;
        int loadStepNo = 0, loaded = 0;
        const int total = count * nSteps;
        auto loadNext = [&]() {
            const int seg = loadList & 3;
            loadStep(aOf(seg), bOf(seg), loadStepNo, loaded % NSTAGE);
            ++loaded;
            if (++loadStepNo == nSteps) {
                loadStepNo = 0;
                loadList >>= 2;
            }
        };
        if (total > 0) {
            loadNext();
        }
        if (total > 1) {
            loadNext();
        }
        int step = 0, stage = 0;
        for (int t = 0; t < total; ++t) {
            if (t + 1 < total) {
                asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            SLICE_BARRIER(); // step t is in LDS, and every wave is done with the stage that step t+2 goes to
            if (t + 2 < total) {
                loadNext();
            }
            multiply(step, stage);
            stage = stage == NSTAGE - 1 ? 0 : stage + 1;
            if (++step == nSteps) {
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
                                for (int j = 0; j < 2; ++j) {
#pragma unroll
                                    for (int e = 0; e < 16; ++e) {
                                        acc[i][j][e] *= ratio;
                                    }
                                }
                            }
                            units = nxt;
                        }
                    }
                }
            }
        }
    };
    TAcc sum;
    float sumScale = 1.f; // factor of `sum` in the epilogue
    bool done = false;
    if constexpr (TYPE == T_I8 && !TN && !KT) {
        if ((p.nSeg == 2 || (p.nSeg == 4 && p.kBytes <= 1536)) && !p.tileGroup && !p.groupOffsets && p.splits <= 1) {
            // Two or four products with row scales of their own: wave pair kg takes the kg-th product, or half of the (kg / 2)-th, so that all of
            // them are one pipeline and one reduction; one after the other, each paid its start and its reduction.  Four of K = 256: 512x256 12.5 ->
            // 7.8 us, 4096x512 15.5 -> 10.7, 8192x512 29.6 -> 19.4; two of 1024: 11.3 -> 9.8, 14.3 -> 12.7, 25.4 -> 23.5.  The operands of a load's four
            // lane groups lie in different arrays, and four products fetch half lines: at K = 2048 that costs what the rest gains (8192x512 71.3 ->
            // 73.9)
            done = true;
            const int share = p.nSeg == 2 ? 1 : 0, steps = (p.kBytes / 64) >> share; // (the halves are every other 64 bytes: whole lines)
            const uint8_t *aPtr[2], *bPtr[4];
            {
                const int r = lane >> 4, slot = lane & 15;
                auto at = [&](int rr, const uint8_t *q0, const uint8_t *q1, const uint8_t *q2, const uint8_t *q3, int64_t ld, int base) {
                    const int ch = slot ^ (rr & 15), pair = ch >> 2, seg = pair >> share;
                    const uint8_t *q = seg == 0 ? q0 : seg == 1 ? q1 : seg == 2 ? q2 : q3;
                    return q + (base + rr) * ld + (pair & ((1 << share) - 1)) * 64 + (ch & 3) * 16;
                };
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    aPtr[i] = at((wave + 8 * i) * 4 + r, p.a, p.segA[0], p.segA[1], p.segA[2], p.lda, rowBase);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bPtr[i] = at((wave + 8 * i) * 4 + r, p.b, p.segB[0], p.segB[1], p.segB[2], p.ldb, colBase);
                }
            }
            auto load = [&](int stage) {
                const unsigned st = ldsBase + stage * STAGE;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(st + (wave + 8 * i) * 1024), "v"(aPtr[i]) : "memory");
                    aPtr[i] += 64 << share;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(st + SA + (wave + 8 * i) * 1024), "v"(bPtr[i]) : "memory");
                    bPtr[i] += 64 << share;
                }
            };
            float rs[4]; // (on their way before the operands)
#pragma unroll
            for (int seg = 0; seg < 4; ++seg) {
                const float *rsp = seg == 0 ? p.rowScale : seg == 1 ? p.segRowScale[0] : seg == 2 ? p.segRowScale[1] : p.segRowScale[2];
                rs[seg] = seg < p.nSeg && rsp ? rsp[row] : 1.f;
            }
            zeroAcc();
            load(0);
            if (steps > 1) {
                load(1);
            }
            int stage = 0;
            for (int t = 0; t < steps; ++t) {
                if (t + 1 < steps) {
                    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
                } else {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                SLICE_BARRIER();
                if (t + 2 < steps) {
                    load(stage == 0 ? NSTAGE - 1 : stage - 1);
                }
                multiply(-1, stage);
                stage = stage == NSTAGE - 1 ? 0 : stage + 1;
            }
            const float f[4] = {factorOf(0) * rs[0], factorOf(1) * rs[1], p.nSeg > 2 ? factorOf(2) * rs[2] : 0.f, p.nSeg > 2 ? factorOf(3) * rs[3] : 0.f};
            partials();
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint8_t *q = lds + er * 512 + ((chunkOf(c) ^ (er & 15)) << 4);
                const v4i q0 = *(const v4i *)q, q1 = *(const v4i *)(q + SBM * SBN * 4), q2 = *(const v4i *)(q + 2 * (SBM * SBN * 4)),
                          q3 = *(const v4i *)(q + 3 * (SBM * SBN * 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = c * 4 + e;
                    if (share) {
                        out[k] = out[k] + (float)(q0[e] + q1[e]) * f[0];
                        sum[k] = q2[e] + q3[e];
                    } else {
                        out[k] = out[k] + (float)q0[e] * f[0];
                        out[k] = out[k] + (float)q1[e] * f[1];
                        out[k] = out[k] + (float)q2[e] * f[2];
                        sum[k] = q3[e];
                    }
                }
            }
            sumScale = share ? f[1] : f[3];
        }
    }
    if constexpr (TYPE == T_I8) {
        for (int seg = 0; seg < p.nSeg && !done; ++seg) {
            zeroAcc();
            float f = factorOf(seg);
            const float *rsp = seg == 0 ? p.rowScale : seg == 1 ? p.segRowScale[0] : seg == 2 ? p.segRowScale[1] : p.segRowScale[2];
            if (rsp) {
                f *= rsp[row];
            }
            float unused = 0;
            runProducts(seg, 1, unused);
            reduce(sum);
            if (seg + 1 < p.nSeg) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    out[e] = out[e] + (float)sum[e] * f;
                }
                __syncthreads(); // the partial tiles have been read: the stages may be refilled
            }
            sumScale = f;
        }
    } else {
        // a product with factor zero (the scale of an all-zero matrix) adds nothing and is left out: it has no units to convert into
        unsigned list = 0;
        int count = 0;
        float units = factorOf(0);
        if (p.nSeg == 1) {
            count = 1;
        } else {
            for (int seg = p.nSeg - 1; seg >= 0; --seg) {
                const float f = factorOf(seg);
                if (f != 0) {
                    list = (list << 2) | seg;
                    ++count;
                    units = f;
                }
            }
        }
        zeroAcc();
        runProducts(list, count, units);
        reduce(sum);
        sumScale = units;
        if (p.rowScale) {
            sumScale *= p.rowScale[row];
        }
    }

    // ---- epilogue
    if (ct == C_I32) {
        if constexpr (TYPE == T_I8 && !KT) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                *(int4 *)(cRow + (int64_t)(colBase + chunkOf(c) * 4) * 4) = make_int4(sum[c * 4], sum[c * 4 + 1], sum[c * 4 + 2], sum[c * 4 + 3]);
            }
        }
        return;
    }
    if constexpr (!KT) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            val[e] = (float)sum[e];
        }
    }
    if (ct == C_I8PACK) {
        float mx = 0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            mx = fmaxf(mx, fabsf(val[e]));
        }
        mx = fmaxf(mx, LaneDpp<DPP_XOR1>(mx));
        mx = fmaxf(mx, LaneDpp<DPP_XOR2>(mx));
        mx = fmaxf(mx, LaneDpp<DPP_HALF_MIRROR>(mx));
        mx *= fabsf(sumScale);
        float discr = 0, mult = 0;
        if (mx > 0 && live) {
            discr = mx / 127;
            mult = 1 / discr;
        }
        uint32_t w[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            w[c] = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                w[c] |= (uint32_t)(CvtToI8(val[c * 4 + e] * sumScale * mult) & 0xff) << (8 * e);
            }
        }
        *(uint4 *)(cRow + colBase + eu * 16) = make_uint4(w[0], w[1], w[2], w[3]);
        if (eu == 0) {
            tileScale[(int64_t)tn * p.ldTileScale + row] = discr;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        out[e] = live ? out[e] + val[e] * sumScale : 0.f;
    }
    if (ct == C_BF16NORM) {
        if (normalize) {
            // the association of the stand-alone pass (sums of four columns, then a butterfly over the 32 of them), so that the stored rows
            // do not depend on whether this epilogue or that pass normalised them
            float q[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                q[c] = (out[c * 4] * out[c * 4] + out[c * 4 + 1] * out[c * 4 + 1]) + (out[c * 4 + 2] * out[c * 4 + 2] + out[c * 4 + 3] * out[c * 4 + 3]);
            }
            float lo = q[0] + q[1], hi = q[2] + q[3];
            lo += LaneDpp<DPP_XOR1>(lo);
            hi += LaneDpp<DPP_XOR1>(hi);
            lo += LaneDpp<DPP_XOR2>(lo);
            hi += LaneDpp<DPP_XOR2>(hi);
            lo += LaneDpp<DPP_HALF_MIRROR>(lo);
            hi += LaneDpp<DPP_HALF_MIRROR>(hi);
            const float sum2 = lo + hi;
            float discr = 0;
            if (sum2 > 0) {
                discr = sqrtf(sum2 / TILE) * p.vecScale; // (once per row and lane: the exact forms cost nothing here)
                const float inv = 1 / discr;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    out[e] *= inv;
                }
            }
            if (eu == 0) {
                tileScale[(int64_t)tn * p.ldTileScale + row] = discr;
            }
        }
        if (rotate && live) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float4 cs = *(const float4 *)(p.rope + (int64_t)row * p.ldRope + chunkOf(c) * 4);
                const float x0 = out[c * 4], y0 = out[c * 4 + 1], x1 = out[c * 4 + 2], y1 = out[c * 4 + 3];
                out[c * 4] = x0 * cs.x - y0 * cs.y;
                out[c * 4 + 1] = y0 * cs.x + x0 * cs.y;
                out[c * 4 + 2] = x1 * cs.z - y1 * cs.w;
                out[c * 4 + 3] = y1 * cs.z + x1 * cs.w;
            }
        }
    }
    if (sp.epi == TS2_EPI_ADD && !live) {
        return;
    }
    if (ct == C_F32) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            *(float4 *)(cRow + (int64_t)(colBase + chunkOf(c) * 4) * 4) = make_float4(out[c * 4], out[c * 4 + 1], out[c * 4 + 2], out[c * 4 + 3]);
        }
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                w[k] = ct == C_F16 ? PackF16x2(out[h * 8 + 2 * k], out[h * 8 + 2 * k + 1]) : PackBf16x2(out[h * 8 + 2 * k], out[h * 8 + 2 * k + 1]);
            }
            *(uint4 *)(cRow + (int64_t)(colBase + h * 64 + eu * 8) * 2) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}
} // namespace

namespace gemmk
{
bool SliceCanRun(const SliceP &sp, int type, bool tn)
{
    const GemmP &p = sp.g;
    // (a contraction of whole 128-byte units: what is left over would not be multiplied)
    if (p.m <= 0 || p.n <= 0 || p.kBytes <= 0 || (p.m % SBM) || (p.n % SBN) || (p.kBytes % BKB) || (p.splits > 1 && p.groupOffsets) || p.splitK > 1) {
        return false;
    }
    if (tn && (int64_t)sp.kLive * (type == T_BF16 ? 2 : 1) > p.kBytes) {
        return false;
    }
    if (type == T_I8 ? (sp.ct == C_F16 && sp.epi != TS2_EPI_STORE) : sp.ct == C_I32) {
        return false;
    }
    if (sp.epi == TS2_EPI_ADD && sp.ct != C_F32 && sp.ct != C_BF16) {
        return false;
    }
    if (((uintptr_t)p.c | (uintptr_t)p.ldc | (uintptr_t)p.a | (uintptr_t)p.lda | (uintptr_t)p.b | (uintptr_t)p.ldb | (uintptr_t)p.cSlab |
            (uintptr_t)p.splitSlab) & 15) {
        return false;
    }
    if (sp.ct == C_BF16NORM && p.rope && (((uintptr_t)p.rope & 15) || (p.ldRope & 3))) {
        return false;
    }
    if (sp.ct == C_I8PACK && p.nSeg > 1) {
        return false;
    }
    if (p.jobs > 1) {
        if (p.jobs > 4 || sp.ct != C_BF16NORM || sp.epi != TS2_EPI_STORE || tn || p.splits > 1 || p.groupOffsets || p.tileGroup || p.nSeg > 1 ||
            p.kTileScale || (p.jobRope && !p.rope)) {
            return false;
        }
        for (int i = 0; i < p.jobs; ++i) {
            if (((uintptr_t)p.jobB[i] | (uintptr_t)p.jobC[i]) & 15 || (((p.jobNormalize >> i) & 1) && !p.jobTileScale[i])) {
                return false;
            }
        }
    }
    if (p.kTileScale) {
        // whole k-tiles of whole steps, up to four per workgroup; the sets of scales change between workgroups only
        if (p.kTileBytes <= 0 || (p.kTileBytes % 64) || (p.kBytes % p.kTileBytes)) {
            return false;
        }
        const int tiles = p.kBytes / p.kTileBytes, slices = p.splits > 1 ? p.splits : 1;
        if (type != T_I8 || p.groupOffsets || p.nSeg > 1 || sp.ct == C_I32 || (tiles + slices - 1) / slices > 4 || (sp.kTileScaleRows % SBM)) {
            return false;
        }
    }
    // lane offsets inside a tile and a step are 32-bit
    const int64_t aRows = tn ? (p.kTileScale ? 4 * p.kTileBytes : SK) : SBM, bRows = tn ? (p.kTileScale ? 4 * p.kTileBytes : SK) : SBN;
    return aRows * p.lda < ((int64_t)1 << 30) && bRows * p.ldb < ((int64_t)1 << 30);
}

int RunSlice(const SliceP &in, int type, bool tn, hipStream_t stream)
{
    if (!SliceCanRun(in, type, tn)) {
        return TS2_ERR_UNSUPPORTED;
    }
    SliceP sp = in;
    sp.g.tilesM = sp.g.m / SBM;
    sp.g.tilesN = sp.g.n / SBN;
    const dim3 grid(sp.g.tilesM * sp.g.tilesN, sp.g.groupOffsets ? sp.g.splitK_groups : sp.g.splits > 1 ? sp.g.splits : 1,
        sp.g.jobs > 1 ? sp.g.jobs : 1);
    if (type == T_I8 && sp.g.kTileScale) {
        if (tn) {
            hipLaunchKernelGGL((GemmSlice<T_I8, true, true>), grid, dim3(512), 0, stream, sp);
        } else {
            hipLaunchKernelGGL((GemmSlice<T_I8, false, true>), grid, dim3(512), 0, stream, sp);
        }
    } else if (type == T_I8) {
        if (tn) {
            hipLaunchKernelGGL((GemmSlice<T_I8, true>), grid, dim3(512), 0, stream, sp);
        } else {
            hipLaunchKernelGGL((GemmSlice<T_I8, false>), grid, dim3(512), 0, stream, sp);
        }
    } else if (type == T_FP8) {
        if (tn) {
            hipLaunchKernelGGL((GemmSlice<T_FP8, true>), grid, dim3(512), 0, stream, sp);
        } else {
            hipLaunchKernelGGL((GemmSlice<T_FP8, false>), grid, dim3(512), 0, stream, sp);
        }
    } else {
        if (tn) {
            hipLaunchKernelGGL((GemmSlice<T_BF16, true>), grid, dim3(512), 0, stream, sp);
        } else {
            hipLaunchKernelGGL((GemmSlice<T_BF16, false>), grid, dim3(512), 0, stream, sp);
        }
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}
} // namespace gemmk
