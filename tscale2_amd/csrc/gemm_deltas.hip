// Packed deltas of many matrices in one launch: what a backward pass of a model with small products leaves for its end (layers.hip).  One
// by one such deltas have 16 to 250 tiles, pay a launch, a start and a tail each, and run on the 64x128 tiles of the kernel for few
// tiles, whose operands cost a line of L2 for every 64 bytes of A; together they fill the chip with larger ones.
//
// A workgroup of eight waves (64x64 accumulators each) owns 256 x 128 of one delta and walks the whole contraction in steps of 128 rows:
// 48 KB of operands, both contraction-major as they lie, global -> LDS without registers, three stages, two of them under way while one is
// multiplied (the pipeline, the transposing reads and the waits are those of gemm_slice.hip).  The bound is the path from L2 to LDS: 64x128
// tiles fetch 48 KB for 2.1 M multiply-adds and 512 lines, these for 4.2 M and 384.  A lane owns a row of the result (operands swapped), so the
// packing's row maxima need one exchange between the two waves of a row; the bytes leave through LDS as whole 128-byte rows.
// Measured (MI355X): 16 products of the e512 d8 int8 step (16384 rows, 464 GOP) 902 us + 180 of packing their slices -> 321; those of a step of 512 x
// 2048 over 4096 tokens in e4m3 (146 GFLOP) 286 + 23 -> 100; of 256 x 1024 over 512 tokens in int8 184 -> 14.  The same batch on 64x128 tiles: 708, 162, 26.
// i8: one scale per kTile rows; the exact int32 sums of up to four k-tiles are added, scaled, in fp32, and these sums to each other, both in tile order: the
// sums of the delta products one by one, bit by bit.  (One chain over all k-tiles had 1.6 times their error from 64 bits at 32 k-tiles.)
#include "gemm_deltas.h"

using namespace gemmk;

namespace
{
constexpr int DBM = 256, DBN = 128, DK = 128; // tile, contraction rows of a step
constexpr int DA = DK * DBM, DSTAGE = DK * (DBM + DBN), DSTAGES = 3;
constexpr int DPITCH = DBN + 16; // bytes between packed rows in LDS
constexpr int DGROUP = 4;        // tile rows that are walked together

typedef __attribute__((address_space(3))) uint8_t *TLds3;

template <int TYPE> __global__ void __launch_bounds__(512, 2) GemmDeltas(DeltaBatchP bp)
{
    typedef typename AccT<TYPE>::type TAcc;
    constexpr bool KT = TYPE == T_I8;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[DSTAGES * DSTAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, half = lane >> 5, l32 = lane & 31;
    const unsigned ldsBase = (unsigned)(uintptr_t)(TLds3)lds;

    // an XCD takes consecutive tiles of the whole list: its L2 holds the operands of one or two products, not an eighth of every one
    const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); // (the grid is a multiple of eight)
    int j = 0;
    while (j + 1 < bp.count && id >= bp.job[j + 1].first) {
        ++j;
    }
    const DeltaJob &d = bp.job[j];
    const int tilesM = (d.gradDim + DBM - 1) / DBM, tilesN = d.srcDim / DBN;
    if (id - d.first >= tilesM * tilesN) {
        return; // (the last workgroups of the grid)
    }
    int tm, tn;
    MapTile(id - d.first, 1, tilesM, tilesN, &tm, &tn, DGROUP);
    const int rowBase = tm * DBM, colBase = tn * DBN;
    const int rowsHere = min(d.gradDim - rowBase, DBM); // 256, or 128 at the end of an odd number of 128s
    const int lda = d.ldGrad, ldb = d.ldSrc;

    // ---- loader: 48 wave-level loads of 1 KB per step, six per wave.  A: 4 contraction rows of 256 bytes, B: 8 of 128; the granules of one MFMA
    // block (32 tile columns) are XOR-swizzled by the row so that a transposing read of 8 rows covers all banks once
    int aOff[4], bOff[2];
    {
        const int ra = lane >> 4, sa = lane & 15, rb = lane >> 3, sb = lane & 7;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = (wave + 8 * i) * 4 + ra;
            const int col = (((sa >> 1) ^ (rr & 7)) << 5) + (sa & 1) * 16;
            aOff[i] = rr * lda + (col < rowsHere ? col : col - 128); // (no such column: any valid bytes, their sums are not stored)
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int rr = (wave + 8 * i) * 8 + rb;
            bOff[i] = rr * ldb + (((sb >> 1) ^ ((rr >> 1) & 3)) << 5) + (sb & 1) * 16;
        }
    }
    const int live = KT ? bp.kBytes : bp.kLive; // (i8: rows beyond the live ones hold zeros)
    const int steps = (live + DK - 1) / DK;
    auto loadStep = [&](int step, int stage) {
        const unsigned st = ldsBase + stage * DSTAGE;
        const int k0 = step * DK, rows = min(live - k0, DK); // later rows read as zeros: the descriptor ends there
        const v4i ra = BufferRsrc(d.grad + (int64_t)k0 * lda + rowBase, (rows - 1) * lda + rowsHere);
        const v4i rb = BufferRsrc(d.src + (int64_t)k0 * ldb + colBase, (rows - 1) * ldb + DBN);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            TS2_LOAD_LDS16(st + (wave + 8 * i) * 1024, aOff[i], ra);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            TS2_LOAD_LDS16(st + DA + (wave + 8 * i) * 1024, bOff[i], rb);
        }
    };

    // ---- operand fragments (see the ring kernel for what a transposing read hands to which lane)
    int tA[2], tB[2];
    {
        const int e8 = (lane & 15) >> 1, kr = 32 * half + e8, part = 16 * ((lane >> 4) & 1) + 8 * (lane & 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            tA[i] = kr * DBM + (((wm * 2 + i) ^ e8) << 5) + part;
            tB[i] = DA + kr * DBN + (((wn * 2 + i) ^ ((e8 >> 1) & 3)) << 5) + part;
        }
    }
    typedef int v2i_t __attribute__((ext_vector_type(2)));
    auto frag = [&](const uint8_t *st, int off, int pitch) -> v8i {
        typedef __attribute__((address_space(3))) v2i_t *TTr8;
        const __attribute__((address_space(3))) uint8_t *q = (const __attribute__((address_space(3))) uint8_t *)TS2_LDS_PTR(st) + off;
        const v2i_t r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q)), r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 8 * pitch)),
                    r2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 16 * pitch)), r3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((TTr8)(q + 24 * pitch));
        return v8i{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
    };
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
    auto multiply = [&](int stage) {
        const uint8_t *st = lds + stage * DSTAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            v8i fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = frag(st, tA[i] + u * 64 * DBM, DBM);
                fb[i] = frag(st, tB[i] + u * 64 * DBN, DBN);
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
#define DELTA_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

    // ---- k-tiles (i8)
    const int kTiles = KT ? bp.kBytes / bp.kTileBytes : 0, perTile = KT ? bp.kTileBytes / DK : 0;
    const float *scales = KT ? d.kTileScale + (d.kTileScaleRows ? (int64_t)min((rowBase + wm * 64) / d.kTileScaleRows, (d.gradDim - 1) / d.kTileScaleRows) * kTiles : 0) : nullptr;
    float total[2][2][16], part[KT ? 2 : 1][2][16];
    float kScale = 0; // lane i: scale of k-tile i of the current 64
    if constexpr (KT) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    total[i][n][e] = 0;
                    part[i][n][e] = 0;
                }
            }
        }
    }
    int left = bp.kGroup;
    auto endOfTile = [&](int kt) {
        if ((kt & 63) == 0) {
            kScale = kt + lane < kTiles ? scales[kt + lane] : 0.f;
        }
        const float sc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(kScale), kt & 63));
        const bool last = --left == 0 || kt + 1 == kTiles;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    part[i][n][e] = __builtin_fmaf(sc, (float)acc[i][n][e], part[i][n][e]);
                }
            }
        }
        if (last) {
            left = bp.kGroup;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        total[i][n][e] += part[i][n][e];
                        part[i][n][e] = 0;
                    }
                }
            }
        }
        zeroAcc();
    };

    zeroAcc();
    loadStep(0, 0);
    if (steps > 1) {
        loadStep(1, 1);
    }
    int stage = 0, inTile = 0, kt = 0;
    for (int t = 0; t < steps; ++t) {
        if (t + 1 < steps) {
            asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        DELTA_BARRIER(); // step t is in LDS, and every wave is done with the stage that step t+2 goes to
        if (t + 2 < steps) {
            loadStep(t + 2, stage == 0 ? 2 : stage - 1);
        }
        multiply(stage);
        stage = stage == DSTAGES - 1 ? 0 : stage + 1;
        if constexpr (KT) {
            if (++inTile == perTile) {
                inTile = 0;
                endOfTile(kt);
                ++kt;
            }
        }
    }
    if constexpr (!KT) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    total[i][n][e] = acc[i][n][e];
                }
            }
        }
    }

    // ---- packing: a lane holds, of row wm * 64 + i * 32 + l32, columns wn * 64 + n * 32 + q * 8 + half * 4 + 0 .. 3
    const float factor = d.alphaPtr ? d.alpha * *d.alphaPtr : d.alpha;
    float *const rowMax = (float *)lds;      // [2][256]
    uint8_t *const bytes = lds + 2 * 256 * 4; // [256][DPITCH]
    DELTA_BARRIER(); // every wave has read its last operands
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float mx = 0;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                mx = fmaxf(mx, fabsf(total[i][n][e]));
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (half == 0) {
            rowMax[wn * 256 + wm * 64 + i * 32 + l32] = mx;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = wm * 64 + i * 32 + l32;
        const float mx = fmaxf(rowMax[r], rowMax[256 + r]) * fabsf(factor);
        float discr = 0, mult = 0;
        if (mx > 0) {
            discr = mx / 127;
            mult = 1 / discr;
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    w |= (uint32_t)(CvtToI8(total[i][n][q * 4 + e] * factor * mult) & 0xff) << (8 * e);
                }
                *(uint32_t *)(bytes + r * DPITCH + wn * 64 + n * 32 + q * 8 + half * 4) = w;
            }
        }
        if (wn == 0 && half == 0 && r < rowsHere) {
            d.tileScale[(int64_t)tn * d.ldTileScale + rowBase + r] = discr;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int r = (tid >> 3) + 64 * k, c = (tid & 7) * 16;
        if (r < rowsHere) {
            *(uint4 *)(d.delta + (int64_t)(rowBase + r) * d.ldDelta + colBase + c) = *(const uint4 *)(bytes + r * DPITCH + c);
        }
    }
}
} // namespace

namespace gemmk
{
bool DeltaBatchCanRun(const DeltaJob &d, int type, int kBytes, int kLive, int kTileBytes)
{
    if ((type != T_I8 && type != T_FP8) || !d.grad || !d.src || !d.delta || !d.tileScale || d.gradDim <= 0 || d.srcDim <= 0 || (d.gradDim % 128) ||
        (d.srcDim % DBN) || kLive <= 0 || kLive > kBytes || d.ldGrad < d.gradDim || d.ldSrc < d.srcDim || d.ldDelta < d.srcDim) {
        return false;
    }
    if (type == T_I8 && (!d.kTileScale || kTileBytes <= 0 || (kTileBytes % DK) || (kBytes % kTileBytes) || (d.kTileScaleRows % 64))) {
        return false;
    }
    // lane offsets inside a step are 32-bit
    return !(((uintptr_t)d.grad | (uintptr_t)d.src | (uintptr_t)d.delta | (uintptr_t)d.ldGrad | (uintptr_t)d.ldSrc | (uintptr_t)d.ldDelta) & 15) &&
           d.ldGrad < (1 << 23) && d.ldSrc < (1 << 23);
}

int RunDeltaBatch(const DeltaJob *jobs, int count, int type, int kBytes, int kLive, int kTileBytes, hipStream_t stream)
{
    // (the groups of Ts2DeltaRows: as few as hold four k-tiles each at most, of equal size)
    const int kTiles = type == T_I8 && kTileBytes > 0 && kBytes > kTileBytes ? kBytes / kTileBytes : 1, groups = (kTiles + 3) / 4, kGroup = (kTiles + groups - 1) / groups;
    for (int done = 0; done < count;) {
        DeltaBatchP bp = {};
        bp.kBytes = kBytes;
        bp.kLive = kLive;
        bp.kTileBytes = kTileBytes;
        bp.kGroup = kGroup;
        int blocks = 0;
        for (; done < count && bp.count < DELTA_JOBS; ++done) {
            if (!DeltaBatchCanRun(jobs[done], type, kBytes, kLive, kTileBytes)) {
                return TS2_ERR_UNSUPPORTED;
            }
            DeltaJob &d = bp.job[bp.count++];
            d = jobs[done];
            d.first = blocks;
            blocks += (d.gradDim + DBM - 1) / DBM * (d.srcDim / DBN);
        }
        const dim3 grid((blocks + 7) / 8 * 8);
        if (type == T_I8) {
            hipLaunchKernelGGL((GemmDeltas<T_I8>), grid, dim3(512), 0, stream, bp);
        } else {
            hipLaunchKernelGGL((GemmDeltas<T_FP8>), grid, dim3(512), 0, stream, bp);
        }
        TS2_CHECK_LAUNCH();
    }
    return TS2_OK;
}
} // namespace gemmk
