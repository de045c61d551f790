// Linear-layer backward operator: the call sequences of TMatMulBuffers (src/gpt/compute/layer_cuda_base.cuh:153-250) expressed
// over the kernels of this library.  Host code only; every step is enqueued on the caller's stream.
#include "common.h"
#include "gemm_slice.h"
#include "gemm_tall.h"
#include "internal.h"

namespace
{
bool Is8(int mode)
{
    return mode == TS2_I8 || mode == TS2_E4M3;
}

int SliceType(int mode)
{
    return mode == TS2_I8 ? gemmk::T_I8 : mode == TS2_E4M3 ? gemmk::T_FP8 : gemmk::T_BF16;
}

// the kernel for few tiles on row-major operands: splits == 1 packs the delta, otherwise fp32 slices go to `partial` (dense slabs)
int DeltaSlice(int mode, int len, int lenRound, int srcDim, int gradDim, const ts2_mat *src, const ts2_mat *grad, const float *kTileScale, int kTile,
    int kTileScaleRows, float alpha, const float *alphaPtr, int splits, float *partial, const ts2_mat *delta, const ts2_mat *tileScale, void *stream)
{
    gemmk::SliceP sp = {};
    gemmk::GemmP &g = sp.g;
    g.a = (const uint8_t *)grad->ptr;
    g.b = (const uint8_t *)src->ptr;
    g.lda = grad->strideBytes;
    g.ldb = src->strideBytes;
    g.m = gradDim;
    g.n = srcDim;
    g.kBytes = lenRound * (mode == TS2_BF16 ? 2 : 1);
    g.kTileScale = kTileScale;
    g.kTileBytes = kTile;
    g.nSeg = 1;
    sp.kLive = len;
    sp.kTileScaleRows = kTileScaleRows;
    sp.epi = TS2_EPI_STORE;
    if (len < 0 || len > lenRound || (gradDim % TILE) || grad->x < gradDim || src->x < srcDim || grad->y < len || src->y < len || delta->x < srcDim || delta->y < gradDim ||
        tileScale->x < gradDim || tileScale->y < srcDim / TILE || !grad->ptr || !src->ptr || !delta->ptr || !tileScale->ptr ||
        (kTileScale && (grad->y < lenRound || src->y < lenRound))) {
        return TS2_ERR_UNSUPPORTED; // (the general path, where there is one, names what is wrong)
    }
    if (splits > 1) {
        g.c = (uint8_t *)partial;
        g.ldc = (int64_t)srcDim * 4;
        g.splits = splits;
        g.splitSlab = (int64_t)gradDim * g.ldc;
        g.alpha = 1.f;
        sp.ct = gemmk::C_F32;
        int rc = gemmk::RunSlice(sp, SliceType(mode), true, (hipStream_t)stream);
        if (rc) {
            return rc;
        }
        ts2_mat part = {partial, g.ldc, srcDim, splits * gradDim};
        return ts2_pack_delta(&part, splits, g.splitSlab, gradDim, srcDim, alpha, alphaPtr, delta, tileScale, stream);
    }
    g.c = (uint8_t *)delta->ptr;
    g.ldc = delta->strideBytes;
    g.splits = 1;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.tileScale = (float *)tileScale->ptr;
    g.ldTileScale = tileScale->strideBytes / 4;
    sp.ct = gemmk::C_I8PACK;
    return gemmk::RunSlice(sp, SliceType(mode), true, (hipStream_t)stream);
}
} // namespace

extern "C" int ts2_matmul_bwd_scratch_bytes(int32_t mode, int32_t lenRound, int32_t srcDim, int32_t gradDim, int32_t kTile, int32_t splits,
    int64_t out[9])
{
    if (!out) {
        return TS2_ERR_NULL;
    }
    if (!Is8(mode)) {
        return TS2_ERR_UNSUPPORTED;
    }
    if (kTile <= 0) {
        kTile = 512;
    }
    if (srcDim <= 0 || gradDim <= 0 || lenRound <= 0 || srcDim % 128 || gradDim % 128 || lenRound % 128 || kTile % 128 || splits < 0 ||
        (mode == TS2_I8 && lenRound % kTile)) {
        return TS2_ERR_SHAPE;
    }
    const int64_t L = lenRound, S = srcDim, G = gradDim, nTiles = (L + kTile - 1) / kTile;
    const bool i8 = mode == TS2_I8;
    out[0] = i8 ? L * G : 0;         // grad8
    out[1] = i8 ? L * 4 : 0;         // grad8RowScale
    out[2] = G * L;                  // gradT
    out[3] = S * L;                  // srcT
    out[4] = i8 ? nTiles * 4 : 0;    // tileMax
    out[5] = i8 ? nTiles * 4 : 0;    // tileScale
    out[6] = S * G;                  // transformT
    out[7] = splits > 1 ? (int64_t)splits * G * S * 4 : 0; // partial
    out[8] = i8 ? L * 4 : 0;         // gradRowAbsMax (optional)
    return TS2_OK;
}

extern "C" int ts2_matmul_backprop_multi(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t gradDim,
    const ts2_mat *transformFast, const ts2_mat *grad, int32_t gradType, const float *gradColScale, const ts2_matmul_bwd_buffers *buf, void *stream)
{
    if (!transformFast || !buf) {
        return TS2_ERR_NULL;
    }
    if (!Is8(mode)) {
        return TS2_ERR_UNSUPPORTED;
    }
    if (srcDim % 128 || gradDim % 128 || lenRound % 128 || len > lenRound) {
        return TS2_ERR_SHAPE;
    }
    if (mode == TS2_I8) {
        if (!grad || !buf->grad8RowScale) {
            return TS2_ERR_NULL;
        }
        int rc = ts2_normalize_vecs_row_max_dither(len, lenRound, grad, gradType, gradColScale, &buf->grad8, buf->grad8RowScale, buf->gradRowAbsMax,
            buf->ditherSeed, stream);
        if (rc) {
            return rc;
        }
    }
    // W [gradDim][srcDim] -> W^T [srcDim][gradDim] so that the dX GEMM contracts over contiguous bytes
    if (buf->transformTValid) {
        return TS2_OK;
    }
    return ts2_transpose_quant(gradDim, gradDim, transformFast, mode, nullptr, nullptr, 0, nullptr, &buf->transformT, mode, nullptr, stream);
}

extern "C" int ts2_matmul_backprop(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t gradDim, const ts2_mat *grad,
    const ts2_matmul_bwd_buffers *buf, float alpha, const float *alphaPtr, const ts2_mat *srcGrad, int32_t srcGradType, int32_t add, void *stream)
{
    if (!buf || !srcGrad) {
        return TS2_ERR_NULL;
    }
    if (!Is8(mode)) {
        return TS2_ERR_UNSUPPORTED;
    }
    ts2_gemm_args g = {};
    if (mode == TS2_I8) {
        g.a = buf->grad8;
        g.rowScale = buf->grad8RowScale;
    } else {
        if (!grad) {
            return TS2_ERR_NULL;
        }
        g.a = *grad;
    }
    g.b = buf->transformT;
    g.c = *srcGrad;
    g.abType = mode;
    g.cType = srcGradType;
    g.m = lenRound;
    g.n = srcDim;
    g.k = gradDim;
    g.mLive = len;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.epilogue = add ? TS2_EPI_ADD : TS2_EPI_STORE;
    g.splitK = 1;
    return ts2_gemm_nt(&g, stream);
}

extern "C" int ts2_matmul_backprop_group(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t gradDim, int32_t count,
    const ts2_mat *const *grad, const ts2_matmul_bwd_buffers *const *bufs, const float *alpha, const float *const *alphaPtr,
    const ts2_mat *srcGrad, int32_t srcGradType, int32_t add, void *stream)
{
    if (!grad || !bufs || !alpha || !srcGrad || count < 1 || count > 4) {
        return TS2_ERR_NULL;
    }
    for (int i = 0; i < count; ++i) {
        if (!bufs[i] || (mode != TS2_I8 && !grad[i])) {
            return TS2_ERR_NULL;
        }
    }
    if (mode == TS2_E4M3) { // (one launch checks the first product's operands only)
        for (int i = 0; i < count; ++i) {
            const ts2_mat &t = bufs[i]->transformT;
            if (grad[i]->x < gradDim || grad[i]->y < lenRound || t.x < gradDim || t.y < srcDim) {
                return TS2_ERR_SHAPE;
            }
        }
    }
    // one launch: the 256x256 tile (or what the dispatcher puts in its place), off its grid the kernel for few tiles while it beats one product
    // after the other: one round of its workgroups always; two products of K = 2048 as two rounds 35.0 -> 31.8 us, as three 42.6 -> 45.8, of
    // K = 1024 as three 32.2 -> 29.5; four of K = 2048 as three 93.1 -> 80.7, of K = 4096 135 -> 147; two of K = 4096 as two 46.0 -> 52.8
    const bool grid256 = (lenRound % 256) == 0 && (srcDim % 256) == 0;
    const int64_t wgs = (int64_t)(lenRound / 64) * (srcDim / 128);
    const bool few = wgs <= 256 || (wgs <= 512 && gradDim <= 2048) || (wgs <= 640 && gradDim <= (count > 2 ? 2048 : 1024));
    bool one = mode == TS2_E4M3 && count > 1 && (srcGradType == TS2_F32 || srcGradType == TS2_BF16) && (grid256 || few);
    for (int i = 1; i < count && one; ++i) {
        one = grad[i]->strideBytes == grad[0]->strideBytes && bufs[i]->transformT.strideBytes == bufs[0]->transformT.strideBytes;
    }
    auto oneByOne = [&]() -> int {
        for (int i = 0; i < count; ++i) {
            int rc = ts2_matmul_backprop(mode, len, lenRound, srcDim, gradDim, grad[i], bufs[i], alpha[i], alphaPtr ? alphaPtr[i] : nullptr, srcGrad,
                srcGradType, add || i > 0, stream);
            if (rc) {
                return rc;
            }
        }
        return TS2_OK;
    };
    if (!one) {
        return oneByOne();
    }
    ts2_gemm_args g = {};
    g.a = *grad[0];
    g.b = bufs[0]->transformT;
    g.c = *srcGrad;
    g.abType = mode;
    g.cType = srcGradType;
    g.m = lenRound;
    g.n = srcDim;
    g.k = gradDim;
    g.mLive = len;
    g.alpha = alpha[0];
    g.alphaPtr = alphaPtr ? alphaPtr[0] : nullptr;
    g.epilogue = add ? TS2_EPI_ADD : TS2_EPI_STORE;
    g.splitK = 1;
    g.extraSegments = count - 1;
    for (int i = 1; i < count; ++i) {
        g.segment[i - 1].a = grad[i]->ptr;
        g.segment[i - 1].b = bufs[i]->transformT.ptr;
        g.segment[i - 1].alpha = alpha[i];
        g.segment[i - 1].alphaPtr = alphaPtr ? alphaPtr[i] : nullptr;
    }
    g.tileConfig = grid256 ? 0 : 65536;
    const int rc = ts2_gemm_nt(&g, stream);
    // (rows of the result off 16 bytes, strides beyond what the kernel for few tiles addresses: one product after the other)
    return rc == TS2_ERR_UNSUPPORTED && !grid256 ? oneByOne() : rc;
}

extern "C" int ts2_matmul_backprop_delta(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t gradDim, const ts2_mat *src,
    const float *srcRowScale, const ts2_mat *grad, int32_t gradType, float alpha, const float *gradScale, int32_t kTile, const ts2_matmul_bwd_buffers *buf,
    const ts2_mat *delta, const ts2_mat *deltaTileScale, void *stream)
{
    if (!buf || !src || !grad || !delta || !deltaTileScale) {
        return TS2_ERR_NULL;
    }
    if (!Is8(mode)) {
        return TS2_ERR_UNSUPPORTED;
    }
    int rc;
    bool kMajor = false;
    ts2_gemm_args g = {};
    if (mode == TS2_I8) {
        if (kTile <= 0 || kTile % 128 || lenRound % kTile || !buf->tileMax || !buf->tileScale) {
            return TS2_ERR_SHAPE;
        }
        if (buf->sortRows) {
            // the reference's order: rows sorted by their scale, gathered through the sorted list by both transposing passes
            if (!buf->gradRowAbsMax || !buf->gradRowAbsMaxValid || !buf->rowOrder || !buf->rowOrderTmp) {
                return TS2_ERR_NULL;
            }
            rc = ts2_sort_rows_by_scale(len, buf->gradRowAbsMax, srcRowScale, buf->rowOrder, buf->rowOrderTmp, stream);
            if (rc) {
                return rc;
            }
            rc = Ts2TransposeQuantRows(len, lenRound, grad, gradType, srcRowScale, nullptr, buf->gradRowAbsMax, kTile, buf->rowOrder, &buf->gradT,
                TS2_I8, buf->tileScale, stream, buf->ditherSeed);
        } else if (buf->gradRowAbsMax && buf->gradRowAbsMaxValid) {
            // the k-tile maxima follow from the row maxima of the dX pass: the transposing quantiser forms them itself
            rc = Ts2TransposeQuantRows(len, lenRound, grad, gradType, srcRowScale, nullptr, buf->gradRowAbsMax, kTile, nullptr, &buf->gradT, TS2_I8,
                buf->tileScale, stream, buf->ditherSeed);
        } else {
            rc = ts2_tile_absmax(len, grad, gradType, srcRowScale, kTile, buf->tileMax, 1, stream);
            if (rc) {
                return rc;
            }
            rc = ts2_transpose_quant_dither(len, lenRound, grad, gradType, srcRowScale, buf->tileMax, kTile, nullptr, &buf->gradT, TS2_I8, buf->tileScale,
                buf->ditherSeed, stream);
        }
        if (rc) {
            return rc;
        }
        g.kTileScale = buf->tileScale;
        g.kTile = kTile;
    } else {
        if (gradType != TS2_E4M3) {
            return TS2_ERR_UNSUPPORTED;
        }
        // both operands as they lie in memory, [token][feature]: the kernel's LDS reads do the transposing
        kMajor = (len == lenRound || buf->padRowsZero) && (gradDim % 256) == 0 && (srcDim % 256) == 0 && grad->y >= lenRound && src->y >= lenRound;
        // widths off the 256 grid, or pad rows that nobody vouches for: the kernel for few tiles, which stops at row len, in place of two
        // transposes and a product.  One round of its workgroups always; two up to 4096 rows (5120x512 over 2048 31.2 -> 20.0 us, 4096 38.1 ->
        // 35.6, 8192 57.9 -> 63.1; 2048x2048 over 4096 39.9 -> 32.0, 8192 57.3 -> 58.1)
        const int cuts = buf->partial.ptr && buf->splits > 1 ? buf->splits : 1;
        // (the scratch of the transposing sequence is part of the call, whichever kernel runs)
        const bool scratch = buf->gradT.ptr && buf->gradT.x >= lenRound && buf->gradT.y >= gradDim && buf->srcT.ptr && buf->srcT.x >= lenRound &&
                             buf->srcT.y >= srcDim;
        if (!kMajor && !buf->gradTValid && cuts == 1 && scratch && (int64_t)(gradDim / 64) * (srcDim / 128) <= (lenRound <= 4096 ? 512 : 256)) {
            rc = DeltaSlice(TS2_E4M3, len, lenRound, srcDim, gradDim, src, grad, nullptr, 0, 0, alpha, gradScale, 1, nullptr, delta, deltaTileScale, stream);
            if (rc != TS2_ERR_UNSUPPORTED) {
                return rc;
            }
        }
        if (!kMajor && !buf->gradTValid) {
            rc = ts2_transpose_quant(len, lenRound, grad, TS2_E4M3, nullptr, nullptr, 0, nullptr, &buf->gradT, TS2_E4M3, nullptr, stream);
            if (rc) {
                return rc;
            }
        }
    }
    const int *rowOrder = (mode == TS2_I8 && buf->sortRows) ? buf->rowOrder : nullptr;
    if (!kMajor && (mode == TS2_E4M3 || !buf->srcTValid || rowOrder)) {
        rc = ts2_transpose_quant(len, lenRound, src, mode, nullptr, nullptr, 0, rowOrder, &buf->srcT, mode, nullptr, stream);
        if (rc) {
            return rc;
        }
    }
    g.a = kMajor ? *grad : buf->gradT;
    g.b = kMajor ? *src : buf->srcT;
    g.kMajor = kMajor ? 1 : 0;
    g.abType = mode;
    g.m = gradDim;
    g.n = srcDim;
    g.k = lenRound;
    const int splits = buf->partial.ptr ? buf->splits : 1;
    if (splits > 1) {
        // few output tiles: slices of the token axis as separate stored products on the large tile, then pack their sum
        int esz = 1;
        int64_t sliceBytes = ((int64_t)lenRound * esz / 128 + splits - 1) / splits * 128;
        bool ok = buf->partial.y >= splits * gradDim && buf->partial.x >= srcDim && (mode != TS2_I8 || sliceBytes % kTile == 0);
        if (!ok) {
            return TS2_ERR_SHAPE;
        }
        g.c = buf->partial;
        g.c.y = gradDim;
        g.cType = TS2_F32;
        g.alpha = 1.f;
        g.epilogue = TS2_EPI_STORE;
        g.splitK = splits;
        g.splitSlabBytes = (int64_t)gradDim * buf->partial.strideBytes;
        // int8: 256x128 tile with eight waves (the k-tile conversions of one wave run under the other's MFMAs)
        g.tileConfig = mode == TS2_I8 ? ((gradDim % 256) == 0 ? (3 | 8) : 2) : (((gradDim % 256) == 0 && (srcDim % 256) == 0) ? 1 : 2);
        rc = ts2_gemm_nt(&g, stream);
        if (rc) {
            return rc;
        }
        return ts2_pack_delta(&buf->partial, splits, g.splitSlabBytes, gradDim, srcDim, alpha, gradScale, delta, deltaTileScale, stream);
    }
    g.c = *delta;
    g.cType = TS2_I8;
    g.alpha = alpha;
    g.alphaPtr = gradScale;
    g.epilogue = TS2_EPI_ROW_TILE_MAXNORM;
    g.tileScale = *deltaTileScale;
    g.splitK = 1;
    return ts2_gemm_nt(&g, stream);
}

extern "C" int ts2_matmul_forward(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t dstDim, const ts2_mat *src,
    const ts2_mat *transformFast, float alpha, const float *alphaPtr, const ts2_mat *res, int32_t resType, int32_t add, void *stream)
{
    if (!src || !transformFast || !res) {
        return TS2_ERR_NULL;
    }
    ts2_gemm_args g = {};
    g.a = *src;
    g.b = *transformFast;
    g.c = *res;
    g.abType = mode;
    g.cType = resType;
    g.m = lenRound;
    g.n = dstDim;
    g.k = srcDim;
    g.mLive = len;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.epilogue = add ? TS2_EPI_ADD : TS2_EPI_STORE;
    g.splitK = 1;
    return ts2_gemm_nt(&g, stream);
}

// Forward<TStoreRowTileNormalize> / Forward<TStoreRowTileNormalizeRope> of the same operator (layer_cuda_base.cuh:183-193 with the store
// functors of cuda_matmul.cuh:495-525 and gpu_rope.cuh:25-60): res = rope(normalise(alpha * (*alphaPtr) * src * W^T)) as bf16 plus the
// per-tile scales.  The product carries the epilogue itself where the 256x256-tile kernel applies; otherwise it is stored in fp32 into
// `raw` (caller scratch [lenRound][dstDim], may be null only when the fused form applies) and finished by the stand-alone pass.
extern "C" int ts2_matmul_forward_norm_rope(int32_t mode, int32_t len, int32_t lenRound, int32_t srcDim, int32_t dstDim, const ts2_mat *src,
    const ts2_mat *transformFast, float alpha, const float *alphaPtr, int32_t normalize, float vecScale, const ts2_mat *ropeBuf,
    const ts2_mat *res, const ts2_mat *tileScale, const ts2_mat *raw, void *stream)
{
    if (!src || !transformFast || !res || (normalize && !tileScale)) {
        return TS2_ERR_NULL;
    }
    ts2_gemm_args g = {};
    g.a = *src;
    g.b = *transformFast;
    g.abType = mode;
    g.m = lenRound;
    g.n = dstDim;
    g.k = srcDim;
    g.mLive = len;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.splitK = 1;
    // the large tile from 192 tiles on; below, the kernel for few tiles or, for fp8 beyond one round of its workgroups, the 128x128 tile
    // (4096x1024, K = 512 .. 4096: 12.5, 15.0, 20.7, 32.3 -> 9.6, 9.7, 13.0, 23.9 us).  int8 and bf16: as product + pass -> for few tiles 512
    // workgroups at any K (K = 512 bytes 21.8 -> 12.7, 4096 35.8 -> 33.2), 768 up to K = 1536 bytes (K = 1024 24.7 -> 21.9;
    // K = 2048 29.2 -> 30.0; an int8 attention and feed-forward pair of 1536 x 3072 over 2000 tokens, whole step 835 -> 826)
    const bool large = lenRound % 256 == 0 && dstDim % 256 == 0 && (int64_t)(lenRound / 256) * (dstDim / 256) >= 192;
    const int64_t wgs = (int64_t)(lenRound / 64) * (dstDim / 128);
    const bool few = wgs <= (mode == TS2_E4M3 ? 256 : (int64_t)srcDim * (mode == TS2_BF16 ? 2 : 1) <= 1536 ? 768 : 512) &&
                     Aligned16(res->ptr, res->strideBytes) && (!ropeBuf || Aligned16(ropeBuf->ptr, ropeBuf->strideBytes));
    // the 128x128 tile, whose normalising store rounds like the stand-alone pass (the large ones use the hardware's square root and
    // reciprocal), reads the rotation table in pairs; the pass takes it at any fp32 address and stride
    const bool small = mode == TS2_E4M3 && (!ropeBuf || (((uintptr_t)ropeBuf->ptr | ropeBuf->strideBytes) & 7) == 0);
    // int8: the 256x128 tile
    gemmk::GemmP shape = {};
    shape.m = lenRound;
    shape.n = dstDim;
    shape.kBytes = srcDim;
    const bool tall = mode == TS2_I8 && lenRound % 256 == 0 && gemmk::PreferTall(shape, gemmk::T_I8, gemmk::C_BF16NORM, TS2_EPI_STORE) &&
                      Aligned16(res->ptr, res->strideBytes) && (!ropeBuf || Aligned16(ropeBuf->ptr, ropeBuf->strideBytes));
    // (the scratch of the two-launch sequence is part of the call, whichever kernel runs; an empty batch: the product's live length of 0
    // would mean all rows, the stand-alone pass clears them)
    const bool scratch = raw && raw->ptr && raw->x >= dstDim && raw->y >= lenRound;
    if (large || (len > 0 && scratch && (few || small || tall))) {
        g.c = *res;
        g.cType = TS2_BF16;
        g.epilogue = TS2_EPI_ROW_TILE_NORM;
        g.normalize = normalize;
        g.vecScale = vecScale;
        if (ropeBuf) {
            g.rope = *ropeBuf;
        }
        if (normalize) {
            g.tileScale = *tileScale;
        }
        g.tileConfig = large || few || tall ? 0 : 2;
        const int rc = ts2_gemm_nt(&g, stream);
        // rows off 16 bytes and the like: a product and the stand-alone pass take them
        if (large || (rc != TS2_ERR_UNSUPPORTED && rc != TS2_ERR_ALIGN)) {
            return rc;
        }
        g.epilogue = TS2_EPI_STORE;
        g.tileConfig = 0;
        g.normalize = 0;
        g.vecScale = 0;
        g.rope = {};
        g.tileScale = {};
    }
    if (!raw) {
        return TS2_ERR_NULL;
    }
    g.c = *raw;
    g.cType = TS2_F32;
    g.epilogue = TS2_EPI_STORE;
    int rc = ts2_gemm_nt(&g, stream);
    if (rc != TS2_OK) {
        return rc;
    }
    return ts2_row_tile_normalize_rope(len, lenRound, raw, TS2_F32, 1.f, normalize, vecScale, ropeBuf, res, tileScale, stream);
}

// ---------------------------------------------------------------------------------------------------------------------------
// Entry points of the model driver (internal.h)

// Time of a delta product in microseconds.  Both kernels walk their contraction at the rate one CU can fill its LDS from the caches, so a
// launch is (rounds of 256 workgroups) x (start and epilogue + steps): 0.7 us per 256-byte step on 64x128 for the kernel for few tiles, 1.17 us
// per 128-byte step on 256x256 for the ring kernel (2048 x 2048 over 8192 rows: 61 us / 75 us measured, 53 / 81 by this).  Slices add a
// write and a read of fp32 per slice (4 TB/s from the caches) and the packing launch: fitted to a packing kernel that asked for one slice after
// the other (512 x 512 of 8 slices: 7.7 us by this, of which packing took 6.0 and now takes 3.2), so the counts are on the low side.
static double DeltaCost(bool ring, int64_t tiles, int64_t rowBytes, int splits, double outElems)
{
    const double rounds = (double)((tiles * splits + 255) / 256);
    const double steps = ring ? (double)((rowBytes / splits + 127) / 128) : (double)((rowBytes / splits + 255) / 256);
    return rounds * (ring ? 6 + 1.17 * steps : 4 + 0.7 * steps) + (splits > 1 ? 3.5 + splits * outElems * 8 / 4e6 : 0);
}

// the cheapest of the forms of a delta product: kernel and slices; `ringRuns`: the ring kernel takes its operands
static double CheapestDelta(int mode, int lenRound, int srcDim, int gradDim, int64_t partialFloats, bool ringRuns, bool *ring, int *splits)
{
    const int64_t outElems = (int64_t)gradDim * srcDim, sliceTiles = (int64_t)(gradDim / 64) * (srcDim / 128);
    const int64_t rowBytes = (int64_t)lenRound * (mode == TS2_BF16 ? 2 : 1);
    double best = 1e30;
    *ring = false;
    *splits = 1;
    for (int s = 1; s <= 32 && (s == 1 || s * outElems <= partialFloats); s *= 2) {
        if (s > 1 && rowBytes / s < 512) {
            break;
        }
        double c = DeltaCost(false, sliceTiles, rowBytes, s, (double)outElems);
        if (c < best) {
            best = c;
            *ring = false;
            *splits = s;
        }
        c = DeltaCost(true, sliceTiles / 8, rowBytes, s, (double)outElems);
        if (ringRuns && c < best) {
            best = c;
            *ring = true;
            *splits = s;
        }
    }
    return best;
}

double Ts2DeltaCost(int mode, int lenRound, int srcDim, int gradDim, int64_t partialFloats)
{
    bool ring;
    int splits;
    return CheapestDelta(mode, lenRound, srcDim, gradDim, partialFloats, gradDim % 256 == 0 && srcDim % 256 == 0, &ring, &splits);
}

int Ts2DeltaRows(int mode, int len, int lenRound, int srcDim, int gradDim, const ts2_mat *src, const ts2_mat *grad, const float *kTileScale, int kTile,
    int kTileScaleRows, float alpha, const float *alphaPtr, float *partial, int64_t partialFloats, const ts2_mat *delta, const ts2_mat *tileScale,
    void *stream)
{
    const int64_t outElems = (int64_t)gradDim * srcDim;
    if (mode == TS2_I8) {
        // up to four k-tiles per workgroup
        const int splits = (lenRound / kTile + 3) / 4;
        if (splits > 1 && splits * outElems > partialFloats) {
            return TS2_ERR_UNSUPPORTED;
        }
        return DeltaSlice(mode, len, lenRound, srcDim, gradDim, src, grad, kTileScale, kTile, kTileScaleRows, alpha, alphaPtr, splits, partial, delta,
            tileScale, stream);
    }
    bool ring;
    int splits;
    CheapestDelta(mode, lenRound, srcDim, gradDim, partialFloats, (gradDim % 256) == 0 && (srcDim % 256) == 0 && grad->y >= lenRound && src->y >= lenRound,
        &ring, &splits);
    if (!ring) {
        return DeltaSlice(mode, len, lenRound, srcDim, gradDim, src, grad, nullptr, 0, 0, alpha, alphaPtr, splits, partial, delta, tileScale, stream);
    }
    ts2_gemm_args g = {};
    g.a = *grad;
    g.b = *src;
    g.abType = mode;
    g.m = gradDim;
    g.n = srcDim;
    g.k = lenRound;
    g.kMajor = 1;
    g.tileConfig = 1;
    g.splitK = 1;
    if (splits > 1) {
        g.c = {partial, (int64_t)srcDim * 4, srcDim, gradDim};
        g.cType = TS2_F32;
        g.alpha = 1.f;
        g.epilogue = TS2_EPI_STORE;
        g.splitK = splits;
        g.splitSlabBytes = outElems * 4;
        int rc = ts2_gemm_nt(&g, stream);
        if (rc) {
            return rc;
        }
        ts2_mat part = {partial, (int64_t)srcDim * 4, srcDim, splits * gradDim};
        return ts2_pack_delta(&part, splits, g.splitSlabBytes, gradDim, srcDim, alpha, alphaPtr, delta, tileScale, stream);
    }
    g.c = *delta;
    g.cType = TS2_I8;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.epilogue = TS2_EPI_ROW_TILE_MAXNORM;
    g.tileScale = *tileScale;
    return ts2_gemm_nt(&g, stream);
}

int Ts2GroupedDeltaRows(int rows, int srcDim, int gradDim, int groups, const int *groupOffsets, const ts2_mat *src, const ts2_mat *grad, float alpha,
    const float *alphaPtr, const ts2_mat *delta, int64_t deltaSlabBytes, const ts2_mat *tileScale, int64_t tileScaleSlabBytes, void *stream)
{
    gemmk::SliceP sp = {};
    gemmk::GemmP &g = sp.g;
    g.a = (const uint8_t *)grad->ptr;
    g.b = (const uint8_t *)src->ptr;
    g.c = (uint8_t *)delta->ptr;
    g.lda = grad->strideBytes;
    g.ldb = src->strideBytes;
    g.ldc = delta->strideBytes;
    g.m = gradDim;
    g.n = srcDim;
    g.kBytes = rows;
    sp.kLive = rows;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr;
    g.tileScale = (float *)tileScale->ptr;
    g.ldTileScale = tileScale->strideBytes / 4;
    g.nSeg = 1;
    g.splits = 1;
    g.groupOffsets = groupOffsets;
    g.splitK_groups = groups;
    g.cSlab = deltaSlabBytes;
    g.tileScaleSlab = tileScaleSlabBytes / 4;
    sp.ct = gemmk::C_I8PACK;
    sp.epi = TS2_EPI_STORE;
    return gemmk::RunSlice(sp, gemmk::T_FP8, true, (hipStream_t)stream);
}

int Ts2BackpropGroupI8(int count, int len, int lenRound, int srcDim, int gradDim, const ts2_mat *grad8, const float *const *rowScale,
    const ts2_mat *transformT, const float *alpha, const float *const *alphaPtr, const ts2_mat *srcGrad, int srcGradType, int add, void *stream)
{
    if (count < 1 || count > 4) {
        return TS2_ERR_SHAPE;
    }
    // one launch: the kernel for few tiles, the 256x128 one (PreferTall), or, for rows off its grid, up to the size where 256x256 tiles fill the chip
    // the 128x128 one (16384 x 512 x 512 inside the e512 step: a sum of four and a sum of two products 111 us together as six launches, 72 as two)
    const bool few = (int64_t)(lenRound / 64) * (srcDim / 128) <= 640;
    const bool tall = srcGradType == TS2_F32 && !add;
    const bool sum = tall && (int64_t)lenRound * srcDim < (int64_t)192 * 65536;
    bool one = count > 1 && (srcGradType == TS2_F32 || srcGradType == TS2_BF16) && (few || tall);
    for (int i = 1; i < count && one; ++i) {
        one = grad8[i].strideBytes == grad8[0].strideBytes && transformT[i].strideBytes == transformT[0].strideBytes;
    }
    if (one) {
        gemmk::SliceP sp = {};
        gemmk::GemmP &g = sp.g;
        g.a = (const uint8_t *)grad8[0].ptr;
        g.b = (const uint8_t *)transformT[0].ptr;
        g.c = (uint8_t *)srcGrad->ptr;
        g.lda = grad8[0].strideBytes;
        g.ldb = transformT[0].strideBytes;
        g.ldc = srcGrad->strideBytes;
        g.m = lenRound;
        g.n = srcDim;
        g.kBytes = gradDim;
        g.mLive = len;
        g.rowScale = rowScale[0];
        g.alpha = alpha[0];
        g.alphaPtr = alphaPtr[0];
        g.splits = 1;
        g.nSeg = count;
        for (int i = 1; i < count; ++i) {
            g.segA[i - 1] = (const uint8_t *)grad8[i].ptr;
            g.segB[i - 1] = (const uint8_t *)transformT[i].ptr;
            g.segAlpha[i - 1] = alpha[i];
            g.segAlphaPtr[i - 1] = alphaPtr[i];
            g.segRowScale[i - 1] = rowScale[i];
        }
        sp.ct = srcGradType == TS2_F32 ? gemmk::C_F32 : gemmk::C_BF16;
        sp.epi = add ? TS2_EPI_ADD : TS2_EPI_STORE;
        if (tall && gemmk::PreferTall(g, gemmk::T_I8, gemmk::C_F32, TS2_EPI_STORE) && gemmk::TallCanRun(g, gemmk::T_I8, gemmk::C_F32, TS2_EPI_STORE)) {
            return gemmk::RunTall(g, gemmk::T_I8, gemmk::C_F32, TS2_EPI_STORE, (hipStream_t)stream);
        }
        if (few && gemmk::SliceCanRun(sp, gemmk::T_I8, false)) {
            return gemmk::RunSlice(sp, gemmk::T_I8, false, (hipStream_t)stream);
        }
        const int rc = sum ? gemmk::RunSumI8(g, (hipStream_t)stream) : TS2_ERR_UNSUPPORTED;
        if (rc != TS2_ERR_UNSUPPORTED) {
            return rc;
        }
    }
    for (int i = 0; i < count; ++i) {
        ts2_gemm_args g = {};
        g.a = grad8[i];
        g.b = transformT[i];
        g.c = *srcGrad;
        g.abType = TS2_I8;
        g.cType = srcGradType;
        g.m = lenRound;
        g.n = srcDim;
        g.k = gradDim;
        g.mLive = len;
        g.rowScale = rowScale[i];
        g.alpha = alpha[i];
        g.alphaPtr = alphaPtr[i];
        g.epilogue = (add || i > 0) ? TS2_EPI_ADD : TS2_EPI_STORE;
        g.splitK = 1;
        int rc = ts2_gemm_nt(&g, stream);
        if (rc) {
            return rc;
        }
    }
    return TS2_OK;
}

// While one product alone fits the chip (256 workgroups, one per CU), a launch is a chain of latencies and four of them cost four.  Whole passes,
// separate -> one launch: 512-token int8 step 1133 -> 1016 us, 777-token prompt 1007 -> 874, 3885-token
// 8-expert step 1632 -> 1538.  Where all of them are more than a round of the kernel for few tiles, PreferJobs (gemm.hip) decides
int Ts2ForwardGroup(int mode, int count, int len, int lenRound, int srcDim, int dstDim, const ts2_mat *src, const ts2_mat *const *w, float alpha,
    const float *const *alphaPtr, int normalizeBits, float vecScale, int rotateBits, const ts2_mat *rope, const ts2_mat *res,
    const ts2_mat *const *tileScale, void *stream)
{
    const int64_t wgs = (int64_t)(lenRound / 64) * (dstDim / 128);
    if (count < 2 || count > 4 || !Is8(mode) || lenRound % 128 || dstDim % 128 || srcDim % 128 || src->x < srcDim || src->y < lenRound) {
        return TS2_ERR_UNSUPPORTED;
    }
    gemmk::SliceP sp = {};
    gemmk::GemmP &g = sp.g;
    g.a = (const uint8_t *)src->ptr;
    g.b = (const uint8_t *)w[0]->ptr;
    g.c = (uint8_t *)res[0].ptr;
    g.lda = src->strideBytes;
    g.ldb = w[0]->strideBytes;
    g.ldc = res[0].strideBytes;
    g.m = lenRound;
    g.n = dstDim;
    g.kBytes = srcDim;
    g.mLive = len;
    g.alpha = alpha;
    g.alphaPtr = alphaPtr[0];
    g.vecScale = vecScale;
    g.splits = 1;
    g.nSeg = 1;
    if (rotateBits) {
        g.rope = (const float *)rope->ptr;
        g.ldRope = rope->strideBytes / 4;
    }
    sp.ct = gemmk::C_BF16NORM;
    sp.epi = TS2_EPI_STORE;
    g.jobs = count;
    g.jobNormalize = normalizeBits;
    g.jobRope = rotateBits;
    for (int i = 0; i < count; ++i) {
        if (w[i]->strideBytes != g.ldb || res[i].strideBytes != g.ldc || w[i]->x < srcDim || w[i]->y < dstDim || res[i].x < dstDim || res[i].y < lenRound) {
            return TS2_ERR_UNSUPPORTED;
        }
        g.jobB[i] = (const uint8_t *)w[i]->ptr;
        g.jobC[i] = (uint8_t *)res[i].ptr;
        g.jobAlphaPtr[i] = alphaPtr[i];
        if ((normalizeBits >> i) & 1) {
            const int64_t ld = tileScale[i]->strideBytes / 4;
            if (tileScale[i]->x < lenRound || tileScale[i]->y < dstDim / TILE || (g.ldTileScale && g.ldTileScale != ld)) {
                return TS2_ERR_UNSUPPORTED;
            }
            g.ldTileScale = ld;
            g.jobTileScale[i] = (float *)tileScale[i]->ptr;
        }
    }
    const int type = SliceType(mode);
    if (gemmk::PreferJobs(g, type)) {
        const int rc = gemmk::RunJobs(g, type, (hipStream_t)stream);
        if (rc != TS2_ERR_UNSUPPORTED) {
            return rc;
        }
    }
    return wgs <= 256 ? gemmk::RunSlice(sp, type, false, (hipStream_t)stream) : TS2_ERR_UNSUPPORTED;
}
