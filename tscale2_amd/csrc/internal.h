// Library-internal entry points (not part of the C ABI): kernels used only by the model driver.
#pragma once
#include "../../include/ts2_abi.h"

int Ts2EmbedForward(int len, int lenRound, int dim, const int *labelPtr, const uint32_t *labels, const ts2_mat *embed, int embType, float mult,
    const float *scalePtr, const ts2_mat *state, void *stream);
// mark: scratch of labelCount ints, or null
int Ts2EmbedBackward(int len, int dim, const int *labelPtr, const uint32_t *labels, const ts2_mat *grad, const ts2_mat *delta, int labelCount,
    int *mark, void *stream);
int Ts2FinalProbabilities(int rows, int vocab, const ts2_mat *logits, const float *bias, const int *target, float gradMult, const ts2_mat *grad,
    void *stream);
int Ts2FinalSoftmaxGradHalf(int rows, int vocab, const ts2_mat *logits, const float *bias, const int *target, float gradMult, const ts2_mat *grad,
    float *lossSum, void *stream);
int Ts2TransposeToBf16(int rows, int rowsRound, int cols, const ts2_mat *src, int srcType, const ts2_mat *dst, void *stream);
int Ts2RowsToBf16(int rows, int rowsRound, int cols, const ts2_mat *src, int srcType, const ts2_mat *dst, void *stream);
int Ts2ZeroRows(const ts2_mat *m, int rows, int rowBytes, void *stream);
int Ts2FillFloats(float *p, int n, float v, void *stream);
// ts2_transpose_quant with the k-tile maxima formed in the kernel from row maxima (rowAbsMax) when tileMax is null
int Ts2TransposeQuantRows(int len, int lenRound, const ts2_mat *src, int srcType, const float *rowMult, const float *tileMax, const float *rowAbsMax,
    int kTile, const int *rowIndex, const ts2_mat *dstT, int dstType, float *tileScale, void *stream, uint32_t ditherSeed = 0);
// resolves, for the current device, what ts2_moe_route_static otherwise resolves on its first call there (no stream operation)
int Ts2MoeRouteSetup();
// the int8 row quantiser (ts2_normalize_vecs_row_max_dither) over `count` <= 4 bf16 gradients of one width <= 4096, one launch
int Ts2QuantRowsBatch(int count, int len, int lenRound, const ts2_mat *src, const ts2_mat *dst, float *const *rowScale, float *const *rowAbsMax,
    const uint32_t *seed, void *stream);
// where a gradient pass leaves the rows it writes quantised as well (the row quantiser's results); seed 0: no dither
struct RowQuantOut {
    uint8_t *dst;
    int64_t dstStride; // bytes
    float *rowScale, *rowAbsMax;
    uint32_t seed;
};
// int8 forms, bf16 gradients, rows of up to 4096: ts2_backprop_row_tile_normalize_lolu (mode 0) / ts2_backprop_lolu_dscale (mode 1, quantises the
// gate's gradient), ts2_backprop_row_tile_normalize_rope of up to three gradients, ts2_backprop_layer_normalize / ts2_backprop_final_normalize
// (rows of up to 1536).  TS2_ERR_UNSUPPORTED: nothing was launched
int Ts2BackpropLoluRows(int mode, int len, int lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale, const ts2_mat *valsSrcTileScale,
    const ts2_mat *grad, const ts2_mat *gradGate, const ts2_mat *gradVals, const ts2_mat *dScale, const RowQuantOut &qGate, const RowQuantOut &qVals,
    void *stream);
int Ts2BackpropNormRopeRows(int count, int len, int lenRound, const ts2_mat *const *grad, float gradMult, const ts2_mat *const *srcNorm,
    const ts2_mat *const *srcTileScale, const ts2_mat *const *ropeBuf, const ts2_mat *const *dst, const RowQuantOut *q, void *stream);
int Ts2BackpropLayerNormalizeRows(bool final, int len, int lenRound, const ts2_mat *normState, const ts2_mat *stateScale, const ts2_mat *dNormState,
    const float *gradScale, const float *gradMult, const ts2_mat *stateGrad, const ts2_mat *stateGradFast, float *nextMaxNorm, const RowQuantOut &q,
    void *stream);
// ts2_scale_grad (bf16) that moves the rows' codes, scales and maxima (q) along with the values when their power of two changes; the second
// form leaves the codes, for rows whose maxima lie within 2^-100 .. 2^100 before and after
int Ts2ScaleGradRows(const float *gradMaxNorm, const float *prevGradMult, const ts2_mat *grad, const ts2_mat *gradFast, int len, float *gradScaleOut,
    float *gradMultOut, const RowQuantOut &q, void *stream);
int Ts2ScaleGradRows(const float *gradMaxNorm, const float *prevGradMult, const ts2_mat *grad, const ts2_mat *gradFast, int len, float *gradScaleOut,
    float *gradMultOut, float *rowScale, float *rowAbsMax, void *stream);
// the k-tile quantiser without the transpose, over `count` <= 4 bf16 gradients of one width: dst[t][x] with one scale per kTile rows,
// tileScale [count][lenRound / kTile]
int Ts2QuantTileRows(int count, int len, int lenRound, int kTile, const ts2_mat *src, const ts2_mat *dst, const float *const *rowAbsMax,
    const uint32_t *seed, const float *rowMult, float *tileScale, void *stream);
// ... over any number of gradients with the same rows, each with a width and a place of its own
struct TileQuantJob {
    const uint8_t *src;
    uint8_t *dst;
    int64_t srcStride, dstStride; // bytes
    const float *rowAbsMax;
    float *tileScale; // [lenRound / kTile]
    int dim;
    uint32_t seed;
};
int Ts2QuantTileRowsJobs(int count, int len, int lenRound, int kTile, const TileQuantJob *jobs, const float *rowMult, void *stream);
// packed delta [gradDim][srcDim] = alpha * *alphaPtr * sum over the rows of grad^T src, both operands row-major as they lie (rows len ..
// lenRound of both hold zeros); mode TS2_I8 (with kTileScale [gradDim / kTileScaleRows][lenRound / kTile]; kTileScaleRows 0 = one set),
// TS2_E4M3 or TS2_BF16.  Chooses kernel and token slices by cost; partial: fp32 scratch for the slices.  TS2_ERR_UNSUPPORTED: no kernel for it
int Ts2DeltaRows(int mode, int len, int lenRound, int srcDim, int gradDim, const ts2_mat *src, const ts2_mat *grad, const float *kTileScale, int kTile,
    int kTileScaleRows, float alpha, const float *alphaPtr, float *partial, int64_t partialFloats, const ts2_mat *delta, const ts2_mat *tileScale,
    void *stream);
// estimated microseconds of that (TS2_E4M3 or TS2_BF16)
double Ts2DeltaCost(int mode, int lenRound, int srcDim, int gradDim, int64_t partialFloats);
// how many deltas of the model's last backward pass waited for its end (a layer's stacked matrices count as one)
int Ts2ModelWaitingDeltas(const ts2_model *M);
// int8: srcGrad (+)= sum_i alpha_i * *alphaPtr_i * rowScale_i[t] * (grad8_i W_i^T), count <= 4 products of one shape added in order
int Ts2BackpropGroupI8(int count, int len, int lenRound, int srcDim, int gradDim, const ts2_mat *grad8, const float *const *rowScale,
    const ts2_mat *transformT, const float *alpha, const float *const *alphaPtr, const ts2_mat *srcGrad, int srcGradType, int add, void *stream);
// forward products of up to four matrices of one shape that read the same source, in one launch: res_i = rope(normalise(alpha *
// *alphaPtr_i * src * W_i^T)) as bf16, normalisation and rotation each where asked for.  TS2_ERR_UNSUPPORTED: not possible, or not worth it;
// nothing was launched then
int Ts2ForwardGroup(int mode, int count, int len, int lenRound, int srcDim, int dstDim, const ts2_mat *src, const ts2_mat *const *w, float alpha,
    const float *const *alphaPtr, int normalizeBits, float vecScale, int rotateBits, const ts2_mat *rope, const ts2_mat *res,
    const ts2_mat *const *tileScale, void *stream);
// ts2_opt_add_delta(.., TS2_BM_GRAD_APPLY) of several matrices in two or three launches (per 16 of them).  Ts2OptBatchable: one dispersion
// estimate per row, rows of at most 4096 elements
bool Ts2OptBatchable(const ts2_opt_matrix *m);
int Ts2OptApplyBatch(int count, const ts2_opt_matrix *const *mats, const ts2_mat *const *delta, const ts2_mat *const *tileScale,
    const ts2_add_gradient_params *params, void *stream);
// ts2_backprop_row_tile_normalize_rope of up to four gradients of one width in one launch
int Ts2BackpropNormRopeGroup(int count, int len, int lenRound, const ts2_mat *const *grad, int gradType, float gradMult, const ts2_mat *const *srcNorm,
    const ts2_mat *const *srcTileScale, const ts2_mat *const *ropeBuf, const ts2_mat *const *dst, int dstType, void *stream);
// dst_i [cols][rows] = src_i [rows][cols]^T for byte matrices whose dimensions are multiples of 128, 32 to a launch
int Ts2TransposeBytesBatch(int count, const ts2_mat *const *src, const ts2_mat *const *dst, const int *rows, const int *cols, void *stream);
// per-group deltas (TMoeDeltaMatMulKernelCall) by the kernel for few tiles: groups * gradDim rows of packed delta
int Ts2GroupedDeltaRows(int rows, int srcDim, int gradDim, int groups, const int *groupOffsets, const ts2_mat *src, const ts2_mat *grad, float alpha,
    const float *alphaPtr, const ts2_mat *delta, int64_t deltaSlabBytes, const ts2_mat *tileScale, int64_t tileScaleSlabBytes, void *stream);
