// Bandwidth-bound fused gradient kernels (tile norm forward/backward + residual add, dynamic gradient scaling, gated sigmoid
// forward/backward, per-row and per-k-tile int8 quantisation, 8-bit transposes).
//
// Mapping for gfx950: one 128-wide tile is held by 32 lanes x 4 elements, so a 64-wide wavefront processes two tiles per
// instruction with 16-byte (fp32), 8-byte (bf16) or 4-byte (8-bit) accesses per lane; reductions stay inside the 32-lane group
// (5 cross-lane steps).  Workgroups are 256 threads (8 tiles in flight) and grids cover every (row, tile) once, so each launch puts
// thousands of workgroups on the 256 CUs; consecutive 32-lane groups walk consecutive tiles of a row, i.e. HBM accesses are fully
// coalesced 512-byte (fp32) runs.  The reference launches one 32-thread block per (tile, row) (src/lib/cuda/cuda_graph.cuh:359-365).
#include "vec.h"
#include "internal.h"
#include <algorithm>

namespace
{
struct Mat {
    uint8_t *p;
    int64_t ld;
};

__host__ __device__ __forceinline__ Mat M(const ts2_mat &m)
{
    Mat r = {(uint8_t *)m.ptr, m.strideBytes};
    return r;
}

template <class TT> __device__ __forceinline__ void *At(const Mat &m, int row, int col)
{
    return m.p + (int64_t)row * m.ld + (int64_t)col * TT::SIZE;
}

__device__ __forceinline__ float &ScaleAt(const Mat &m, int tile, int row)
{
    return *(float *)(m.p + (int64_t)tile * m.ld + (int64_t)row * 4);
}

// Every 32-lane group owns U consecutive rows of one tile column and issues the loads of all U rows before it touches any of them:
// with one row per group a wave has a single 4-16 byte load per lane in flight and the kernels sit at 30-50 % of what a copy reaches.
constexpr int U = 4;

// first row and tile of this 32-lane group; returns false when the whole group is out of range
__device__ __forceinline__ bool Unit(int rows, int tiles, int *row0, int *tile, int *lane32)
{
    long u = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 5;
    *lane32 = threadIdx.x & 31;
    long rb = u / tiles;
    *tile = (int)(u - rb * tiles);
    *row0 = (int)(rb * U);
    return *row0 < rows;
}

inline dim3 GridFor(int rows, int tiles)
{
    long units = (long)((rows + U - 1) / U) * tiles;
    return dim3((unsigned)((units * 32 + 255) / 256));
}

// non-negative float max through the integer ordering, like the reference's atomicMax((int*)p, __float_as_int(x))
// Nothing waits for it.  (Looking first whether the value there is lower already saves most of the updates, 10 ns each on one address, but the
// answer takes microseconds while the address is contended and holds the workgroup's place that long: maxima of the k-tiles of 16384 x 4096
// 76.3 us with the look, 30.5 without, normalisation backward of 16384 x 1024 e4m3 48.3 / 44.2, of 32768 x 2048 185.4 / 177.8.)
__device__ __forceinline__ void AtomicMaxPos(float *p, float v)
{
    atomicMax((int *)p, __float_as_int(v));
}

// lanes 0..U-1 of the group store the U per-row scalars of one tile column (16 contiguous bytes)
__device__ __forceinline__ void StoreScales(const Mat &m, int tile, int row0, int rows, int h, const float (&v)[U])
{
    float mine = 0;
#pragma unroll
    for (int k = 0; k < U; ++k) {
        mine = h == k ? v[k] : mine;
    }
    if (h < U && row0 + h < rows) {
        ScaleAt(m, tile, row0 + h) = mine;
    }
}

// --------------------------------------------------------------------------------------------------------------------------
template <class TSrc, class TDst>
__global__ void __launch_bounds__(256) LayerNormalizeStateVecs(int len, int lenRound, int tiles, float vecScale, Mat state, Mat normState, Mat normScale)
{
    int t0, tile, h;
    if (!Unit(lenRound, tiles, &t0, &tile, &h)) {
        return;
    }
    int col = tile * TILE + h * 4;
    F4 v[U];
    float discr[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        v[k] = t0 + k < len ? Load4<TSrc>(At<TSrc>(state, t0 + k, col)) : ZeroF4();
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        discr[k] = 0;
        float sum2 = Half32Sum(HSum(v[k] * v[k]));
        if (sum2 > 0) {
            discr[k] = sqrtf(sum2 / TILE) * vecScale;
            v[k] = v[k] * (1 / discr[k]);
        }
        if (t0 + k < lenRound) {
            Store4<TDst>(At<TDst>(normState, t0 + k, col), v[k]);
        }
    }
    StoreScales(normScale, tile, t0, lenRound, h, discr);
}

// the maximum over a workgroup of NT threads to *p
template <int NT> __device__ __forceinline__ void PublishBlockMax(float v, float *red, float *p)
{
    v = WaveMax(v);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0 && p) {
        float m = red[0];
#pragma unroll
        for (int w = 1; w < NT / 64; ++w) {
            m = fmaxf(m, red[w]);
        }
        AtomicMaxPos(p, m);
    }
}

// Every workgroup walks many units and issues ONE atomic max at the end: one atomic per unit (the reference's scheme,
// gpu_layer_norm.cuh:111-114) serialises half a million updates of a single address at this problem size.
template <class TNorm, class TFast, bool FINAL, int NT>
__global__ void __launch_bounds__(NT) BackpropLayerNormalize(int len, int rows, int tiles, Mat normState, Mat stateScale, Mat dNormState,
    const float *combinerScale, const float *gradScale, const float *gradMult, Mat stateGrad, Mat stateGradFast, float *nextMaxNorm)
{
    __shared__ float red[NT / 64];
    const int h = threadIdx.x & 31;
    const long units = (long)((rows + U - 1) / U) * tiles;
    float s = 1;
    if (!FINAL) {
        if (combinerScale) {
            s *= *combinerScale;
        }
        if (gradScale) {
            s *= *gradScale;
        }
    }
    const float gm = (!FINAL && gradMult) ? *gradMult : 1.f;
    float gmax = 0;
    for (long u = ((long)blockIdx.x * NT + threadIdx.x) >> 5; u < units; u += (long)gridDim.x * (NT / 32)) {
        long rb = u / tiles;
        int tile = (int)(u - rb * tiles);
        int t0 = (int)rb * U;
        int col = tile * TILE + h * 4;
        F4 vec[U], grad[U], prev[U];
        float sc[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            int t = t0 + k;
            bool live = t < len;
            vec[k] = live ? Load4<TNorm>(At<TNorm>(normState, t, col)) : ZeroF4();
            grad[k] = live ? Load4<TF32>(At<TF32>(dNormState, t, col)) : ZeroF4();
            prev[k] = (live && !FINAL) ? Load4<TF32>(At<TF32>(stateGrad, t, col)) : ZeroF4();
            sc[k] = live ? ScaleAt(stateScale, tile, t) : 0.f;
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            int t = t0 + k;
            if (t >= rows) {
                continue;
            }
            F4 g = ZeroF4();
            if (t < len) {
                g = FINAL ? grad[k] : grad[k] * s;
                g = TileNormBackprop(vec[k] * sc[k], g);
                if (!FINAL) {
                    g = g + prev[k];
                }
                gmax = fmaxf(gmax, HMaxAbs(g));
            }
            Store4<TF32>(At<TF32>(stateGrad, t, col), g);
            Store4<TFast>(At<TFast>(stateGradFast, t, col), g * gm);
        }
    }
    PublishBlockMax<NT>(gmax, red, nextMaxNorm);
}

// e4m3 norm state and e4m3 fast gradient with eight elements per lane (a tile = 16 lanes, 16-byte accesses to the fp32 arrays): the
// form the fp8 model runs.  Same arithmetic per element as BackpropLayerNormalize; Row16Sum is defined with the 8-wide LoLU kernel.
__device__ __forceinline__ float Row16SumFwd(float v);

template <bool FINAL, int NT>
__global__ void __launch_bounds__(NT) BackpropLayerNormalize8(int len, int rows, int tiles, Mat normState, Mat stateScale, Mat dNormState,
    const float *combinerScale, const float *gradScale, const float *gradMult, Mat stateGrad, Mat stateGradFast, float *nextMaxNorm)
{
    __shared__ float red[NT / 64];
    const int l16 = threadIdx.x & 15;
    const long units = (long)rows * tiles;
    float s = 1;
    if (!FINAL) {
        if (combinerScale) {
            s *= *combinerScale;
        }
        if (gradScale) {
            s *= *gradScale;
        }
    }
    const float gm = (!FINAL && gradMult) ? *gradMult : 1.f;
    float gmax = 0;
    // every lane of a wave takes part in every iteration (the reductions are cross-lane): the loop bound is wave-uniform
    const long unitFirst = ((long)blockIdx.x * NT + (threadIdx.x & ~63)) >> 4;
    for (long ub = unitFirst; ub < units; ub += (long)gridDim.x * (NT / 16)) {
        const long u = ub + ((threadIdx.x & 63) >> 4);
        const bool any = u < units;
        const int t = any ? (int)(u / tiles) : 0;
        const int tile = any ? (int)(u - (long)t * tiles) : 0;
        const int col = tile * TILE + l16 * 8;
        const bool live = any && t < len;
        uint2 nv = live ? *(const uint2 *)At<TE4M3>(normState, t, col) : make_uint2(0, 0);
        F4 g0 = live ? Load4<TF32>(At<TF32>(dNormState, t, col)) : ZeroF4();
        F4 g1 = live ? Load4<TF32>(At<TF32>(dNormState, t, col + 4)) : ZeroF4();
        F4 p0 = (live && !FINAL) ? Load4<TF32>(At<TF32>(stateGrad, t, col)) : ZeroF4();
        F4 p1 = (live && !FINAL) ? Load4<TF32>(At<TF32>(stateGrad, t, col + 4)) : ZeroF4();
        const float sc = live ? ScaleAt(stateScale, tile, t) : 0.f;
        float src[8], g[8];
        const float nf[8] = {__builtin_amdgcn_cvt_f32_fp8((int)nv.x, 0), __builtin_amdgcn_cvt_f32_fp8((int)nv.x, 1), __builtin_amdgcn_cvt_f32_fp8((int)nv.x, 2),
            __builtin_amdgcn_cvt_f32_fp8((int)nv.x, 3), __builtin_amdgcn_cvt_f32_fp8((int)nv.y, 0), __builtin_amdgcn_cvt_f32_fp8((int)nv.y, 1),
            __builtin_amdgcn_cvt_f32_fp8((int)nv.y, 2), __builtin_amdgcn_cvt_f32_fp8((int)nv.y, 3)};
        const float gin[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        const float prev[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
        float sum2 = 0, dp = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            src[e] = nf[e] * sc;
            g[e] = FINAL ? gin[e] : gin[e] * s;
            sum2 += src[e] * src[e];
            dp += src[e] * g[e];
        }
        sum2 = Row16SumFwd(sum2);
        dp = Row16SumFwd(dp);
        if (!any) {
            continue;
        }
        float sigma = 0, scale = 0;
        if (sum2 != 0) {
            float inv = 1 / sum2;
            sigma = dp * inv;
            scale = sqrtf(TILE * inv);
        }
        float out[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float x = 0;
            if (live) {
                x = sum2 != 0 ? (g[e] - src[e] * sigma) * scale : 0.f;
                if (!FINAL) {
                    x += prev[e];
                }
                gmax = fmaxf(gmax, fabsf(x));
            }
            out[e] = x;
        }
        Store4<TF32>(At<TF32>(stateGrad, t, col), MakeF4(out[0], out[1], out[2], out[3]));
        Store4<TF32>(At<TF32>(stateGrad, t, col + 4), MakeF4(out[4], out[5], out[6], out[7]));
        uint32_t lo = CvtPkE4m3(out[0] * gm, out[1] * gm) | (CvtPkE4m3(out[2] * gm, out[3] * gm) << 16);
        uint32_t hi = CvtPkE4m3(out[4] * gm, out[5] * gm) | (CvtPkE4m3(out[6] * gm, out[7] * gm) << 16);
        *(uint2 *)At<TE4M3>(stateGradFast, t, col) = make_uint2(lo, hi);
    }
    PublishBlockMax<NT>(gmax, red, nextMaxNorm);
}

__device__ __forceinline__ float ComputeGradMult(float gradMaxNorm)
{
    if (gradMaxNorm == 0) {
        return 1;
    }
    return __uint_as_float(__float_as_uint(128.f / gradMaxNorm) & 0xff800000u);
}

// 32 lanes move the codes of rows t0 .. t0 + U to another power of two of the gradients.  The codes stay and scale and maximum move along, exactly,
// while bf16 holds the row at both powers: rows whose maximum leaves 2^-100 .. 2^100 (bf16 rounds their smaller elements to fewer bits, and from 2^-121
// on the reciprocal of the scale overflows) or that bf16 has rounded to zero (scale 1) are quantised again from the fp32 gradients.
__device__ __forceinline__ void MoveRowCodes(int t0, int len, int dim, const Mat &grad, float gradMult, float ratio, int h, const RowQuantOut &q)
{
    auto held = [](float x) { return x >= 0x1p-100f && x <= 0x1p100f; };
    bool again = false;
    if (h < U && t0 + h < len) {
        const float top = q.rowAbsMax[t0 + h], scale = q.rowScale[t0 + h];
        again = q.dst && (top == 0 ? scale != 0 : !held(top) || !held(top * ratio));
        if (!again) {
            q.rowScale[t0 + h] = scale * ratio;
            q.rowAbsMax[t0 + h] = top * ratio;
        }
    }
    const unsigned rows = (unsigned)(__ballot(again) >> (threadIdx.x & 32)); // (of these 32 lanes: the others may be elsewhere)
    for (int k = 0; k < U; ++k) {
        if (!((rows >> k) & 1)) {
            continue;
        }
        const int t = t0 + k;
        auto load = [&](int col) {
            const F4 v = Load4<TF32>(At<TF32>(grad, t, col)) * gradMult;
            const uint32_t lo = PackBf16x2(v.x, v.y), hi = PackBf16x2(v.z, v.w);
            return MakeF4(__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u), __uint_as_float(hi << 16), __uint_as_float(hi & 0xffff0000u));
        };
        float mx = 0;
        for (int col = h * 4; col < dim; col += 128) {
            mx = fmaxf(mx, HMaxAbs(load(col)));
        }
        for (int d = 16; d > 0; d >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, d));
        }
        const float discr = mx > 0 ? mx / 127 : 0.f, mult = mx > 0 ? 1 / discr : 0.f;
        for (int col = h * 4; col < dim; col += 128) {
            const F4 v = load(col);
            uint8_t *const dst = q.dst + (int64_t)t * q.dstStride + col;
            if (q.seed) {
                *(uint32_t *)dst = QuantDither4(v.x, v.y, v.z, v.w, mult, DitherWord(q.seed, t, col >> 2));
            } else {
                Store4<TI8>(dst, v * mult);
            }
        }
        if (h == 0) {
            q.rowScale[t] = discr;
            q.rowAbsMax[t] = mx;
        }
    }
}

// ROWS: the rows are quantised already (q)
template <class TFast, bool ROWS>
__global__ void __launch_bounds__(256) ScaleGrad(int len, int tiles, const float *gradMaxNorm, const float *prevGradMult, Mat grad, Mat gradFast,
    float *gradScaleOut, float *gradMultOut, RowQuantOut q)
{
    int t0, tile, h;
    float gradMult = ComputeGradMult(*gradMaxNorm);
    bool rewrite = !prevGradMult || gradMult != *prevGradMult;
    if (blockIdx.x == 0 && threadIdx.x == 0) { // (null when a later launch has to publish, see ts2_scale_grad)
        if (gradScaleOut) {
            *gradScaleOut = 1 / gradMult;
        }
        if (gradMultOut) {
            *gradMultOut = gradMult;
        }
    }
    if (Unit(len, tiles, &t0, &tile, &h) && rewrite) {
        int col = tile * TILE + h * 4;
        F4 v[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            v[k] = t0 + k < len ? Load4<TF32>(At<TF32>(grad, t0 + k, col)) : ZeroF4();
        }
#pragma unroll
        for (int k = 0; k < U; ++k) {
            if (t0 + k < len) {
                Store4<TFast>(At<TFast>(gradFast, t0 + k, col), v[k] * gradMult);
            }
        }
        // the rows' codes (int8) belong to values times the old power of two
        if (ROWS && tile == 0) {
            MoveRowCodes(t0, len, tiles * TILE, grad, gradMult, gradMult / *prevGradMult, h, q);
        }
    }
}

// for callers that pass a cell the rewrite kernel reads (prevGradMult, gradMaxNorm) as an output: published after that kernel
__global__ void PublishGradMult(const float *gradMaxNorm, float *gradScaleOut, float *gradMultOut)
{
    float gradMult = ComputeGradMult(*gradMaxNorm);
    if (gradScaleOut) {
        *gradScaleOut = 1 / gradMult;
    }
    if (gradMultOut) {
        *gradMultOut = gradMult;
    }
}

template <class TDst>
__global__ void __launch_bounds__(256) MatrixLoLU(int len, int lenRound, int tiles, Mat gate, Mat vals, float resMult, Mat res)
{
    int t0, tile, h;
    if (!Unit(lenRound, tiles, &t0, &tile, &h)) {
        return;
    }
    int col = tile * TILE + h * 4;
    F4 g[U], v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        bool live = t0 + k < len;
        g[k] = live ? Load4<TBF16>(At<TBF16>(gate, t0 + k, col)) : ZeroF4();
        v[k] = live ? Load4<TBF16>(At<TBF16>(vals, t0 + k, col)) : ZeroF4();
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        if (t0 + k < lenRound) {
            Store4<TDst>(At<TDst>(res, t0 + k, col), t0 + k < len ? v[k] * LoLU4(g[k]) * resMult : ZeroF4());
        }
    }
}

// The e4m3 result from bf16 inputs with eight elements per lane (16-byte loads, 8-byte stores; no reduction in this kernel, so the
// tile structure does not matter): the form the model's FFN and attention forward use.  Two row segments per lane in flight.
__global__ void __launch_bounds__(256) MatrixLoLU8(int len, int lenRound, int dim8, Mat gate, Mat vals, float resMult, Mat res)
{
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    const long total = (long)lenRound * dim8;
    const long stride = (long)gridDim.x * 256;
    uint4 g[2], v[2];
    long id[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        id[k] = idx + k * stride;
        const int t = (int)(id[k] / dim8), c = (int)(id[k] - (long)t * dim8) * 8;
        const bool live = id[k] < total && t < len;
        g[k] = live ? *(const uint4 *)At<TBF16>(gate, t, c) : make_uint4(0, 0, 0, 0);
        v[k] = live ? *(const uint4 *)At<TBF16>(vals, t, c) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (id[k] >= total) {
            continue;
        }
        const int t = (int)(id[k] / dim8), c = (int)(id[k] - (long)t * dim8) * 8;
        const uint32_t gw[4] = {g[k].x, g[k].y, g[k].z, g[k].w}, vw[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        uint32_t out[2] = {0, 0};
        if (t < len) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float g0 = __uint_as_float(gw[w] << 16), g1 = __uint_as_float(gw[w] & 0xffff0000u);
                float v0 = __uint_as_float(vw[w] << 16), v1 = __uint_as_float(vw[w] & 0xffff0000u);
                out[w >> 1] |= CvtPkE4m3(v0 * LoLU1(g0) * resMult, v1 * LoLU1(g1) * resMult) << ((w & 1) * 16);
            }
        }
        *(uint2 *)At<TE4M3>(res, t, c) = make_uint2(out[0], out[1]);
    }
}

// Sixteen elements per lane: two 16-byte loads per input (the second is served by the line the first brought in) and one 16-byte store
__global__ void __launch_bounds__(256) MatrixLoLU16(int len, int lenRound, int dim16, Mat gate, Mat vals, float resMult, Mat res)
{
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    const long total = (long)lenRound * dim16;
    if (id >= total) {
        return;
    }
    const int t = (int)(id / dim16), c = (int)(id - (long)t * dim16) * 16;
    uint32_t out[4] = {0, 0, 0, 0};
    if (t < len) {
        const uint4 g0 = *(const uint4 *)At<TBF16>(gate, t, c), g1 = *(const uint4 *)At<TBF16>(gate, t, c + 8);
        const uint4 v0 = *(const uint4 *)At<TBF16>(vals, t, c), v1 = *(const uint4 *)At<TBF16>(vals, t, c + 8);
        const uint32_t gw[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w}, vw[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            float ga = __uint_as_float(gw[w] << 16), gb = __uint_as_float(gw[w] & 0xffff0000u);
            float va = __uint_as_float(vw[w] << 16), vb = __uint_as_float(vw[w] & 0xffff0000u);
            out[w >> 1] |= CvtPkE4m3(va * LoLU1(ga) * resMult, vb * LoLU1(gb) * resMult) << ((w & 1) * 16);
        }
    }
    *(uint4 *)At<TE4M3>(res, t, c) = make_uint4(out[0], out[1], out[2], out[3]);
}

// MODE 0: FFN (tile-norm backward of vals fused); MODE 1: attention (dScale fused)
template <class TGrad, class TOutG, class TOutV, int MODE>
__global__ void __launch_bounds__(256) BackpropLoLU(int len, int lenRound, int tiles, Mat gate, Mat vals, float valsScale, Mat valsSrcTileScale,
    Mat gradArr, Mat gradGate, Mat gradVals, Mat dScale)
{
    int t0, tile, h;
    if (!Unit(lenRound, tiles, &t0, &tile, &h)) {
        return;
    }
    int col = tile * TILE + h * 4;
    F4 g[U], v[U], grad[U];
    float ts[U], ds[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        int t = t0 + k;
        bool live = t < len;
        g[k] = live ? Load4<TBF16>(At<TBF16>(gate, t, col)) : ZeroF4();
        v[k] = live ? Load4<TBF16>(At<TBF16>(vals, t, col)) : ZeroF4();
        grad[k] = live ? Load4<TGrad>(At<TGrad>(gradArr, t, col)) : ZeroF4();
        ts[k] = (MODE == 0 && live) ? ScaleAt(valsSrcTileScale, tile, t) : 0.f;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        int t = t0 + k;
        ds[k] = 0;
        if (t >= lenRound) {
            continue;
        }
        F4 resGate = ZeroF4(), resVals = ZeroF4();
        if (t < len) {
            F4 vv = v[k] * valsScale;
            F4 mult = LoLU4(g[k]);
            resGate = grad[k] * vv * LoLUGrad4(mult);
            resVals = grad[k] * mult;
            if (MODE == 0) {
                // un-normalised source = normalised * (tile scale / valsScale)
                F4 src = vv * (ts[k] / valsScale);
                resVals = TileNormBackprop(src, resVals);
            } else {
                ds[k] = Half32Sum(HSum(vv * resVals));
            }
        }
        Store4<TOutG>(At<TOutG>(gradGate, t, col), resGate);
        Store4<TOutV>(At<TOutV>(gradVals, t, col), resVals);
    }
    if (MODE == 1) {
        StoreScales(dScale, tile, t0, lenRound, h, ds);
    }
}

// The FFN flavour (MODE 0) for bf16 gradients and e4m3 results with eight elements per lane: a 128-wide tile is 16 lanes, so a wave
// holds four (row, tile) units, the tile sums are four DPP steps inside a row of 16 lanes, loads are 16 bytes and stores 8.  Two
// units per lane in flight.  Same arithmetic per element as BackpropLoLU<.., 0>.
__device__ __forceinline__ float Row16Sum(float v);
__device__ __forceinline__ float Row16SumFwd(float v)
{
    return Row16Sum(v);
}

__device__ __forceinline__ float Row16Sum(float v)
{
    v += LaneDpp<DPP_XOR1>(v);
    v += LaneDpp<DPP_XOR2>(v);
    v += LaneDpp<DPP_HALF_MIRROR>(v);
    v += LaneDpp<DPP_MIRROR>(v);
    return v;
}

__global__ void __launch_bounds__(256) BackpropLoLU8(int len, int lenRound, int tiles, Mat gate, Mat vals, float valsScale, Mat valsSrcTileScale,
    Mat gradArr, Mat gradGate, Mat gradVals)
{
    constexpr int UU = 2;
    const int l16 = threadIdx.x & 15;
    const long unit0 = ((long)blockIdx.x * 256 + threadIdx.x) >> 4; // (row, tile) units; consecutive units = consecutive tiles of a row
    const long units = (long)lenRound * tiles;
    const long stride = ((long)gridDim.x * 256) >> 4;
    uint4 g[UU], v[UU], gr[UU];
    float ts[UU];
    int row[UU], col[UU];
    bool any[UU], live[UU];
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        long u = unit0 + k * stride;
        any[k] = u < units;
        row[k] = any[k] ? (int)(u / tiles) : 0;
        int tile = any[k] ? (int)(u - (long)row[k] * tiles) : 0;
        col[k] = tile * TILE + l16 * 8;
        live[k] = any[k] && row[k] < len;
        g[k] = live[k] ? *(const uint4 *)At<TBF16>(gate, row[k], col[k]) : make_uint4(0, 0, 0, 0);
        v[k] = live[k] ? *(const uint4 *)At<TBF16>(vals, row[k], col[k]) : make_uint4(0, 0, 0, 0);
        gr[k] = live[k] ? *(const uint4 *)At<TBF16>(gradArr, row[k], col[k]) : make_uint4(0, 0, 0, 0);
        ts[k] = live[k] ? ScaleAt(valsSrcTileScale, tile, row[k]) : 0.f;
    }
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        const uint32_t gw[4] = {g[k].x, g[k].y, g[k].z, g[k].w}, vw[4] = {v[k].x, v[k].y, v[k].z, v[k].w}, rw[4] = {gr[k].x, gr[k].y, gr[k].z, gr[k].w};
        float resGate[8], resVals[8], src[8];
        float sum2 = 0, dp = 0;
        const float srcMult = ts[k] / valsScale;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t sh = (e & 1) ? 0xffff0000u : 0u;
            float ge = (e & 1) ? __uint_as_float(gw[e >> 1] & sh) : __uint_as_float(gw[e >> 1] << 16);
            float ve = (e & 1) ? __uint_as_float(vw[e >> 1] & sh) : __uint_as_float(vw[e >> 1] << 16);
            float de = (e & 1) ? __uint_as_float(rw[e >> 1] & sh) : __uint_as_float(rw[e >> 1] << 16);
            float vv = ve * valsScale;
            float mult = LoLU1(ge);
            resGate[e] = de * vv * (mult * (1 - mult) * 2.f);
            resVals[e] = de * mult;
            // un-normalised source = normalised * (tile scale / valsScale)
            src[e] = vv * srcMult;
            sum2 += src[e] * src[e];
            dp += src[e] * resVals[e];
        }
        sum2 = Row16Sum(sum2);
        dp = Row16Sum(dp);
        if (!any[k]) {
            continue;
        }
        uint32_t og[2] = {0, 0}, ov[2] = {0, 0};
        if (live[k]) {
            float sigma = 0, scale = 0;
            if (sum2 != 0) {
                float inv = 1 / sum2;
                sigma = dp * inv;
                scale = sqrtf(TILE * inv);
            }
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float a0 = sum2 != 0 ? (resVals[2 * w] - src[2 * w] * sigma) * scale : 0.f;
                float a1 = sum2 != 0 ? (resVals[2 * w + 1] - src[2 * w + 1] * sigma) * scale : 0.f;
                ov[w >> 1] |= CvtPkE4m3(a0, a1) << ((w & 1) * 16);
                og[w >> 1] |= CvtPkE4m3(resGate[2 * w], resGate[2 * w + 1]) << ((w & 1) * 16);
            }
        }
        *(uint2 *)At<TE4M3>(gradGate, row[k], col[k]) = make_uint2(og[0], og[1]);
        *(uint2 *)At<TE4M3>(gradVals, row[k], col[k]) = make_uint2(ov[0], ov[1]);
    }
}

// A 128 x 128 block of bytes staged in LDS as [t][x] (pitch PITCH) goes out transposed: dst[x][t], 16 bytes (16 t) per store.
// thread -> (tq = block of 16 t, xq = x quad)
template <int PITCH> __device__ __forceinline__ void TransposeOut128(const uint8_t *buf, const Mat &dst, int xBlock, int tBlock, int tid)
{
    const int tq = tid & 7, xq = tid >> 3;
    uint32_t out[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint8_t *b = buf + (tq * 16 + j * 4) * PITCH + xq * 4;
        uint32_t r0 = *(const uint32_t *)(b);
        uint32_t r1 = *(const uint32_t *)(b + PITCH);
        uint32_t r2 = *(const uint32_t *)(b + 2 * PITCH);
        uint32_t r3 = *(const uint32_t *)(b + 3 * PITCH);
        // 4x4 byte transpose.  __builtin_amdgcn_perm(hi, lo, sel): result byte i = byte sel[i] of {hi:lo} (lo = bytes 0-3)
        uint32_t a = __builtin_amdgcn_perm(r1, r0, 0x05010400); // r0.b0 r1.b0 r0.b1 r1.b1
        uint32_t bb = __builtin_amdgcn_perm(r1, r0, 0x07030602); // r0.b2 r1.b2 r0.b3 r1.b3
        uint32_t c = __builtin_amdgcn_perm(r3, r2, 0x05010400);
        uint32_t d = __builtin_amdgcn_perm(r3, r2, 0x07030602);
        out[0][j] = __builtin_amdgcn_perm(c, a, 0x05040100); // column 0: r0.b0 r1.b0 r2.b0 r3.b0
        out[1][j] = __builtin_amdgcn_perm(c, a, 0x07060302);
        out[2][j] = __builtin_amdgcn_perm(d, bb, 0x05040100);
        out[3][j] = __builtin_amdgcn_perm(d, bb, 0x07060302);
    }
    int x = xBlock + xq * 4;
    int tcol = tBlock + tq * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        *(uint4 *)(dst.p + (int64_t)(x + i) * dst.ld + tcol) = make_uint4(out[i][0], out[i][1], out[i][2], out[i][3]);
    }
}

// BackpropLoLU8 that also leaves the transposed copies of both results (gradGateT, gradValsT: [dim][lenRound]) which the delta
// products of the two matrices contract over: a workgroup takes a block of 128 rows x one tile, computes it 16 rows at a time with
// the arithmetic of BackpropLoLU8, stores the row-major bytes and stages them in LDS for the transposed stores.  Saves reading both
// results back for their transposes.
__global__ void __launch_bounds__(256) BackpropLoLU8T(int len, int lenRound, Mat gate, Mat vals, float valsScale, Mat valsSrcTileScale, Mat gradArr,
    Mat gradGate, Mat gradVals, Mat gradGateT, Mat gradValsT)
{
    constexpr int PITCH = 132;
    __shared__ __attribute__((aligned(16))) uint8_t bufG[128 * PITCH], bufV[128 * PITCH];
    const int tid = threadIdx.x, l16 = tid & 15, lr = tid >> 4;
    const int tile = blockIdx.x, tBlock = blockIdx.y * 128;
    const int col = tile * TILE + l16 * 8;
    for (int r0 = 0; r0 < 128; r0 += 64) {
        uint4 g[4], v[4], gr[4];
        float ts[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int row = tBlock + r0 + k * 16 + lr;
            const bool live = row < len;
            g[k] = live ? *(const uint4 *)At<TBF16>(gate, row, col) : make_uint4(0, 0, 0, 0);
            v[k] = live ? *(const uint4 *)At<TBF16>(vals, row, col) : make_uint4(0, 0, 0, 0);
            gr[k] = live ? *(const uint4 *)At<TBF16>(gradArr, row, col) : make_uint4(0, 0, 0, 0);
            ts[k] = live ? ScaleAt(valsSrcTileScale, tile, row) : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = r0 + k * 16 + lr, row = tBlock + r;
            const uint32_t gw[4] = {g[k].x, g[k].y, g[k].z, g[k].w}, vw[4] = {v[k].x, v[k].y, v[k].z, v[k].w}, rw[4] = {gr[k].x, gr[k].y, gr[k].z, gr[k].w};
            float resGate[8], resVals[8], src[8];
            float sum2 = 0, dp = 0;
            const float srcMult = ts[k] / valsScale;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t sh = 0xffff0000u;
                float ge = (e & 1) ? __uint_as_float(gw[e >> 1] & sh) : __uint_as_float(gw[e >> 1] << 16);
                float ve = (e & 1) ? __uint_as_float(vw[e >> 1] & sh) : __uint_as_float(vw[e >> 1] << 16);
                float de = (e & 1) ? __uint_as_float(rw[e >> 1] & sh) : __uint_as_float(rw[e >> 1] << 16);
                float vv = ve * valsScale;
                float mult = LoLU1(ge);
                resGate[e] = de * vv * (mult * (1 - mult) * 2.f);
                resVals[e] = de * mult;
                src[e] = vv * srcMult;
                sum2 += src[e] * src[e];
                dp += src[e] * resVals[e];
            }
            sum2 = Row16Sum(sum2);
            dp = Row16Sum(dp);
            uint32_t og[2] = {0, 0}, ov[2] = {0, 0};
            if (row < len) {
                float sigma = 0, scale = 0;
                if (sum2 != 0) {
                    float inv = 1 / sum2;
                    sigma = dp * inv;
                    scale = sqrtf(TILE * inv);
                }
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    float a0 = sum2 != 0 ? (resVals[2 * w] - src[2 * w] * sigma) * scale : 0.f;
                    float a1 = sum2 != 0 ? (resVals[2 * w + 1] - src[2 * w + 1] * sigma) * scale : 0.f;
                    ov[w >> 1] |= CvtPkE4m3(a0, a1) << ((w & 1) * 16);
                    og[w >> 1] |= CvtPkE4m3(resGate[2 * w], resGate[2 * w + 1]) << ((w & 1) * 16);
                }
            }
            *(uint2 *)At<TE4M3>(gradGate, row, col) = make_uint2(og[0], og[1]);
            *(uint2 *)At<TE4M3>(gradVals, row, col) = make_uint2(ov[0], ov[1]);
            *(uint32_t *)(bufG + r * PITCH + l16 * 8) = og[0];
            *(uint32_t *)(bufG + r * PITCH + l16 * 8 + 4) = og[1];
            *(uint32_t *)(bufV + r * PITCH + l16 * 8) = ov[0];
            *(uint32_t *)(bufV + r * PITCH + l16 * 8 + 4) = ov[1];
        }
    }
    __syncthreads();
    TransposeOut128<PITCH>(bufG, gradGateT, tile * TILE, tBlock, tid);
    TransposeOut128<PITCH>(bufV, gradValsT, tile * TILE, tBlock, tid);
}

// The attention flavour (MODE 1) with eight elements per lane: bf16 gate, values and gradient in, e4m3 gate gradient and bf16 value
// gradient out, and the per-(head, row) sum <values, value gradient> that the attention backward subtracts (dScale).
__global__ void __launch_bounds__(256) BackpropLoLUAtt8(int len, int lenRound, int tiles, Mat gate, Mat vals, float valsScale, Mat gradArr,
    Mat gradGate, Mat gradVals, Mat dScale)
{
    constexpr int UU = 2;
    const int l16 = threadIdx.x & 15;
    const long unit0 = ((long)blockIdx.x * 256 + threadIdx.x) >> 4; // (row, tile) units; consecutive units = consecutive tiles of a row
    const long units = (long)lenRound * tiles;
    const long stride = ((long)gridDim.x * 256) >> 4;
    uint4 g[UU], v[UU], gr[UU];
    int row[UU], tile[UU];
    bool any[UU], live[UU];
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        long u = unit0 + k * stride;
        any[k] = u < units;
        row[k] = any[k] ? (int)(u / tiles) : 0;
        tile[k] = any[k] ? (int)(u - (long)row[k] * tiles) : 0;
        const int col = tile[k] * TILE + l16 * 8;
        live[k] = any[k] && row[k] < len;
        g[k] = live[k] ? *(const uint4 *)At<TBF16>(gate, row[k], col) : make_uint4(0, 0, 0, 0);
        v[k] = live[k] ? *(const uint4 *)At<TBF16>(vals, row[k], col) : make_uint4(0, 0, 0, 0);
        gr[k] = live[k] ? *(const uint4 *)At<TBF16>(gradArr, row[k], col) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        const uint32_t gw[4] = {g[k].x, g[k].y, g[k].z, g[k].w}, vw[4] = {v[k].x, v[k].y, v[k].z, v[k].w}, rw[4] = {gr[k].x, gr[k].y, gr[k].z, gr[k].w};
        float resGate[8], resVals[8];
        float dp = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t sh = 0xffff0000u;
            float ge = (e & 1) ? __uint_as_float(gw[e >> 1] & sh) : __uint_as_float(gw[e >> 1] << 16);
            float ve = (e & 1) ? __uint_as_float(vw[e >> 1] & sh) : __uint_as_float(vw[e >> 1] << 16);
            float de = (e & 1) ? __uint_as_float(rw[e >> 1] & sh) : __uint_as_float(rw[e >> 1] << 16);
            float vv = ve * valsScale;
            float mult = LoLU1(ge);
            resGate[e] = de * vv * (mult * (1 - mult) * 2.f);
            resVals[e] = de * mult;
            dp += vv * resVals[e];
        }
        dp = Row16Sum(dp); // zero for rows past len: their inputs were read as zero
        if (!any[k]) {
            continue;
        }
        const int col = tile[k] * TILE + l16 * 8;
        uint32_t og[2] = {0, 0}, ov[4] = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            og[w >> 1] |= CvtPkE4m3(resGate[2 * w], resGate[2 * w + 1]) << ((w & 1) * 16);
            ov[w] = PackBf16x2(resVals[2 * w], resVals[2 * w + 1]);
        }
        *(uint2 *)At<TE4M3>(gradGate, row[k], col) = make_uint2(og[0], og[1]);
        *(uint4 *)At<TBF16>(gradVals, row[k], col) = make_uint4(ov[0], ov[1], ov[2], ov[3]);
        if (l16 == 0) {
            ScaleAt(dScale, tile[k], row[k]) = dp;
        }
    }
}

// Workgroups walk rows with a grid stride; a row stays in registers between the abs-max pass and the quantise pass when it has at
// most 4096 elements (REG) and the next row is fetched before the current one is reduced, so a workgroup always has loads in
// flight.  Longer rows are read twice (the second read is served by L2).
template <class TSrc, bool REG>
__global__ void __launch_bounds__(256) NormalizeVecsRowMax(int len, int lenRound, int dim, Mat src, const float *colScale, Mat dst, float *rowScale,
    float *rowAbsMax, uint32_t seed)
{
    __shared__ float red[2][4], redPlain[2][4];
    const int tid = threadIdx.x;
    F4 next[4];
    auto fetch = [&](int t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int col = tid * 4 + i * 1024;
            next[i] = (REG && t < len && col < dim) ? Load4<TSrc>(At<TSrc>(src, t, col)) : ZeroF4();
        }
    };
    fetch(blockIdx.x);
    int phase = 0;
    for (int t = blockIdx.x; t < lenRound; t += gridDim.x, phase ^= 1) {
        if (t >= len) {
            for (int col = tid * 4; col < dim; col += 1024) {
                *(uint32_t *)At<TI8>(dst, t, col) = 0;
            }
            if (tid == 0) {
                rowScale[t] = 0;
                if (rowAbsMax) {
                    rowAbsMax[t] = 0;
                }
            }
            continue;
        }
        float mx = 0, plain = 0; // plain: abs-max of the row before the column scales (what the delta's k-tile scale is built from)
        F4 keep[4];
        if (REG) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                keep[i] = next[i];
            }
            fetch(t + gridDim.x);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                plain = fmaxf(plain, HMaxAbs(keep[i]));
            }
            if (colScale) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int col = tid * 4 + i * 1024;
                    if (col < dim) {
                        keep[i] = keep[i] * Load4<TF32>(colScale + col);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                mx = fmaxf(mx, HMaxAbs(keep[i]));
            }
        } else {
            for (int col = tid * 4; col < dim; col += 1024) {
                F4 v = Load4<TSrc>(At<TSrc>(src, t, col));
                plain = fmaxf(plain, HMaxAbs(v));
                if (colScale) {
                    v = v * Load4<TF32>(colScale + col);
                }
                mx = fmaxf(mx, HMaxAbs(v));
            }
        }
        mx = WaveMax(mx);
        plain = WaveMax(plain);
        if ((tid & 63) == 0) {
            red[phase][tid >> 6] = mx;
            redPlain[phase][tid >> 6] = plain;
        }
        __syncthreads(); // the two phases of the exchange arrays make one barrier per row enough
        mx = fmaxf(fmaxf(red[phase][0], red[phase][1]), fmaxf(red[phase][2], red[phase][3]));
        if (tid == 0 && rowAbsMax) {
            rowAbsMax[t] = fmaxf(fmaxf(redPlain[phase][0], redPlain[phase][1]), fmaxf(redPlain[phase][2], redPlain[phase][3]));
        }
        float discr = 0, mult = 0;
        if (mx > 0) {
            discr = mx / 127;
            mult = 1 / discr;
        }
        if (REG) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int col = tid * 4 + i * 1024;
                if (col < dim) {
                    if (seed) {
                        *(uint32_t *)At<TI8>(dst, t, col) = QuantDither4(keep[i].x, keep[i].y, keep[i].z, keep[i].w, mult, DitherWord(seed, t, col >> 2));
                    } else {
                        Store4<TI8>(At<TI8>(dst, t, col), keep[i] * mult);
                    }
                }
            }
        } else {
            for (int col = tid * 4; col < dim; col += 1024) {
                F4 v = Load4<TSrc>(At<TSrc>(src, t, col));
                if (colScale) {
                    v = v * Load4<TF32>(colScale + col);
                }
                if (seed) {
                    *(uint32_t *)At<TI8>(dst, t, col) = QuantDither4(v.x, v.y, v.z, v.w, mult, DitherWord(seed, t, col >> 2));
                } else {
                    Store4<TI8>(At<TI8>(dst, t, col), v * mult);
                }
            }
        }
        if (tid == 0) {
            rowScale[t] = discr;
        }
    }
}

// The same quantiser with one wave per row for bf16 rows of at most NCH * 512 <= 4096 elements (a multiple of 8): a lane holds NCH chunks
// of 8 consecutive elements (16-byte loads, 8-byte stores, each instruction of the wave covering 1 KB / 512 B of the row), the row
// maxima are wave reductions, and no workgroup barrier or LDS exchange is left.  Same arithmetic per element as NormalizeVecsRowMax.
// Batch: blockIdx.y = source, the gradients of a layer's matrices go in one launch (rows of 384 elements, 16384 of them: 13.6 us each one by one
// with a workgroup per row).
struct RowQuantJobs {
    Mat src[4], dst[4];
    float *rowScale[4], *rowAbsMax[4];
    uint32_t seed[4];
};

// codes, scale and (where asked for) plain maximum of a row that a wave holds as NCH chunks of 8 elements per lane; mx, plain: maxima of the
// lane's own elements, with and without column scales.  Returns the row's maximum with them
template <int NCH>
__device__ __forceinline__ float StoreRowCodes(const F4 (&v)[NCH][2], const bool (&in)[NCH], int lane, int t, float mx, float plain, uint8_t *out,
    float *rowScale, float *rowAbsMax, uint32_t seed)
{
    mx = WaveMax(mx);
    plain = WaveMax(plain);
    float discr = 0, mult = 0;
    if (mx > 0) {
        discr = mx / 127;
        mult = 1 / discr;
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        if (!in[i]) {
            continue;
        }
        if (seed) {
            const int col4 = (i * 64 + lane) * 2;
            *(uint2 *)(out + (i * 64 + lane) * 8) =
                make_uint2(QuantDither4(v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, mult, DitherWord(seed, t, col4)),
                    QuantDither4(v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w, mult, DitherWord(seed, t, col4 + 1)));
            continue;
        }
        F4 a = v[i][0] * mult, b = v[i][1] * mult;
        uint32_t lo = (uint32_t)(CvtToI8(a.x) & 0xff) | ((uint32_t)(CvtToI8(a.y) & 0xff) << 8) | ((uint32_t)(CvtToI8(a.z) & 0xff) << 16) |
                      ((uint32_t)(CvtToI8(a.w) & 0xff) << 24);
        uint32_t hi = (uint32_t)(CvtToI8(b.x) & 0xff) | ((uint32_t)(CvtToI8(b.y) & 0xff) << 8) | ((uint32_t)(CvtToI8(b.z) & 0xff) << 16) |
                      ((uint32_t)(CvtToI8(b.w) & 0xff) << 24);
        *(uint2 *)(out + (i * 64 + lane) * 8) = make_uint2(lo, hi);
    }
    if (lane == 0) {
        rowScale[t] = discr;
        if (rowAbsMax) {
            rowAbsMax[t] = plain;
        }
    }
    return mx;
}

__device__ __forceinline__ void Unpack8(const uint4 &raw, F4 (&v)[2])
{
    v[0] = MakeF4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u));
    v[1] = MakeF4(__uint_as_float(raw.z << 16), __uint_as_float(raw.z & 0xffff0000u), __uint_as_float(raw.w << 16), __uint_as_float(raw.w & 0xffff0000u));
}

// FULL: rows of exactly NCH * 512 elements.
template <int NCH, bool FULL>
__device__ __forceinline__ void NormalizeRowsWaveOf(int len, int lenRound, int dim, const Mat &src, const float *colScale, const Mat &dst,
    float *rowScale, float *rowAbsMax, uint32_t seed)
{
    const int lane = threadIdx.x & 63;
    bool in[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        in[i] = FULL || (i * 64 + lane) * 8 < dim;
    }
    const int nWaves = gridDim.x * 4;
    // the column scales of the lane's chunks stay in registers for all the rows the wave walks
    F4 cs[NCH][2];
    if (colScale) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            cs[i][0] = in[i] ? Load4<TF32>(colScale + (i * 64 + lane) * 8) : ZeroF4();
            cs[i][1] = in[i] ? Load4<TF32>(colScale + (i * 64 + lane) * 8 + 4) : ZeroF4();
        }
    }
    for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < lenRound; t += nWaves) {
        uint8_t *out = dst.p + (int64_t)t * dst.ld;
        if (t >= len) {
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                if (in[i]) {
                    *(uint2 *)(out + (i * 64 + lane) * 8) = make_uint2(0u, 0u);
                }
            }
            if (lane == 0) {
                rowScale[t] = 0;
                if (rowAbsMax) {
                    rowAbsMax[t] = 0;
                }
            }
            continue;
        }
        const uint8_t *row = src.p + (int64_t)t * src.ld;
        uint4 raw[NCH];
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            raw[i] = in[i] ? *(const uint4 *)(row + (i * 64 + lane) * 16) : make_uint4(0, 0, 0, 0);
        }
        F4 v[NCH][2];
        float mx = 0, plain = 0;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            v[i][0] = MakeF4(__uint_as_float(raw[i].x << 16), __uint_as_float(raw[i].x & 0xffff0000u), __uint_as_float(raw[i].y << 16),
                __uint_as_float(raw[i].y & 0xffff0000u));
            v[i][1] = MakeF4(__uint_as_float(raw[i].z << 16), __uint_as_float(raw[i].z & 0xffff0000u), __uint_as_float(raw[i].w << 16),
                __uint_as_float(raw[i].w & 0xffff0000u));
            plain = fmaxf(plain, fmaxf(HMaxAbs(v[i][0]), HMaxAbs(v[i][1])));
            if (colScale) {
                v[i][0] = v[i][0] * cs[i][0];
                v[i][1] = v[i][1] * cs[i][1];
            }
            mx = fmaxf(mx, fmaxf(HMaxAbs(v[i][0]), HMaxAbs(v[i][1])));
        }
        StoreRowCodes<NCH>(v, in, lane, t, mx, plain, out, rowScale, rowAbsMax, seed);
    }
}

template <int NCH, bool FULL>
__global__ void __launch_bounds__(256) NormalizeRowsWaveBatch(int len, int lenRound, int dim, RowQuantJobs jobs)
{
    const int j = blockIdx.y;
    NormalizeRowsWaveOf<NCH, FULL>(len, lenRound, dim, jobs.src[j], nullptr, jobs.dst[j], jobs.rowScale[j], jobs.rowAbsMax[j], jobs.seed[j]);
}

// one source: its description lies in scalar registers from the start (16384 x 4096: 36.5 us, 37.6 through the job table)
template <int NCH, bool FULL>
__global__ void __launch_bounds__(256) NormalizeRowsWave(int len, int lenRound, int dim, Mat src, const float *colScale, Mat dst, float *rowScale,
    float *rowAbsMax, uint32_t seed)
{
    NormalizeRowsWaveOf<NCH, FULL>(len, lenRound, FULL ? NCH * 512 : dim, src, colScale, dst, rowScale, rowAbsMax, seed);
}

// ---- int8: gradient passes that also quantise the rows they write, for the dX product that reads them next (the arithmetic of the passes and of
// NormalizeRowsWave).  A wave owns a row, a lane NCH chunks of 8 elements of it, so that a 128-wide tile is 16 lanes (a lane adds its two groups of
// four before the first step across lanes: the same tree of sums as on 32 lanes) and the row's maximum is a wave reduction over values that are
// still in registers.  A quantiser of its own reads everything again and costs a launch: per layer of the 512-token int8 step 6.1 + 3.1, 7.4 +
// 3.5, 5.7 + 3.7 us -> 4.5, 5.7, 4.3; 16384 x 512 (normalisation, gate) 27.3 + 7.6, 28.1 + 12.5 -> 28.7, 24.3; 16384 x 384 (gate; Q, K, V) 16 + 24.6 +
// 24 -> 16.2, 26.3

// rope pairs are (cos, sin) interleaved: a lane holds two of them
__device__ __forceinline__ F4 ApplyRope4(F4 v, F4 rope, float dir)
{
    float s0 = rope.y * dir, s1 = rope.w * dir;
    return MakeF4(v.x * rope.x - v.y * s0, v.x * s0 + v.y * rope.x, v.z * rope.z - v.w * s1, v.z * s1 + v.w * rope.z);
}

__device__ __forceinline__ uint4 Pack8(const F4 &a, const F4 &b)
{
    return make_uint4(PackBf16x2(a.x, a.y), PackBf16x2(a.z, a.w), PackBf16x2(b.x, b.y), PackBf16x2(b.z, b.w));
}

// TileNormBackprop of a tile on 16 lanes; ownSum2, ownDp: the lane's parts of sum(src * src) and sum(src * g)
__device__ __forceinline__ void TileNormBackprop8(const F4 (&src)[2], F4 (&g)[2], float ownSum2, float ownDp)
{
    const float sum2 = Row16Sum(ownSum2), dp = Row16Sum(ownDp);
    if (sum2 == 0) {
        g[0] = g[1] = ZeroF4();
        return;
    }
    const float inv = 1 / sum2;
    const float sigma = dp * inv, scale = sqrtf(TILE * inv);
    g[0] = (g[0] - src[0] * sigma) * scale;
    g[1] = (g[1] - src[1] * sigma) * scale;
}

__device__ __forceinline__ void TileNormBackprop8(const F4 (&src)[2], F4 (&g)[2])
{
    TileNormBackprop8(src, g, HSum(src[0] * src[0]) + HSum(src[1] * src[1]), HSum(src[0] * g[0]) + HSum(src[1] * g[1]));
}

// a row of bf16 values that the wave kept (zeros beyond the live rows), quantised; returns its maximum
template <int NCH> __device__ __forceinline__ float QuantKeptRow(const uint4 (&kept)[NCH], const bool (&in)[NCH], int lane, int t, const RowQuantOut &q)
{
    F4 v[NCH][2];
    float mx = 0;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        Unpack8(kept[i], v[i]);
        mx = fmaxf(mx, fmaxf(HMaxAbs(v[i][0]), HMaxAbs(v[i][1])));
    }
    return StoreRowCodes<NCH>(v, in, lane, t, mx, mx, q.dst + (int64_t)t * q.dstStride, q.rowScale, q.rowAbsMax, q.seed);
}

// BackpropLoLU<TBF16, TBF16, TBF16, MODE> over whole rows; MODE 1 quantises the gate's gradient only
template <int NCH, int MODE>
__global__ void __launch_bounds__(256) BackpropLoLURows(int len, int lenRound, int dim, Mat gate, Mat vals, float valsScale, Mat valsSrcTileScale,
    Mat gradArr, Mat gradGate, Mat gradVals, Mat dScale, RowQuantOut qGate, RowQuantOut qVals)
{
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= lenRound) {
        return;
    }
    const bool live = t < len;
    bool in[NCH];
    uint4 g[NCH], v[NCH], grad[NCH];
    float ts[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int col = (i * 64 + lane) * 8;
        in[i] = col < dim;
        const bool use = live && in[i];
        g[i] = use ? *(const uint4 *)At<TBF16>(gate, t, col) : make_uint4(0, 0, 0, 0);
        v[i] = use ? *(const uint4 *)At<TBF16>(vals, t, col) : make_uint4(0, 0, 0, 0);
        grad[i] = use ? *(const uint4 *)At<TBF16>(gradArr, t, col) : make_uint4(0, 0, 0, 0);
        ts[i] = use && MODE == 0 ? ScaleAt(valsSrcTileScale, col / TILE, t) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int col = (i * 64 + lane) * 8;
        F4 gg[2], vv[2], gr[2], resGate[2], resVals[2];
        Unpack8(g[i], gg);
        Unpack8(v[i], vv);
        Unpack8(grad[i], gr);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            vv[k] = vv[k] * valsScale;
            const F4 mult = LoLU4(gg[k]);
            resGate[k] = gr[k] * vv[k] * LoLUGrad4(mult);
            resVals[k] = gr[k] * mult;
        }
        if (MODE == 0) {
            const float unNorm = ts[i] / valsScale;
            const F4 src[2] = {vv[0] * unNorm, vv[1] * unNorm};
            TileNormBackprop8(src, resVals);
        } else {
            const float ds = Row16Sum(HSum(vv[0] * resVals[0]) + HSum(vv[1] * resVals[1]));
            if (in[i] && (lane & 15) == 0) {
                ScaleAt(dScale, col / TILE, t) = live ? ds : 0.f;
            }
        }
        // (rows that are not live hold zeros)
        g[i] = live ? Pack8(resGate[0], resGate[1]) : make_uint4(0, 0, 0, 0);
        v[i] = live ? Pack8(resVals[0], resVals[1]) : make_uint4(0, 0, 0, 0);
        if (in[i]) {
            *(uint4 *)At<TBF16>(gradGate, t, col) = g[i];
            *(uint4 *)At<TBF16>(gradVals, t, col) = v[i];
        }
    }
    QuantKeptRow<NCH>(g, in, lane, t, qGate);
    if (MODE == 0) {
        QuantKeptRow<NCH>(v, in, lane, t, qVals);
    }
}

// BackpropRowTileNormalizeRope<TBF16, TBF16> over whole rows, blockIdx.y = gradient
struct NormRopeRowJobs {
    Mat grad[3], srcNorm[3], srcTileScale[3], rope[3], dst[3];
    RowQuantOut q[3];
};
template <int NCH> __global__ void __launch_bounds__(256) BackpropNormRopeRows(int len, int lenRound, int dim, float gradMult, NormRopeRowJobs jobs)
{
    const int j = blockIdx.y;
    const Mat grad = jobs.grad[j], srcNorm = jobs.srcNorm[j], srcTileScale = jobs.srcTileScale[j], rope = jobs.rope[j], dst = jobs.dst[j];
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= lenRound) {
        return;
    }
    const bool live = t < len;
    bool in[NCH];
    uint4 g[NCH], sn[NCH];
    float sc[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int col = (i * 64 + lane) * 8;
        in[i] = col < dim;
        const bool use = live && in[i];
        g[i] = use ? *(const uint4 *)At<TBF16>(grad, t, col) : make_uint4(0, 0, 0, 0);
        sn[i] = use && srcNorm.p ? *(const uint4 *)At<TBF16>(srcNorm, t, col) : make_uint4(0, 0, 0, 0);
        sc[i] = use && srcNorm.p ? ScaleAt(srcTileScale, col / TILE, t) : 0.f;
    }
    F4 rp[2] = {ZeroF4(), ZeroF4()};
    if (rope.p && live) {
        rp[0] = Load4<TF32>(At<TF32>(rope, t, (lane & 15) * 8));
        rp[1] = Load4<TF32>(At<TF32>(rope, t, (lane & 15) * 8 + 4));
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        F4 x[2], s[2];
        Unpack8(g[i], x);
        x[0] = x[0] * gradMult;
        x[1] = x[1] * gradMult;
        if (srcNorm.p) {
            Unpack8(sn[i], s);
            const F4 src[2] = {s[0] * sc[i], s[1] * sc[i]};
            TileNormBackprop8(src, x);
        }
        if (rope.p) {
            x[0] = ApplyRope4(x[0], rp[0], -1.f);
            x[1] = ApplyRope4(x[1], rp[1], -1.f);
        }
        g[i] = live ? Pack8(x[0], x[1]) : make_uint4(0, 0, 0, 0);
        if (in[i]) {
            *(uint4 *)At<TBF16>(dst, t, (i * 64 + lane) * 8) = g[i];
        }
    }
    QuantKeptRow<NCH>(g, in, lane, t, jobs.q[j]);
}

// BackpropLayerNormalize<TI8, TBF16, FINAL> over whole rows; the codes belong to the multiplier known here and move to the next one in ScaleGrad.
// Rows len .. lenRound: codes and scales are cleared, FINAL clears its results there too
template <int NCH, bool FINAL, int NT>
__global__ void __launch_bounds__(NT) BackpropLayerNormalizeRows(int len, int lenRound, int dim, Mat normState, Mat stateScale, Mat dNormState,
    const float *gradScale, const float *gradMult, Mat stateGrad, Mat stateGradFast, float *nextMaxNorm, RowQuantOut q)
{
    __shared__ float red[NT / 64];
    const int lane = threadIdx.x & 63;
    const float s = !FINAL && gradScale ? *gradScale : 1.f, gm = !FINAL && gradMult ? *gradMult : 1.f;
    float gmax = 0;
    for (int t = blockIdx.x * (NT / 64) + (threadIdx.x >> 6); t < lenRound; t += gridDim.x * (NT / 64)) {
        const bool live = t < len;
        bool in[NCH];
        uint2 nv[NCH];
        F4 grad[NCH][2], prev[NCH][2];
        float sc[NCH];
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int col = (i * 64 + lane) * 8;
            in[i] = col < dim;
            const bool use = live && in[i];
            nv[i] = use ? *(const uint2 *)At<TI8>(normState, t, col) : make_uint2(0, 0);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                grad[i][k] = use ? Load4<TF32>(At<TF32>(dNormState, t, col + k * 4)) : ZeroF4();
                prev[i][k] = use && !FINAL ? Load4<TF32>(At<TF32>(stateGrad, t, col + k * 4)) : ZeroF4();
            }
            sc[i] = use ? ScaleAt(stateScale, col / TILE, t) : 0.f;
        }
        uint4 kept[NCH];
        float top = 0;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int col = (i * 64 + lane) * 8;
            const F4 src[2] = {Load4<TI8>(&nv[i].x) * sc[i], Load4<TI8>(&nv[i].y) * sc[i]};
            F4 g[2] = {grad[i][0], grad[i][1]};
            if (!FINAL) {
                g[0] = g[0] * s;
                g[1] = g[1] * s;
            }
            // (the products that the compiler fuses in BackpropLayerNormalize, so that the gradients are its bits)
            auto squares = [](const F4 &a) { return __builtin_fmaf(a.x, a.x, a.y * a.y) + __builtin_fmaf(a.z, a.z, a.w * a.w); };
            auto dot = [](const F4 &a, const F4 &b) { return __builtin_fmaf(a.y, b.y, a.x * b.x) + __builtin_fmaf(a.w, b.w, a.z * b.z); };
            TileNormBackprop8(src, g, squares(src[0]) + squares(src[1]), dot(src[0], g[0]) + dot(src[1], g[1]));
            if (!FINAL) {
                g[0] = g[0] + prev[i][0];
                g[1] = g[1] + prev[i][1];
            }
            if (!live) {
                g[0] = g[1] = ZeroF4();
            }
            top = fmaxf(top, fmaxf(HMaxAbs(g[0]), HMaxAbs(g[1])));
            kept[i] = Pack8(g[0] * gm, g[1] * gm);
            if (in[i] && (FINAL || live)) {
                Store4<TF32>(At<TF32>(stateGrad, t, col), g[0]);
                Store4<TF32>(At<TF32>(stateGrad, t, col + 4), g[1]);
                *(uint4 *)At<TBF16>(stateGradFast, t, col) = kept[i];
            }
        }
        gmax = fmaxf(gmax, top);
        if (QuantKeptRow<NCH>(kept, in, lane, t, q) == 0 && __any(top != 0) && lane == 0) {
            q.rowScale[t] = 1; // the codes are zeros, the gradients are not (MoveRowCodes)
        }
    }
    PublishBlockMax<NT>(gmax, red, nextMaxNorm);
}

// Row-major k-tile quantiser: dst[t][x] = sat_i8(rne(src[t][x] * rowMult[t] / scale)) with one scale per kTile rows, formed from the row maxima
// that the row quantiser left (the arithmetic and the dither of TransposeQuant, without its transpose: the delta product reads both
// operands contraction-major).  A workgroup takes QT_ROWS rows, which lie in one k-tile; rows in [len, lenRound) are cleared.  blockIdx.y =
// source; tileScale: [sources][lenRound / kTile].  Rows per workgroup 32 -> 8: 512 x 1024, two gradients 13.1 -> 5.3 us; 16384 x 512 9.6 -> 7.9
constexpr int QT_ROWS = 8;
constexpr int QT_JOBS = 48; // most sources of a launch (56 bytes of its arguments each)
template <int COUNT> struct TileQuantJobs {
    TileQuantJob job[COUNT];
};

template <int COUNT>
__global__ void __launch_bounds__(256) QuantTileRows(int len, int lenRound, int kTile, TileQuantJobs<COUNT> jobs, const float *rowMult)
{
    __shared__ float red[4];
    const TileQuantJob &job = jobs.job[blockIdx.y];
    const Mat src = {(uint8_t *)job.src, job.srcStride}, dst = {job.dst, job.dstStride};
    const float *rowAbsMax = job.rowAbsMax;
    const uint32_t seed = job.seed;
    const int dim = job.dim;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = blockIdx.x * QT_ROWS, k0 = t0 / kTile * kTile;
    float mx = 0;
    for (int t = k0 + tid; t < k0 + kTile && t < len; t += 256) {
        float m = rowAbsMax[t];
        if (rowMult) {
            m *= fabsf(rowMult[t]);
        }
        mx = fmaxf(mx, m);
    }
    mx = WaveMax(mx);
    if (lane == 0) {
        red[wave] = mx;
    }
    __syncthreads();
    const float tm = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float mult = tm > 0 ? 1 / (tm / 127) : 0.f;
    if (tid == 0 && t0 == k0) {
        job.tileScale[t0 / kTile] = tm > 0 ? tm / 127 : 1.f;
    }
    // units of 8 elements, walked by the whole workgroup: four 16-byte loads in flight per lane.  (Asked for before the maxima, the first four of them cost
    // launches of few gradients and of 1024 columns 4-5 %: 16384 x 512, two gradients 14.3 -> 15.1, 8192 x 1024, 24 of them 113 -> 120; 40 of 16384 x 384
    // and 512 gained 202 -> 188.)
    const int perRow = dim / 8, units = QT_ROWS * perRow;
    const unsigned magic = (0x400000u + perRow - 1) / perRow; // u / perRow = u * magic >> 22 for u < units, perRow in 1 .. 512
    for (int u0 = tid; u0 < units; u0 += 1024) {
        uint4 raw[4];
        float rm[4];
        int r[4], c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int u = u0 + k * 256, row = (int)((unsigned)u * magic >> 22);
            r[k] = u < units ? t0 + row : lenRound;
            c[k] = (u - row * perRow) * 8;
            raw[k] = r[k] < len ? *(const uint4 *)At<TBF16>(src, r[k], c[k]) : make_uint4(0, 0, 0, 0);
            rm[k] = (rowMult && r[k] < len) ? rowMult[r[k]] : 1.f;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (r[k] >= lenRound) {
                continue;
            }
            const uint32_t w[4] = {raw[k].x, raw[k].y, raw[k].z, raw[k].w};
            uint32_t packed[2] = {0, 0};
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t word = seed ? DitherWord(seed, r[k], c[k] / 4 + q) : 0u;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t v = w[q * 2 + (e >> 1)];
                    float x = __uint_as_float((e & 1) ? v & 0xffff0000u : v << 16);
                    if (rowMult) {
                        x = x * rm[k];
                    }
                    const float y = seed ? __builtin_fmaf(x, mult, DitherOffset(word, e)) : x * mult;
                    packed[q] |= (uint32_t)(CvtToI8(y) & 0xff) << (8 * e);
                }
            }
            *(uint2 *)At<TI8>(dst, r[k], c[k]) = r[k] < len ? make_uint2(packed[0], packed[1]) : make_uint2(0u, 0u);
        }
    }
}

__global__ void FillFloats(float *p, int n, float v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

// tileMax[kt] = max over the k-tile's rows of rowAbsMax[t] * |rowMult[t]|: the k-tile abs-max when the row maxima are already known
__global__ void __launch_bounds__(256) TileMaxFromRows(int len, const float *rowAbsMax, const float *rowMult, int kTile, float *tileMax)
{
    __shared__ float red[4];
    int t0 = blockIdx.x * kTile;
    float mx = 0;
    for (int t = t0 + threadIdx.x; t < t0 + kTile && t < len; t += 256) {
        float m = rowAbsMax[t];
        if (rowMult) {
            m *= fabsf(rowMult[t]);
        }
        mx = fmaxf(mx, m);
    }
    mx = WaveMax(mx);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        tileMax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
}

// abs-max of 16 raw bytes holding fp32 or bf16 values
template <class TSrc> __device__ __forceinline__ float AbsMax16(v4i raw)
{
    float m = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t w = (uint32_t)raw[e];
        if (TSrc::SIZE == 4) {
            m = fmaxf(m, fabsf(__uint_as_float(w)));
        } else {
            m = fmaxf(m, fmaxf(fabsf(__uint_as_float(w << 16)), fabsf(__uint_as_float(w & 0xffff0000u))));
        }
    }
    return m;
}

// grid (row bytes / 4096 rounded up, len/ROWS): a workgroup reduces ROWS rows x 4096 bytes with 16-byte loads, four rows in flight,
// and issues one atomic.  ROWS divides 128, hence kTile.
template <class TSrc>
__global__ void __launch_bounds__(256) TileAbsMax(int len, int dim, Mat src, const float *rowMult, int kTile, float *tileMax)
{
    constexpr int ROWS = 16;
    __shared__ float red[4];
    int tid = threadIdx.x;
    int byteCol = blockIdx.x * 4096 + tid * 16;
    int t0 = blockIdx.y * ROWS;
    float mx = 0;
    if (byteCol < dim * TSrc::SIZE) {
        for (int r = 0; r < ROWS; r += 4) {
            v4i raw[4];
            float rm[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int t = t0 + r + k;
                raw[k] = t < len ? *(const v4i *)(src.p + (int64_t)t * src.ld + byteCol) : (v4i){0, 0, 0, 0};
                rm[k] = (rowMult && t < len) ? fabsf(rowMult[t]) : 1.f;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                mx = fmaxf(mx, AbsMax16<TSrc>(raw[k]) * rm[k]);
            }
        }
    }
    mx = WaveMax(mx);
    if ((tid & 63) == 0) {
        red[tid >> 6] = mx;
    }
    __syncthreads();
    if (tid == 0) {
        mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        AtomicMaxPos(&tileMax[t0 / kTile], mx);
    }
}

// 128 (rows t) x 128 (columns x) tile.  Loads are 16 bytes per lane with four rows in flight, conversion, byte tile in LDS, then
// every thread transposes a 16 (t) x 4 (x) block with v_perm_b32 and stores 16 bytes to each of 4 destination rows; 8 neighbouring
// lanes cover the 128 bytes of one destination row.
template <class TSrc, bool QUANT>
__global__ void __launch_bounds__(256) TransposeQuant(int len, int lenRound, Mat src, const float *rowMult, const float *tileMax, int kTile,
    const int *rowIndex, Mat dst, float *tileScale, const float *rowAbsMax, uint32_t seed)
{
    constexpr int PITCH = 132;
    __shared__ __attribute__((aligned(16))) uint8_t buf[128 * PITCH];
    int tid = threadIdx.x;
    int xBlock = blockIdx.x * 128;
    int tBlock = blockIdx.y * 128;
    constexpr int SB = QUANT ? TSrc::SIZE : 1;     // source bytes per element
    constexpr int LPR = 128 * SB / 16;             // lanes per row: 8 (1-byte), 16 (bf16), 32 (fp32)
    constexpr int RPP = 256 / LPR;                 // rows per pass
    constexpr int EPL = 16 / SB;                   // elements per lane
    const int lr = tid / LPR, lc = tid % LPR;
    float mult = 0, tm = 0;
    if (QUANT) {
        if (rowAbsMax) {
            // the k-tile's abs-max from the row maxima (max over its rows of rowAbsMax[t] * |rowMult[t]|), as TileMaxFromRows forms it
            __shared__ float redT[4];
            const int k0 = (tBlock / kTile) * kTile;
            float mx = 0;
            for (int t = k0 + tid; t < k0 + kTile && t < len; t += 256) {
                const int sr = rowIndex ? rowIndex[t] : t; // (a gathered tile: the maxima of the rows that land in it)
                if (sr < 0) {
                    continue;
                }
                float m = rowAbsMax[sr];
                if (rowMult) {
                    m *= fabsf(rowMult[sr]);
                }
                mx = fmaxf(mx, m);
            }
            mx = WaveMax(mx);
            if ((tid & 63) == 0) {
                redT[tid >> 6] = mx;
            }
            __syncthreads();
            tm = fmaxf(fmaxf(redT[0], redT[1]), fmaxf(redT[2], redT[3]));
        } else {
            tm = tileMax[tBlock / kTile];            // one 128-row block lies inside one k-tile (kTile is a multiple of 128)
        }
        mult = tm > 0 ? 1 / (tm / 127) : 0.f;        // same two roundings as scale = max/127, mult = 1/scale
    }
    for (int r0 = 0; r0 < 128; r0 += RPP * 4) {
        v4i raw[4];
        float rm[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int r = r0 + k * RPP + lr;
            int t = tBlock + r;
            raw[k] = (v4i){0, 0, 0, 0};
            rm[k] = 0;
            if (t < len) {
                int srcRow = rowIndex ? rowIndex[t] : t;
                if (srcRow >= 0) {
                    raw[k] = *(const v4i *)(src.p + (int64_t)srcRow * src.ld + (int64_t)(xBlock + lc * EPL) * SB);
                    rm[k] = (QUANT && rowMult) ? rowMult[srcRow] : 1.f;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int r = r0 + k * RPP + lr;
            uint8_t *d = buf + r * PITCH + lc * EPL;
            if (!QUANT) {
                *(uint32_t *)d = (uint32_t)raw[k][0];
                *(uint32_t *)(d + 4) = (uint32_t)raw[k][1];
                *(uint32_t *)(d + 8) = (uint32_t)raw[k][2];
                *(uint32_t *)(d + 12) = (uint32_t)raw[k][3];
            } else {
                float f[EPL];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t w = (uint32_t)raw[k][e];
                    if (SB == 4) {
                        f[e] = __uint_as_float(w);
                    } else {
                        f[(2 * e) % EPL] = __uint_as_float(w << 16);
                        f[(2 * e + 1) % EPL] = __uint_as_float(w & 0xffff0000u);
                    }
                }
                uint32_t packed[EPL / 4];
#pragma unroll
                for (int q = 0; q < EPL / 4; ++q) {
                    packed[q] = 0;
                    // (the dither's row is the position in the contraction, its column the gradient's)
                    const uint32_t word = seed ? DitherWord(seed, tBlock + r, (xBlock + lc * EPL) / 4 + q) : 0u;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float x = f[q * 4 + e];
                        if (rowMult) {
                            x = x * rm[k];
                        }
                        const float y = seed ? __builtin_fmaf(x, mult, DitherOffset(word, e)) : x * mult;
                        packed[q] |= (uint32_t)(CvtToI8(y) & 0xff) << (8 * e);
                    }
                }
                *(uint32_t *)d = packed[0];
                if (EPL == 8) {
                    *(uint32_t *)(d + 4) = packed[EPL / 4 - 1];
                }
            }
        }
    }
    __syncthreads();
    TransposeOut128<PITCH>(buf, dst, xBlock, tBlock, tid);
    if (QUANT && tileScale && blockIdx.x == 0 && tid == 0) {
        tileScale[tBlock / kTile] = tm > 0 ? tm / 127 : 1.f;
    }
}


// dst_i = src_i^T for up to TRANSPOSE_JOBS byte matrices in one launch (dimensions multiples of 128; a workgroup per 128x128 tile):
// after an update every matrix of a model is transposed again (28 of a 512-wide model: 123 -> 8.7 us)
constexpr int TRANSPOSE_JOBS = 32;
struct TransposeJobs {
    Mat src[TRANSPOSE_JOBS], dst[TRANSPOSE_JOBS];
    int tilesX[TRANSPOSE_JOBS], first[TRANSPOSE_JOBS + 1]; // column tiles of src; tiles before the job
};

__global__ void __launch_bounds__(256) TransposeBytes(int count, TransposeJobs jobs)
{
    constexpr int PITCH = 132;
    __shared__ __attribute__((aligned(16))) uint8_t buf[128 * PITCH];
    int j = 0;
    while (j + 1 < count && (int)blockIdx.x >= jobs.first[j + 1]) {
        ++j;
    }
    const int tile = blockIdx.x - jobs.first[j], xBlock = tile % jobs.tilesX[j] * 128, tBlock = tile / jobs.tilesX[j] * 128;
    const Mat src = jobs.src[j];
    const int tid = threadIdx.x, lr = tid >> 3, lc = tid & 7;
    v4i raw[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        raw[k] = *(const v4i *)(src.p + (int64_t)(tBlock + k * 32 + lr) * src.ld + xBlock + lc * 16);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t *d = (uint32_t *)(buf + (k * 32 + lr) * PITCH + lc * 16);
        d[0] = (uint32_t)raw[k][0];
        d[1] = (uint32_t)raw[k][1];
        d[2] = (uint32_t)raw[k][2];
        d[3] = (uint32_t)raw[k][3];
    }
    __syncthreads();
    TransposeOut128<PITCH>(buf, jobs.dst[j], xBlock, tBlock, tid);
}

template <class TSrc>
__global__ void __launch_bounds__(256) RowTileNormalizeRope(int len, int lenRound, int tiles, Mat src, float srcMult, int normalize, float vecScale,
    Mat rope, Mat dst, Mat tileScale)
{
    int t0, tile, h;
    if (!Unit(lenRound, tiles, &t0, &tile, &h)) {
        return;
    }
    int col = tile * TILE + h * 4;
    F4 v[U], rp[U];
    float discr[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        bool live = t0 + k < len;
        v[k] = live ? Load4<TSrc>(At<TSrc>(src, t0 + k, col)) : ZeroF4();
        rp[k] = (live && rope.p) ? Load4<TF32>(At<TF32>(rope, t0 + k, h * 4)) : ZeroF4();
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        discr[k] = 0;
        if (t0 + k >= lenRound) {
            continue;
        }
        F4 x = v[k] * srcMult;
        if (t0 + k < len) {
            if (normalize) {
                float sum2 = Half32Sum(HSum(x * x));
                if (sum2 > 0) {
                    discr[k] = sqrtf(sum2 / TILE) * vecScale;
                    x = x * (1 / discr[k]);
                }
            }
            if (rope.p) {
                x = ApplyRope4(x, rp[k], 1.f);
            }
        }
        Store4<TBF16>(At<TBF16>(dst, t0 + k, col), x);
    }
    if (normalize) {
        StoreScales(tileScale, tile, t0, lenRound, h, discr);
    }
}

// blockIdx.y = job: the gradients of Q, K and V go in one launch (4096 x 512, e4m3: 3 x 4.4 -> 7.7 us; 16384 x 384, bf16: 3 x 9.8 -> 24.3).
// N = 1: one gradient, its description in scalar registers from the start (16384 x 512, bf16: 15.1 us, 15.4 through the table)
template <int N> struct NormRopeJobs {
    Mat grad[N], srcNorm[N], srcTileScale[N], rope[N], dst[N];
};

template <class TGrad, class TDst, int N>
__global__ void __launch_bounds__(256) BackpropRowTileNormalizeRope(int len, int lenRound, int tiles, float gradMult, NormRopeJobs<N> jobs)
{
    const int j = N == 1 ? 0 : blockIdx.y;
    const Mat grad = jobs.grad[j], srcNorm = jobs.srcNorm[j], srcTileScale = jobs.srcTileScale[j], rope = jobs.rope[j], dst = jobs.dst[j];
    int t0, tile, h;
    if (!Unit(lenRound, tiles, &t0, &tile, &h)) {
        return;
    }
    int col = tile * TILE + h * 4;
    F4 g[U], sn[U], rp[U];
    float sc[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        int t = t0 + k;
        bool live = t < len;
        g[k] = live ? Load4<TGrad>(At<TGrad>(grad, t, col)) : ZeroF4();
        sn[k] = (live && srcNorm.p) ? Load4<TBF16>(At<TBF16>(srcNorm, t, col)) : ZeroF4();
        sc[k] = (live && srcNorm.p) ? ScaleAt(srcTileScale, tile, t) : 0.f;
        rp[k] = (live && rope.p) ? Load4<TF32>(At<TF32>(rope, t, h * 4)) : ZeroF4();
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        int t = t0 + k;
        if (t >= lenRound) {
            continue;
        }
        F4 x = g[k] * gradMult;
        if (t < len) {
            if (srcNorm.p) {
                x = TileNormBackprop(sn[k] * sc[k], x);
            }
            if (rope.p) {
                x = ApplyRope4(x, rp[k], -1.f);
            }
        }
        Store4<TDst>(At<TDst>(dst, t, col), x);
    }
}

// bf16 gradient -> e4m3 with eight elements per lane (a tile = 16 lanes, the tile sums are four DPP steps, the rotated pairs sit in
// one lane): the form the model's attention backward uses.  Same arithmetic per element as BackpropRowTileNormalizeRope.
template <int N>
__global__ void __launch_bounds__(256) BackpropRowTileNormalizeRope8(int len, int lenRound, int tiles, float gradMult, NormRopeJobs<N> jobs)
{
    const int j = N == 1 ? 0 : blockIdx.y;
    const Mat grad = jobs.grad[j], srcNorm = jobs.srcNorm[j], srcTileScale = jobs.srcTileScale[j], rope = jobs.rope[j], dst = jobs.dst[j];
    constexpr int UU = 2;
    const int l16 = threadIdx.x & 15;
    const long unit0 = ((long)blockIdx.x * 256 + threadIdx.x) >> 4;
    const long units = (long)lenRound * tiles;
    const long stride = ((long)gridDim.x * 256) >> 4;
    uint4 g[UU], sn[UU];
    F4 rp[UU][2];
    float sc[UU];
    int row[UU], col[UU];
    bool any[UU], live[UU];
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        long u = unit0 + k * stride;
        any[k] = u < units;
        row[k] = any[k] ? (int)(u / tiles) : 0;
        int tile = any[k] ? (int)(u - (long)row[k] * tiles) : 0;
        col[k] = tile * TILE + l16 * 8;
        live[k] = any[k] && row[k] < len;
        g[k] = live[k] ? *(const uint4 *)At<TBF16>(grad, row[k], col[k]) : make_uint4(0, 0, 0, 0);
        sn[k] = (live[k] && srcNorm.p) ? *(const uint4 *)At<TBF16>(srcNorm, row[k], col[k]) : make_uint4(0, 0, 0, 0);
        sc[k] = (live[k] && srcNorm.p) ? ScaleAt(srcTileScale, tile, row[k]) : 0.f;
        rp[k][0] = (live[k] && rope.p) ? Load4<TF32>(At<TF32>(rope, row[k], l16 * 8)) : ZeroF4();
        rp[k][1] = (live[k] && rope.p) ? Load4<TF32>(At<TF32>(rope, row[k], l16 * 8 + 4)) : ZeroF4();
    }
#pragma unroll
    for (int k = 0; k < UU; ++k) {
        const uint32_t gw[4] = {g[k].x, g[k].y, g[k].z, g[k].w}, sw[4] = {sn[k].x, sn[k].y, sn[k].z, sn[k].w};
        float x[8], src[8];
        float sum2 = 0, dp = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float ge = (e & 1) ? __uint_as_float(gw[e >> 1] & 0xffff0000u) : __uint_as_float(gw[e >> 1] << 16);
            float se = (e & 1) ? __uint_as_float(sw[e >> 1] & 0xffff0000u) : __uint_as_float(sw[e >> 1] << 16);
            x[e] = ge * gradMult;
            src[e] = se * sc[k];
            sum2 += src[e] * src[e];
            dp += src[e] * x[e];
        }
        if (srcNorm.p) { // uniform
            sum2 = Row16Sum(sum2);
            dp = Row16Sum(dp);
        }
        if (!any[k]) {
            continue;
        }
        uint32_t out[2] = {0, 0};
        if (live[k]) {
            if (srcNorm.p) {
                float sigma = 0, scale = 0;
                if (sum2 != 0) {
                    float inv = 1 / sum2;
                    sigma = dp * inv;
                    scale = sqrtf(TILE * inv);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = sum2 != 0 ? (x[e] - src[e] * sigma) * scale : 0.f;
                }
            }
            if (rope.p) {
                F4 lo = ApplyRope4(MakeF4(x[0], x[1], x[2], x[3]), rp[k][0], -1.f);
                F4 hi = ApplyRope4(MakeF4(x[4], x[5], x[6], x[7]), rp[k][1], -1.f);
                x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
                x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
            }
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                out[w >> 1] |= CvtPkE4m3(x[2 * w], x[2 * w + 1]) << ((w & 1) * 16);
            }
        }
        *(uint2 *)At<TE4M3>(dst, row[k], col[k]) = make_uint2(out[0], out[1]);
    }
}

// sum of `splits` fp32 partial products (slabs of [rows][cols]) -> packed delta: per row and 128-column tile scale = maxabs/127,
// bytes = sat_i8(rne(v/scale)), TileScale[tile][row] = scale: the arithmetic of the GEMM's ROW_TILE_MAXNORM epilogue applied to the sum.
//
// Bounded by latency: one slice after the other is one trip to memory each.  So RU rows times SU slices are requested together (the sum keeps
// the order of the slices, and its bits).  Against four rows of one slice at a time: 512 x 512 of 8 slices 6.0 -> 3.2 us, 1024 x 512 of 32
// 30.6 -> 12.0, 1024 x 1024 of 8 7.5 -> 4.3, 256 x 256 of one 3.5 -> 2.8; 8192 x 2048 of 2 28.8 -> 23.9.
template <int RU, int SU>
__global__ void __launch_bounds__(256) PackDelta(int rows, int tiles, int splits, const uint8_t *partial, int64_t ldPartial, int64_t slab, float alpha,
    const float *alphaPtr, Mat delta, Mat tileScale)
{
    const long u = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 5;
    const int h = threadIdx.x & 31, tile = (int)(u % tiles), t0 = (int)(u / tiles) * RU;
    if (t0 >= rows) {
        return;
    }
    float scale = alpha;
    if (alphaPtr) {
        scale *= *alphaPtr;
    }
    const int col = tile * TILE + h * 4;
    const uint8_t *src = partial + (int64_t)t0 * ldPartial + (int64_t)col * 4;
    F4 v[RU];
#pragma unroll
    for (int k = 0; k < RU; ++k) {
        v[k] = ZeroF4();
    }
    for (int s0 = 0; s0 < splits; s0 += SU) {
        F4 x[SU][RU];
#pragma unroll
        for (int j = 0; j < SU; ++j) {
#pragma unroll
            for (int k = 0; k < RU; ++k) {
                x[j][k] = s0 + j < splits && t0 + k < rows ? Load4<TF32>(src + (int64_t)(s0 + j) * slab + k * ldPartial) : ZeroF4();
            }
        }
#pragma unroll
        for (int j = 0; j < SU; ++j) {
            if (s0 + j < splits) {
#pragma unroll
                for (int k = 0; k < RU; ++k) {
                    v[k] = v[k] + x[j][k];
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < RU; ++k) {
        const float mx = Half32Max(HMaxAbs(v[k])) * fabsf(scale);
        float discr = 0, mult = 0;
        if (mx > 0) {
            discr = mx / 127;
            mult = 1 / discr;
        }
        if (t0 + k < rows) {
            Store4<TI8>(At<TI8>(delta, t0 + k, col), v[k] * scale * mult);
            if (h == 0) {
                ScaleAt(tileScale, tile, t0 + k) = discr;
            }
        }
    }
}

bool MatOk(const ts2_mat *m, int rows, int cols, int elemSize)
{
    return m && m->ptr && m->y >= rows && m->x >= cols && (m->strideBytes % 4) == 0 && m->strideBytes >= (int64_t)cols * elemSize;
}

int ElemSize(int type)
{
    switch (type) {
    case TS2_F32:
    case TS2_I32:
        return 4;
    case TS2_BF16:
        return 2;
    default:
        return 1;
    }
}
} // namespace

#define STREAM ((hipStream_t)stream)

extern "C" int ts2_layer_normalize_state_vecs(const ts2_mat *state, int32_t stateType, int32_t len, int32_t lenRound, float vecScale,
    const ts2_mat *normState, int32_t normType, const ts2_mat *normStateScale, void *stream)
{
    if (!state || !normState || !normStateScale) {
        return TS2_ERR_NULL;
    }
    int dim = state->x;
    if (dim % TILE || lenRound < len || !MatOk(state, len, dim, ElemSize(stateType)) || !MatOk(normState, lenRound, dim, ElemSize(normType)) ||
        !MatOk(normStateScale, dim / TILE, lenRound, 4)) {
        return TS2_ERR_SHAPE;
    }
    int tiles = dim / TILE;
    TS2_DISPATCH_TYPE(stateType, TS, TS2_DISPATCH_TYPE(normType, TD,
        hipLaunchKernelGGL((LayerNormalizeStateVecs<TS, TD>), GridFor(lenRound, tiles), dim3(256), 0, STREAM, len, lenRound, tiles, vecScale,
            M(*state), M(*normState), M(*normStateScale))));
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

static int BackpropNormImpl(bool final, int len, int rows, const ts2_mat *normState, int normType, const ts2_mat *stateScale,
    const ts2_mat *dNormState, const float *combinerScale, const float *gradScale, const float *gradMult, const ts2_mat *stateGrad,
    const ts2_mat *stateGradFast, int fastType, float *nextMaxNorm, void *stream)
{
    if (!normState || !stateScale || !dNormState || !stateGrad || !stateGradFast) {
        return TS2_ERR_NULL;
    }
    int dim = dNormState->x;
    if (dim % TILE || !MatOk(normState, len, dim, ElemSize(normType)) || !MatOk(stateScale, dim / TILE, len, 4) ||
        !MatOk(dNormState, len, dim, 4) || !MatOk(stateGrad, rows, dim, 4) || !MatOk(stateGradFast, rows, dim, ElemSize(fastType))) {
        return TS2_ERR_SHAPE;
    }
    if (normType == TS2_F32 || (fastType != TS2_BF16 && fastType != TS2_E4M3)) {
        return TS2_ERR_UNSUPPORTED;
    }
    int tiles = dim / TILE;
    // One update of the maximum per workgroup, 10 ns each on its one address: 1024 threads each, two workgroups per CU, once there are more than
    // 100 (e4m3) or 256 workgroups of 256 and until many times as much work outweighs the queue and small workgroups share the memory better.
    // This pass and the final one, workgroups of 256 -> of 1024, us: e4m3 200 x 1024 3.5, 3.3 -> 3.6, 3.3; 500 x 512 3.8, 3.5 -> 3.6, 3.3;
    // 1024 x 512 5.4, 5.3 -> 4.1, 3.7; 4096 x 512 15.7, 15.7 -> 7.5, 7.1; 16384 x 1024 103, 101 -> 44.2, 33.4; 16384 x 2048 117, 107 -> 92.4,
    // 68.8; 65536 x 1024, both together, 305 -> 350; int8 1024 x 512 5.7, 5.4 -> 6.2, 5.8; 4096 x 1024 51.4, 50.8 -> 13.2, 11.2; 16384 x 2048
    // 104, 92.2 -> 102, 79.7.  The widest int8 passes, 2048 -> 4096 workgroups, 32768 x 2048: 197, 169 -> 202, 154
    const long units4 = (long)((rows + U - 1) / U) * tiles, units1 = (long)rows * tiles;
    auto grid = [](long units, int perBlock, int most) { const long n = (units + perBlock - 1) / perBlock; return dim3((unsigned)(n < most ? n : most)); };
    if (normType == TS2_E4M3 && fastType == TS2_E4M3 && (((uintptr_t)normState->ptr | normState->strideBytes | (uintptr_t)stateGradFast->ptr |
                                                         stateGradFast->strideBytes) & 7) == 0 &&
        Aligned16(dNormState->ptr, dNormState->strideBytes) && Aligned16(stateGrad->ptr, stateGrad->strideBytes)) {
#define LAUNCH_BN8(FINAL, NT)                                                                                                              \
    hipLaunchKernelGGL((BackpropLayerNormalize8<FINAL, NT>), grid(units1, NT / 16, NT == 256 ? 8192 : 512), dim3(NT), 0, STREAM, len, rows, tiles, M(*normState), \
        M(*stateScale), M(*dNormState), combinerScale, gradScale, gradMult, M(*stateGrad), M(*stateGradFast), nextMaxNorm)
        const bool many = units1 > 1600 && units1 <= 262144;
        if (final) {
            if (many) {
                LAUNCH_BN8(true, 1024);
            } else {
                LAUNCH_BN8(true, 256);
            }
        } else {
            if (many) {
                LAUNCH_BN8(false, 1024);
            } else {
                LAUNCH_BN8(false, 256);
            }
        }
#undef LAUNCH_BN8
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
#define LAUNCH_BN_AS(TN, TFA, FINAL, NT)                                                                                                   \
    hipLaunchKernelGGL((BackpropLayerNormalize<TN, TFA, FINAL, NT>), grid(units4, NT / 32, NT == 256 ? (FINAL ? 4096 : 2048) : 512), dim3(NT), 0, STREAM, len, rows, tiles,    \
        M(*normState), M(*stateScale), M(*dNormState), combinerScale, gradScale, gradMult, M(*stateGrad), M(*stateGradFast), nextMaxNorm)
#define LAUNCH_BN(TN, TFA)                                                                                                                 \
    if (units4 <= 2048 || units4 > 65536) {                                                                                                               \
        if (final) {                                                                                                                       \
            LAUNCH_BN_AS(TN, TFA, true, 256);                                                                                              \
        } else {                                                                                                                           \
            LAUNCH_BN_AS(TN, TFA, false, 256);                                                                                             \
        }                                                                                                                                  \
    } else if (final) {                                                                                                                    \
        LAUNCH_BN_AS(TN, TFA, true, 1024);                                                                                                 \
    } else {                                                                                                                               \
        LAUNCH_BN_AS(TN, TFA, false, 1024);                                                                                                \
    }
    if (fastType == TS2_BF16) {
        TS2_DISPATCH_TYPE(normType, TN, LAUNCH_BN(TN, TBF16));
    } else {
        TS2_DISPATCH_TYPE(normType, TN, LAUNCH_BN(TN, TE4M3));
    }
#undef LAUNCH_BN
#undef LAUNCH_BN_AS
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_backprop_layer_normalize(const ts2_mat *normState, int32_t normType, const ts2_mat *stateScale, const ts2_mat *dNormState,
    const float *combinerScale, const float *gradScale, const float *gradMult, const ts2_mat *stateGrad, const ts2_mat *stateGradFast,
    int32_t fastType, float *nextLayerGradMaxNorm, int32_t len, void *stream)
{
    return BackpropNormImpl(false, len, len, normState, normType, stateScale, dNormState, combinerScale, gradScale, gradMult, stateGrad,
        stateGradFast, fastType, nextLayerGradMaxNorm, stream);
}

extern "C" int ts2_backprop_final_normalize(int32_t len, int32_t lenRound, const ts2_mat *normState, int32_t normType, const ts2_mat *stateScale,
    const ts2_mat *dNormState, const ts2_mat *stateGrad, const ts2_mat *stateGradFast, int32_t fastType, float *nextLayerGradMaxNorm,
    void *stream)
{
    return BackpropNormImpl(true, len, lenRound, normState, normType, stateScale, dNormState, nullptr, nullptr, nullptr, stateGrad, stateGradFast,
        fastType, nextLayerGradMaxNorm, stream);
}

extern "C" int ts2_scale_grad(const float *gradMaxNorm, const float *prevGradMult, const ts2_mat *grad, const ts2_mat *gradFast, int32_t fastType,
    int32_t len, float *gradScaleOut, float *gradMultOut, void *stream)
{
    if (!gradMaxNorm || !grad || !gradFast) {
        return TS2_ERR_NULL;
    }
    int dim = grad->x;
    if (dim % TILE || !MatOk(grad, len, dim, 4) || !MatOk(gradFast, len, dim, ElemSize(fastType))) {
        return TS2_ERR_SHAPE;
    }
    int tiles = dim / TILE;
    auto reads = [&](const float *p) { return p && (p == gradMaxNorm || p == prevGradMult); };
    const bool later = reads(gradScaleOut) || reads(gradMultOut);
    float *scaleNow = later ? nullptr : gradScaleOut, *multNow = later ? nullptr : gradMultOut;
    if (fastType == TS2_BF16) {
        hipLaunchKernelGGL((ScaleGrad<TBF16, false>), GridFor(len, tiles), dim3(256), 0, STREAM, len, tiles, gradMaxNorm, prevGradMult, M(*grad),
            M(*gradFast), scaleNow, multNow, RowQuantOut{});
    } else if (fastType == TS2_E4M3) {
        hipLaunchKernelGGL((ScaleGrad<TE4M3, false>), GridFor(len, tiles), dim3(256), 0, STREAM, len, tiles, gradMaxNorm, prevGradMult, M(*grad),
            M(*gradFast), scaleNow, multNow, RowQuantOut{});
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    if (!later) {
        return TS2_OK;
    }
    hipLaunchKernelGGL(PublishGradMult, dim3(1), dim3(1), 0, STREAM, gradMaxNorm, gradScaleOut, gradMultOut);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_matrix_lolu(int32_t len, int32_t lenRound, const ts2_mat *gate, const ts2_mat *vals, float resMult, const ts2_mat *res,
    int32_t resType, void *stream)
{
    if (!gate || !vals || !res) {
        return TS2_ERR_NULL;
    }
    int dim = res->x;
    if (dim % TILE || !MatOk(gate, len, dim, 2) || !MatOk(vals, len, dim, 2) || !MatOk(res, lenRound, dim, ElemSize(resType))) {
        return TS2_ERR_SHAPE;
    }
    int tiles = dim / TILE;
    if (resType == TS2_E4M3 && Aligned16(gate->ptr, gate->strideBytes) && Aligned16(vals->ptr, vals->strideBytes) &&
        Aligned16(res->ptr, res->strideBytes)) {
        const long lanes = (long)lenRound * (dim / 16);
        hipLaunchKernelGGL(MatrixLoLU16, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, STREAM, len, lenRound, dim / 16, M(*gate), M(*vals),
            resMult, M(*res));
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
    if (resType == TS2_E4M3 && Aligned16(gate->ptr, gate->strideBytes) && Aligned16(vals->ptr, vals->strideBytes) &&
        (((uintptr_t)res->ptr | res->strideBytes) & 7) == 0) {
        const long lanes = ((long)lenRound * (dim / 8) + 1) / 2;
        hipLaunchKernelGGL(MatrixLoLU8, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, STREAM, len, lenRound, dim / 8, M(*gate), M(*vals),
            resMult, M(*res));
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
    TS2_DISPATCH_TYPE(resType, TD,
        hipLaunchKernelGGL((MatrixLoLU<TD>), GridFor(lenRound, tiles), dim3(256), 0, STREAM, len, lenRound, tiles, M(*gate), M(*vals), resMult,
            M(*res)));
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

template <int MODE>
static int BackpropLoluImpl(int len, int lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale, const ts2_mat *tileScale,
    const ts2_mat *grad, int gradType, const ts2_mat *gradGate, int ggType, const ts2_mat *gradVals, int gvType, const ts2_mat *dScale, void *stream)
{
    if (!gate || !vals || !grad || !gradGate || !gradVals || (MODE == 0 ? !tileScale : !dScale)) {
        return TS2_ERR_NULL;
    }
    int dim = grad->x;
    if (dim % TILE || !MatOk(gate, len, dim, 2) || !MatOk(vals, len, dim, 2) || !MatOk(grad, len, dim, ElemSize(gradType)) ||
        !MatOk(gradGate, lenRound, dim, ElemSize(ggType)) || !MatOk(gradVals, lenRound, dim, ElemSize(gvType))) {
        return TS2_ERR_SHAPE;
    }
    if (MODE == 0 ? !MatOk(tileScale, dim / TILE, len, 4) : !MatOk(dScale, dim / TILE, lenRound, 4)) {
        return TS2_ERR_SHAPE;
    }
    int tiles = dim / TILE;
    Mat ts = MODE == 0 ? M(*tileScale) : Mat{nullptr, 0};
    Mat ds = MODE == 1 ? M(*dScale) : Mat{nullptr, 0};
    if ((gradType != TS2_BF16 && gradType != TS2_F32) || (ggType != TS2_BF16 && ggType != TS2_E4M3) || (gvType != TS2_BF16 && gvType != TS2_E4M3)) {
        return TS2_ERR_UNSUPPORTED;
    }
    if (MODE == 0 && gradType == TS2_BF16 && ggType == TS2_E4M3 && gvType == TS2_E4M3 && Aligned16(gate->ptr, gate->strideBytes) &&
        Aligned16(vals->ptr, vals->strideBytes) && Aligned16(grad->ptr, grad->strideBytes) &&
        (((uintptr_t)gradGate->ptr | gradGate->strideBytes | (uintptr_t)gradVals->ptr | gradVals->strideBytes) & 7) == 0) {
        const long lanes = ((long)lenRound * tiles * 16 + 1) / 2;
        hipLaunchKernelGGL(BackpropLoLU8, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, STREAM, len, lenRound, tiles, M(*gate), M(*vals), valsScale,
            ts, M(*grad), M(*gradGate), M(*gradVals));
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
    if (MODE == 1 && gradType == TS2_BF16 && ggType == TS2_E4M3 && gvType == TS2_BF16 && Aligned16(gate->ptr, gate->strideBytes) &&
        Aligned16(vals->ptr, vals->strideBytes) && Aligned16(grad->ptr, grad->strideBytes) && Aligned16(gradVals->ptr, gradVals->strideBytes) &&
        (((uintptr_t)gradGate->ptr | gradGate->strideBytes) & 7) == 0) {
        const long lanes = ((long)lenRound * tiles * 16 + 1) / 2;
        hipLaunchKernelGGL(BackpropLoLUAtt8, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, STREAM, len, lenRound, tiles, M(*gate), M(*vals),
            valsScale, M(*grad), M(*gradGate), M(*gradVals), ds);
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
#define LAUNCH_BL(TG, TOG, TOV)                                                                                                            \
    hipLaunchKernelGGL((BackpropLoLU<TG, TOG, TOV, MODE>), GridFor(lenRound, tiles), dim3(256), 0, STREAM, len, lenRound, tiles, M(*gate),  \
        M(*vals), valsScale, ts, M(*grad), M(*gradGate), M(*gradVals), ds)
    if (gradType == TS2_BF16) {
        if (ggType == TS2_BF16 && gvType == TS2_BF16) {
            LAUNCH_BL(TBF16, TBF16, TBF16);
        } else if (ggType == TS2_E4M3 && gvType == TS2_E4M3) {
            LAUNCH_BL(TBF16, TE4M3, TE4M3);
        } else if (ggType == TS2_E4M3 && gvType == TS2_BF16) {
            LAUNCH_BL(TBF16, TE4M3, TBF16);
        } else {
            return TS2_ERR_UNSUPPORTED;
        }
    } else {
        if (ggType == TS2_BF16 && gvType == TS2_BF16) {
            LAUNCH_BL(TF32, TBF16, TBF16);
        } else if (ggType == TS2_E4M3 && gvType == TS2_E4M3) {
            LAUNCH_BL(TF32, TE4M3, TE4M3);
        } else if (ggType == TS2_E4M3 && gvType == TS2_BF16) {
            LAUNCH_BL(TF32, TE4M3, TBF16);
        } else {
            return TS2_ERR_UNSUPPORTED;
        }
    }
#undef LAUNCH_BL
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_backprop_row_tile_normalize_lolu(int32_t len, int32_t lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale,
    const ts2_mat *valsSrcTileScale, const ts2_mat *grad, int32_t gradType, const ts2_mat *gradGate, const ts2_mat *gradVals,
    int32_t gradOutType, void *stream)
{
    return BackpropLoluImpl<0>(len, lenRound, gate, vals, valsScale, valsSrcTileScale, grad, gradType, gradGate, gradOutType, gradVals,
        gradOutType, nullptr, stream);
}

extern "C" int ts2_backprop_lolu_dscale(int32_t len, int32_t lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale,
    const ts2_mat *grad, int32_t gradType, const ts2_mat *gradGate, int32_t gradGateType, const ts2_mat *gradVals, int32_t gradValsType,
    const ts2_mat *dScale, void *stream)
{
    return BackpropLoluImpl<1>(len, lenRound, gate, vals, valsScale, nullptr, grad, gradType, gradGate, gradGateType, gradVals, gradValsType,
        dScale, stream);
}

extern "C" int ts2_tile_max_from_rows(int32_t len, const float *rowAbsMax, const float *rowMult, int32_t kTile, float *tileMax, void *stream)
{
    if (!rowAbsMax || !tileMax) {
        return TS2_ERR_NULL;
    }
    if (kTile <= 0 || kTile % 128 || len <= 0) {
        return TS2_ERR_SHAPE;
    }
    hipLaunchKernelGGL(TileMaxFromRows, dim3((len + kTile - 1) / kTile), dim3(256), 0, STREAM, len, rowAbsMax, rowMult, kTile, tileMax);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_normalize_vecs_row_max_dither(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *colScale,
    const ts2_mat *dst, float *rowScale, float *rowAbsMax, uint32_t ditherSeed, void *stream);

extern "C" int ts2_normalize_vecs_row_max2(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *colScale,
    const ts2_mat *dst, float *rowScale, float *rowAbsMax, void *stream)
{
    return ts2_normalize_vecs_row_max_dither(len, lenRound, src, srcType, colScale, dst, rowScale, rowAbsMax, 0, stream);
}

extern "C" int ts2_normalize_vecs_row_max(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *colScale,
    const ts2_mat *dst, float *rowScale, void *stream)
{
    return ts2_normalize_vecs_row_max2(len, lenRound, src, srcType, colScale, dst, rowScale, nullptr, stream);
}

// (column scales: one source only)
static int LaunchRowQuant(int count, int len, int lenRound, int dim, const RowQuantJobs &jobs, const float *colScale, void *stream)
{
    // with column scales a wave walks several rows (the scales stay in registers), else one row per wave
    const int wgs = (lenRound + 3) / 4;
    const dim3 grid(colScale && wgs > 2048 ? 2048 : wgs, count);
#define LAUNCH_RW(N)                                                                                                                       \
    if (count == 1 && dim == N * 512) {                                                                                                    \
        hipLaunchKernelGGL((NormalizeRowsWave<N, true>), grid, dim3(256), 0, STREAM, len, lenRound, dim, jobs.src[0], colScale, jobs.dst[0], jobs.rowScale[0], jobs.rowAbsMax[0], jobs.seed[0]); \
    } else if (count == 1) {                                                                                                               \
        hipLaunchKernelGGL((NormalizeRowsWave<N, false>), grid, dim3(256), 0, STREAM, len, lenRound, dim, jobs.src[0], colScale, jobs.dst[0], jobs.rowScale[0], jobs.rowAbsMax[0], jobs.seed[0]); \
    } else if (dim == N * 512) {                                                                                                           \
        hipLaunchKernelGGL((NormalizeRowsWaveBatch<N, true>), grid, dim3(256), 0, STREAM, len, lenRound, dim, jobs);                       \
    } else {                                                                                                                               \
        hipLaunchKernelGGL((NormalizeRowsWaveBatch<N, false>), grid, dim3(256), 0, STREAM, len, lenRound, dim, jobs);                      \
    }
    switch ((dim + 511) / 512) {
    case 1: LAUNCH_RW(1); break;
    case 2: LAUNCH_RW(2); break;
    case 3: LAUNCH_RW(3); break;
    case 4: LAUNCH_RW(4); break;
    case 5: LAUNCH_RW(5); break;
    case 6: LAUNCH_RW(6); break;
    case 7: LAUNCH_RW(7); break;
    default: LAUNCH_RW(8); break;
    }
#undef LAUNCH_RW
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

// The row quantiser over `count` bf16 gradients of one shape.  Rows of dst 8-byte, of src 16-byte aligned; widths up to 4096
int Ts2QuantRowsBatch(int count, int len, int lenRound, const ts2_mat *src, const ts2_mat *dst, float *const *rowScale, float *const *rowAbsMax,
    const uint32_t *seed, void *stream)
{
    if (count < 1 || count > 4 || dst[0].x % 8 || dst[0].x > 4096 || lenRound < len) {
        return TS2_ERR_SHAPE;
    }
    RowQuantJobs jobs = {};
    for (int i = 0; i < count; ++i) {
        if (dst[i].x != dst[0].x || !MatOk(&src[i], len, dst[0].x, 2) || !MatOk(&dst[i], lenRound, dst[0].x, 1)) {
            return TS2_ERR_SHAPE;
        }
        if (!Aligned16(src[i].ptr, src[i].strideBytes) || (((uintptr_t)dst[i].ptr | dst[i].strideBytes) & 7)) {
            return TS2_ERR_ALIGN;
        }
        jobs.src[i] = M(src[i]);
        jobs.dst[i] = M(dst[i]);
        jobs.rowScale[i] = rowScale[i];
        jobs.rowAbsMax[i] = rowAbsMax[i];
        jobs.seed[i] = seed[i];
    }
    return LaunchRowQuant(count, len, lenRound, dst[0].x, jobs, nullptr, stream);
}

#define LAUNCH_ROW_CHUNKS(K, ...)                                                                                                          \
    switch ((dim + 511) / 512) {                                                                                                           \
    case 1: { constexpr int N = 1; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                            \
    case 2: { constexpr int N = 2; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                            \
    case 3: { constexpr int N = 3; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                            \
    case 4: { constexpr int N = 4; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                            \
    case 5: case 6: { constexpr int N = 6; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                    \
    default: { constexpr int N = 8; hipLaunchKernelGGL(K, __VA_ARGS__); } break;                                                           \
    }

static bool RowQuantOk(const RowQuantOut &q, int dim)
{
    return q.dst && q.rowScale && q.dstStride >= dim && (((uintptr_t)q.dst | (uintptr_t)q.dstStride) & 7) == 0;
}

int Ts2BackpropLoluRows(int mode, int len, int lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale, const ts2_mat *valsSrcTileScale,
    const ts2_mat *grad, const ts2_mat *gradGate, const ts2_mat *gradVals, const ts2_mat *dScale, const RowQuantOut &qGate, const RowQuantOut &qVals,
    void *stream)
{
    const int dim = gradGate->x;
    if (dim % TILE || dim > 4096 || lenRound <= 0 || lenRound < len || !MatOk(gate, len, dim, 2) || !MatOk(vals, len, dim, 2) || !MatOk(grad, len, dim, 2) ||
        !MatOk(gradGate, lenRound, dim, 2) || !MatOk(gradVals, lenRound, dim, 2) || (mode == 0 && !MatOk(valsSrcTileScale, dim / TILE, len, 4)) ||
        (mode == 1 && !MatOk(dScale, dim / TILE, lenRound, 4)) || !RowQuantOk(qGate, dim) || (mode == 0 && !RowQuantOk(qVals, dim))) {
        return TS2_ERR_UNSUPPORTED;
    }
    if (!Aligned16(gate->ptr, gate->strideBytes) || !Aligned16(vals->ptr, vals->strideBytes) || !Aligned16(grad->ptr, grad->strideBytes) ||
        !Aligned16(gradGate->ptr, gradGate->strideBytes) || !Aligned16(gradVals->ptr, gradVals->strideBytes)) {
        return TS2_ERR_UNSUPPORTED;
    }
    const dim3 blocks((lenRound + 3) / 4);
    if (mode == 0) {
        LAUNCH_ROW_CHUNKS((BackpropLoLURows<N, 0>), blocks, dim3(256), 0, STREAM, len, lenRound, dim, M(*gate), M(*vals), valsScale, M(*valsSrcTileScale),
            M(*grad), M(*gradGate), M(*gradVals), Mat{nullptr, 0}, qGate, qVals)
    } else {
        LAUNCH_ROW_CHUNKS((BackpropLoLURows<N, 1>), blocks, dim3(256), 0, STREAM, len, lenRound, dim, M(*gate), M(*vals), valsScale, Mat{nullptr, 0},
            M(*grad), M(*gradGate), M(*gradVals), M(*dScale), qGate, qVals)
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2BackpropNormRopeRows(int count, int len, int lenRound, const ts2_mat *const *grad, float gradMult, const ts2_mat *const *srcNorm,
    const ts2_mat *const *srcTileScale, const ts2_mat *const *ropeBuf, const ts2_mat *const *dst, const RowQuantOut *q, void *stream)
{
    if (count < 1 || count > 3 || lenRound <= 0 || lenRound < len) {
        return TS2_ERR_UNSUPPORTED;
    }
    const int dim = dst[0]->x;
    NormRopeRowJobs jobs = {};
    for (int i = 0; i < count; ++i) {
        if (dim % TILE || dim > 4096 || dst[i]->x != dim || !MatOk(grad[i], len, dim, 2) || !MatOk(dst[i], lenRound, dim, 2) || !RowQuantOk(q[i], dim) ||
            !Aligned16(grad[i]->ptr, grad[i]->strideBytes) || !Aligned16(dst[i]->ptr, dst[i]->strideBytes) ||
            (srcNorm[i] && (!MatOk(srcNorm[i], len, dim, 2) || !Aligned16(srcNorm[i]->ptr, srcNorm[i]->strideBytes) ||
                               !MatOk(srcTileScale[i], dim / TILE, len, 4))) ||
            (ropeBuf[i] && (!MatOk(ropeBuf[i], len, TILE, 4) || !Aligned16(ropeBuf[i]->ptr, ropeBuf[i]->strideBytes)))) {
            return TS2_ERR_UNSUPPORTED;
        }
        jobs.grad[i] = M(*grad[i]);
        jobs.dst[i] = M(*dst[i]);
        if (srcNorm[i]) {
            jobs.srcNorm[i] = M(*srcNorm[i]);
            jobs.srcTileScale[i] = M(*srcTileScale[i]);
        }
        if (ropeBuf[i]) {
            jobs.rope[i] = M(*ropeBuf[i]);
        }
        jobs.q[i] = q[i];
    }
    LAUNCH_ROW_CHUNKS((BackpropNormRopeRows<N>), dim3((lenRound + 3) / 4, count), dim3(256), 0, STREAM, len, lenRound, dim, gradMult, jobs)
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2BackpropLayerNormalizeRows(bool final, int len, int lenRound, const ts2_mat *normState, const ts2_mat *stateScale, const ts2_mat *dNormState,
    const float *gradScale, const float *gradMult, const ts2_mat *stateGrad, const ts2_mat *stateGradFast, float *nextMaxNorm, const RowQuantOut &q,
    void *stream)
{
    const int dim = dNormState->x;
    if (dim % TILE || dim > 1536 || lenRound <= 0 || lenRound < len || !MatOk(normState, len, dim, 1) || !MatOk(stateScale, dim / TILE, len, 4) ||
        !MatOk(dNormState, len, dim, 4) || !MatOk(stateGrad, final ? lenRound : len, dim, 4) || !MatOk(stateGradFast, final ? lenRound : len, dim, 2) ||
        !RowQuantOk(q, dim) || (((uintptr_t)normState->ptr | normState->strideBytes) & 7) || !Aligned16(dNormState->ptr, dNormState->strideBytes) ||
        !Aligned16(stateGrad->ptr, stateGrad->strideBytes) || !Aligned16(stateGradFast->ptr, stateGradFast->strideBytes)) {
        return TS2_ERR_UNSUPPORTED;
    }
    // one update of the maximum per workgroup, 10 ns each on its one address: workgroups of 1024 threads beyond 256 small ones
    const bool large = lenRound > 1024;
    const dim3 blocks(large ? (lenRound / 16 < 512 ? lenRound / 16 : 512) : (lenRound + 3) / 4);
#define BN_ROWS_OF(N, FINAL, NT)                                                                                                           \
    hipLaunchKernelGGL((BackpropLayerNormalizeRows<N, FINAL, NT>), blocks, dim3(NT), 0, STREAM, len, lenRound, dim, M(*normState), M(*stateScale), \
        M(*dNormState), gradScale, gradMult, M(*stateGrad), M(*stateGradFast), nextMaxNorm, q)
#define BN_ROWS(FINAL, NT)                                                                                                                 \
    if (dim <= 512) {                                                                                                                      \
        BN_ROWS_OF(1, FINAL, NT);                                                                                                          \
    } else if (dim <= 1024) {                                                                                                              \
        BN_ROWS_OF(2, FINAL, NT);                                                                                                          \
    } else {                                                                                                                               \
        BN_ROWS_OF(3, FINAL, NT); /* (wider rows do not fit the registers of 16 waves) */                                                  \
    }
    if (final && large) {
        BN_ROWS(true, 1024)
    } else if (final) {
        BN_ROWS(true, 256)
    } else if (large) {
        BN_ROWS(false, 1024)
    } else {
        BN_ROWS(false, 256)
    }
#undef BN_ROWS
#undef BN_ROWS_OF
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2ScaleGradRows(const float *gradMaxNorm, const float *prevGradMult, const ts2_mat *grad, const ts2_mat *gradFast, int len, float *gradScaleOut,
    float *gradMultOut, const RowQuantOut &q, void *stream)
{
    const int tiles = grad->x / TILE;
    hipLaunchKernelGGL((ScaleGrad<TBF16, true>), GridFor(len, tiles), dim3(256), 0, STREAM, len, tiles, gradMaxNorm, prevGradMult, M(*grad), M(*gradFast),
        gradScaleOut, gradMultOut, q);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2ScaleGradRows(const float *gradMaxNorm, const float *prevGradMult, const ts2_mat *grad, const ts2_mat *gradFast, int len, float *gradScaleOut,
    float *gradMultOut, float *rowScale, float *rowAbsMax, void *stream)
{
    return Ts2ScaleGradRows(gradMaxNorm, prevGradMult, grad, gradFast, len, gradScaleOut, gradMultOut, RowQuantOut{nullptr, 0, rowScale, rowAbsMax, 0}, stream);
}

// The row-major k-tile quantiser over any number of bf16 gradients with the same rows
int Ts2QuantTileRowsJobs(int count, int len, int lenRound, int kTile, const TileQuantJob *jobs, const float *rowMult, void *stream)
{
    if (count < 1 || lenRound < len || kTile <= 0 || kTile % 128 || lenRound % kTile) {
        return TS2_ERR_SHAPE;
    }
    for (int i = 0; i < count; ++i) {
        if (((uintptr_t)jobs[i].src | (uintptr_t)jobs[i].srcStride) & 15 || ((uintptr_t)jobs[i].dst | (uintptr_t)jobs[i].dstStride) & 7) {
            return TS2_ERR_ALIGN;
        }
        if (jobs[i].dim <= 0 || jobs[i].dim > 4096 || jobs[i].dim % 8 || jobs[i].srcStride < jobs[i].dim * 2 || jobs[i].dstStride < jobs[i].dim) {
            return TS2_ERR_SHAPE;
        }
    }
    for (int done = 0; done < count; done += QT_JOBS) {
        const int n = count - done < QT_JOBS ? count - done : QT_JOBS;
        const dim3 grid(lenRound / QT_ROWS, n);
        if (n <= 4) {
            TileQuantJobs<4> part = {};
            std::copy(jobs + done, jobs + done + n, part.job);
            hipLaunchKernelGGL((QuantTileRows<4>), grid, dim3(256), 0, STREAM, len, lenRound, kTile, part, rowMult);
        } else {
            TileQuantJobs<QT_JOBS> part = {};
            std::copy(jobs + done, jobs + done + n, part.job);
            hipLaunchKernelGGL((QuantTileRows<QT_JOBS>), grid, dim3(256), 0, STREAM, len, lenRound, kTile, part, rowMult);
        }
        TS2_CHECK_LAUNCH();
    }
    return TS2_OK;
}

// ... over `count` gradients of one shape; tileScale [count][lenRound / kTile]
int Ts2QuantTileRows(int count, int len, int lenRound, int kTile, const ts2_mat *src, const ts2_mat *dst, const float *const *rowAbsMax,
    const uint32_t *seed, const float *rowMult, float *tileScale, void *stream)
{
    if (count < 1 || count > 4 || dst[0].x % 8 || lenRound < len || kTile <= 0 || kTile % 128 || lenRound % kTile) {
        return TS2_ERR_SHAPE;
    }
    TileQuantJob jobs[4];
    for (int i = 0; i < count; ++i) {
        if (dst[i].x != dst[0].x || !MatOk(&src[i], len, dst[0].x, 2) || !MatOk(&dst[i], lenRound, dst[0].x, 1)) {
            return TS2_ERR_SHAPE;
        }
        jobs[i] = {(const uint8_t *)src[i].ptr, (uint8_t *)dst[i].ptr, src[i].strideBytes, dst[i].strideBytes, rowAbsMax[i],
            tileScale + (int64_t)i * (lenRound / kTile), dst[0].x, seed[i]};
    }
    return Ts2QuantTileRowsJobs(count, len, lenRound, kTile, jobs, rowMult, stream);
}

extern "C" int ts2_normalize_vecs_row_max_dither(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *colScale,
    const ts2_mat *dst, float *rowScale, float *rowAbsMax, uint32_t ditherSeed, void *stream)
{
    if (!src || !dst || !rowScale) {
        return TS2_ERR_NULL;
    }
    int dim = dst->x;
    if (dim % 4 || lenRound < len || !MatOk(src, len, dim, ElemSize(srcType)) || !MatOk(dst, lenRound, dim, 1)) {
        return TS2_ERR_SHAPE;
    }
    const bool reg = dim <= 4096;
    if (srcType == TS2_BF16 && dim % 8 == 0 && dim <= 4096 && Aligned16(src->ptr, src->strideBytes) && (((uintptr_t)dst->ptr | dst->strideBytes) & 7) == 0 &&
        (!colScale || ((uintptr_t)colScale & 15) == 0)) {
        RowQuantJobs jobs = {};
        jobs.src[0] = M(*src);
        jobs.dst[0] = M(*dst);
        jobs.rowScale[0] = rowScale;
        jobs.rowAbsMax[0] = rowAbsMax;
        jobs.seed[0] = ditherSeed;
        return LaunchRowQuant(1, len, lenRound, dim, jobs, colScale, stream);
    }
#define LAUNCH_RM(TS, REG) hipLaunchKernelGGL((NormalizeVecsRowMax<TS, REG>), dim3(lenRound < 4096 ? lenRound : 4096), dim3(256), 0, STREAM, len, lenRound, dim, M(*src), colScale, M(*dst), rowScale, rowAbsMax, ditherSeed)
    if (srcType == TS2_BF16) {
        if (reg) {
            LAUNCH_RM(TBF16, true);
        } else {
            LAUNCH_RM(TBF16, false);
        }
    } else if (srcType == TS2_F32) {
        if (reg) {
            LAUNCH_RM(TF32, true);
        } else {
            LAUNCH_RM(TF32, false);
        }
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_tile_absmax(int32_t len, const ts2_mat *src, int32_t srcType, const float *rowMult, int32_t kTile, float *tileMax, int32_t clear,
    void *stream)
{
    if (!src || !tileMax) {
        return TS2_ERR_NULL;
    }
    int dim = src->x;
    if (dim % 4 || kTile <= 0 || kTile % 128 || !MatOk(src, len, dim, ElemSize(srcType))) {
        return TS2_ERR_SHAPE;
    }
    if (((uintptr_t)src->ptr % 16) || (src->strideBytes % 16) || ((int64_t)dim * ElemSize(srcType)) % 16) {
        return TS2_ERR_ALIGN;
    }
    int nTiles = (len + kTile - 1) / kTile;
    if (clear) {
        hipLaunchKernelGGL(FillFloats, dim3((nTiles + 255) / 256), dim3(256), 0, STREAM, tileMax, nTiles, 0.f);
        TS2_CHECK_LAUNCH();
    }
    dim3 grid((dim * ElemSize(srcType) + 4095) / 4096, (len + 15) / 16);
    if (srcType == TS2_BF16) {
        hipLaunchKernelGGL((TileAbsMax<TBF16>), grid, dim3(256), 0, STREAM, len, dim, M(*src), rowMult, kTile, tileMax);
    } else if (srcType == TS2_F32) {
        hipLaunchKernelGGL((TileAbsMax<TF32>), grid, dim3(256), 0, STREAM, len, dim, M(*src), rowMult, kTile, tileMax);
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_transpose_quant(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *rowMult, const float *tileMax,
    int32_t kTile, const int32_t *rowIndex, const ts2_mat *dstT, int32_t dstType, float *tileScale, void *stream)
{
    return Ts2TransposeQuantRows(len, lenRound, src, srcType, rowMult, tileMax, nullptr, kTile, rowIndex, dstT, dstType, tileScale, stream);
}

extern "C" int ts2_transpose_quant_dither(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, const float *rowMult, const float *tileMax,
    int32_t kTile, const int32_t *rowIndex, const ts2_mat *dstT, int32_t dstType, float *tileScale, uint32_t ditherSeed, void *stream)
{
    return Ts2TransposeQuantRows(len, lenRound, src, srcType, rowMult, tileMax, nullptr, kTile, rowIndex, dstT, dstType, tileScale, stream, ditherSeed);
}

// ts2_transpose_quant whose k-tile maxima may come from the row maxima instead (rowAbsMax, with tileMax null; with a row index: the
// maxima of the rows gathered into the tile): the kernel then forms each k-tile's maximum itself and the separate
// ts2_tile_max_from_rows launch is not needed
int Ts2TransposeQuantRows(int len, int lenRound, const ts2_mat *src, int srcType, const float *rowMult, const float *tileMax, const float *rowAbsMax,
    int kTile, const int *rowIndex, const ts2_mat *dstT, int dstType, float *tileScale, void *stream, uint32_t ditherSeed)
{
    if (!src || !dstT) {
        return TS2_ERR_NULL;
    }
    int dim = dstT->y;
    if (dim % 128 || lenRound % 128 || lenRound < len || dstT->x < lenRound || src->x < dim || (dstT->strideBytes % 4) ||
        dstT->strideBytes < lenRound) {
        return TS2_ERR_SHAPE;
    }
    if (((uintptr_t)src->ptr % 16) || (src->strideBytes % 16) || ((uintptr_t)dstT->ptr % 16) || (dstT->strideBytes % 16)) {
        return TS2_ERR_ALIGN;
    }
    dim3 grid(dim / 128, lenRound / 128);
    bool quant = dstType == TS2_I8 && (srcType == TS2_BF16 || srcType == TS2_F32);
    if (quant) {
        if ((!tileMax && !rowAbsMax) || kTile <= 0 || kTile % 128) {
            return TS2_ERR_SHAPE;
        }
        if (tileMax) {
            rowAbsMax = nullptr;
        }
        if (srcType == TS2_BF16) {
            hipLaunchKernelGGL((TransposeQuant<TBF16, true>), grid, dim3(256), 0, STREAM, len, lenRound, M(*src), rowMult, tileMax, kTile, rowIndex,
                M(*dstT), tileScale, rowAbsMax, ditherSeed);
        } else {
            hipLaunchKernelGGL((TransposeQuant<TF32, true>), grid, dim3(256), 0, STREAM, len, lenRound, M(*src), rowMult, tileMax, kTile, rowIndex,
                M(*dstT), tileScale, rowAbsMax, ditherSeed);
        }
    } else if (ElemSize(srcType) == 1 && dstType == srcType) {
        hipLaunchKernelGGL((TransposeQuant<TI8, false>), grid, dim3(256), 0, STREAM, len, lenRound, M(*src), nullptr, nullptr, 128, rowIndex,
            M(*dstT), nullptr, nullptr, 0u);
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2TransposeBytesBatch(int count, const ts2_mat *const *src, const ts2_mat *const *dst, int const *rows, const int *cols, void *stream)
{
    for (int i = 0; i < count; ++i) {
        if (rows[i] <= 0 || cols[i] <= 0 || rows[i] % 128 || cols[i] % 128 || src[i]->x < cols[i] || src[i]->y < rows[i] || dst[i]->x < rows[i] || dst[i]->y < cols[i]) {
            return TS2_ERR_SHAPE;
        }
        if (!Aligned16(src[i]->ptr, src[i]->strideBytes) || !Aligned16(dst[i]->ptr, dst[i]->strideBytes)) {
            return TS2_ERR_ALIGN;
        }
    }
    for (int done = 0; done < count; done += TRANSPOSE_JOBS) {
        TransposeJobs jobs = {};
        const int n = count - done < TRANSPOSE_JOBS ? count - done : TRANSPOSE_JOBS;
        for (int i = 0; i < n; ++i) {
            jobs.src[i] = M(*src[done + i]);
            jobs.dst[i] = M(*dst[done + i]);
            jobs.tilesX[i] = cols[done + i] / 128;
            jobs.first[i + 1] = jobs.first[i] + jobs.tilesX[i] * (rows[done + i] / 128);
        }
        hipLaunchKernelGGL(TransposeBytes, dim3(jobs.first[n]), dim3(256), 0, STREAM, n, jobs);
        TS2_CHECK_LAUNCH();
    }
    return TS2_OK;
}

extern "C" int ts2_row_tile_normalize_rope(int32_t len, int32_t lenRound, const ts2_mat *src, int32_t srcType, float srcMult, int32_t normalize,
    float vecScale, const ts2_mat *ropeBuf, const ts2_mat *dst, const ts2_mat *tileScale, void *stream)
{
    if (!src || !dst || (normalize && !tileScale)) {
        return TS2_ERR_NULL;
    }
    int dim = dst->x;
    if (dim % TILE || !MatOk(src, len, dim, ElemSize(srcType)) || !MatOk(dst, lenRound, dim, 2) ||
        (normalize && !MatOk(tileScale, dim / TILE, lenRound, 4)) || (ropeBuf && !MatOk(ropeBuf, len, TILE, 4))) {
        return TS2_ERR_SHAPE;
    }
    int tiles = dim / TILE;
    Mat rope = ropeBuf ? M(*ropeBuf) : Mat{nullptr, 0};
    Mat ts = normalize ? M(*tileScale) : Mat{nullptr, 0};
    if (srcType == TS2_F32) {
        hipLaunchKernelGGL((RowTileNormalizeRope<TF32>), GridFor(lenRound, tiles), dim3(256), 0, STREAM, len, lenRound, tiles, M(*src), srcMult,
            normalize, vecScale, rope, M(*dst), ts);
    } else if (srcType == TS2_BF16) {
        hipLaunchKernelGGL((RowTileNormalizeRope<TBF16>), GridFor(lenRound, tiles), dim3(256), 0, STREAM, len, lenRound, tiles, M(*src), srcMult,
            normalize, vecScale, rope, M(*dst), ts);
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_backprop_row_tile_normalize_rope(int32_t len, int32_t lenRound, const ts2_mat *grad, int32_t gradType, float gradMult,
    const ts2_mat *srcNorm, const ts2_mat *srcTileScale, const ts2_mat *ropeBuf, const ts2_mat *dst, int32_t dstType, void *stream)
{
    return Ts2BackpropNormRopeGroup(1, len, lenRound, &grad, gradType, gradMult, &srcNorm, &srcTileScale, &ropeBuf, &dst, dstType, stream);
}

// the same for up to four gradients of one width, each with or without normalisation and rotation
int Ts2BackpropNormRopeGroup(int count, int len, int lenRound, const ts2_mat *const *grad, int gradType, float gradMult, const ts2_mat *const *srcNorm,
    const ts2_mat *const *srcTileScale, const ts2_mat *const *ropeBuf, const ts2_mat *const *dst, int dstType, void *stream)
{
    if (count < 1 || count > 4) {
        return TS2_ERR_SHAPE;
    }
    NormRopeJobs<4> jobs = {};
    bool wide = gradType == TS2_BF16 && dstType == TS2_E4M3; // eight elements per lane
    for (int i = 0; i < count; ++i) {
        if (!grad[i] || !dst[i] || (srcNorm[i] && !srcTileScale[i])) {
            return TS2_ERR_NULL;
        }
        const int dim = dst[i]->x;
        if (dim % TILE || dim != dst[0]->x || !MatOk(grad[i], len, dim, ElemSize(gradType)) || !MatOk(dst[i], lenRound, dim, ElemSize(dstType)) ||
            (srcNorm[i] && (!MatOk(srcNorm[i], len, dim, 2) || !MatOk(srcTileScale[i], dim / TILE, len, 4))) ||
            (ropeBuf[i] && !MatOk(ropeBuf[i], len, TILE, 4))) {
            return TS2_ERR_SHAPE;
        }
        jobs.grad[i] = M(*grad[i]);
        jobs.dst[i] = M(*dst[i]);
        if (srcNorm[i]) {
            jobs.srcNorm[i] = M(*srcNorm[i]);
            jobs.srcTileScale[i] = M(*srcTileScale[i]);
        }
        if (ropeBuf[i]) {
            jobs.rope[i] = M(*ropeBuf[i]);
        }
        wide = wide && Aligned16(grad[i]->ptr, grad[i]->strideBytes) && (!srcNorm[i] || Aligned16(srcNorm[i]->ptr, srcNorm[i]->strideBytes)) &&
               (!ropeBuf[i] || Aligned16(ropeBuf[i]->ptr, ropeBuf[i]->strideBytes)) && (((uintptr_t)dst[i]->ptr | dst[i]->strideBytes) & 7) == 0;
    }
    const int tiles = dst[0]->x / TILE;
    if (gradType != TS2_F32 && gradType != TS2_BF16) {
        return TS2_ERR_UNSUPPORTED;
    }
    const NormRopeJobs<1> one = {{jobs.grad[0]}, {jobs.srcNorm[0]}, {jobs.srcTileScale[0]}, {jobs.rope[0]}, {jobs.dst[0]}};
    if (wide) {
        const long lanes = ((long)lenRound * tiles * 16 + 1) / 2;
        const dim3 grid((unsigned)((lanes + 255) / 256), count);
        if (count == 1) {
            hipLaunchKernelGGL(BackpropRowTileNormalizeRope8<1>, grid, dim3(256), 0, STREAM, len, lenRound, tiles, gradMult, one);
        } else {
            hipLaunchKernelGGL(BackpropRowTileNormalizeRope8<4>, grid, dim3(256), 0, STREAM, len, lenRound, tiles, gradMult, jobs);
        }
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
    const dim3 grid(GridFor(lenRound, tiles).x, count);
#define LAUNCH_BR(TG, TD)                                                                                                                  \
    if (count == 1)                                                                                                                        \
        hipLaunchKernelGGL((BackpropRowTileNormalizeRope<TG, TD, 1>), grid, dim3(256), 0, STREAM, len, lenRound, tiles, gradMult, one);     \
    else                                                                                                                                   \
        hipLaunchKernelGGL((BackpropRowTileNormalizeRope<TG, TD, 4>), grid, dim3(256), 0, STREAM, len, lenRound, tiles, gradMult, jobs)
    if (gradType == TS2_F32) {
        TS2_DISPATCH_TYPE(dstType, TD, LAUNCH_BR(TF32, TD));
    } else {
        TS2_DISPATCH_TYPE(dstType, TD, LAUNCH_BR(TBF16, TD));
    }
#undef LAUNCH_BR
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_pack_delta(const ts2_mat *partial, int32_t splits, int64_t slabBytes, int32_t rows, int32_t cols, float alpha, const float *alphaPtr,
    const ts2_mat *delta, const ts2_mat *deltaTileScale, void *stream)
{
    if (!partial || !delta || !deltaTileScale) {
        return TS2_ERR_NULL;
    }
    if (cols % TILE || splits < 1 || !MatOk(partial, rows, cols, 4) || !MatOk(delta, rows, cols, 1) || !MatOk(deltaTileScale, cols / TILE, rows, 4) ||
        (slabBytes & 15) || (partial->strideBytes & 15) || ((uintptr_t)partial->ptr & 15)) {
        return TS2_ERR_SHAPE;
    }
    int tiles = cols / TILE;
    // While more than two slices together fit the L2s (32 MB), a row and eight slices at a time: 512 x 512 of 8 slices 3.2 us (3.7 with two
    // rows and two slices), 2048 x 1024 of 4 4.7 (5.2); beyond them two rows and two slices: 2048 x 1024 of 8 12.3 (14.1 with one and eight),
    // 8192 x 2048 of one 15.9.  Many slices from beyond the memory-side cache (256 MB) come one at a time: 2048 x 2048 of 32 89 (94)
    const int64_t bytes = (int64_t)splits * rows * cols * 4;
    const int form = splits > 2 && bytes <= 32 << 20 ? 1 : splits >= 8 && bytes > 256 << 20 ? 4 : 2; // rows of a group of lanes
    const long units = (long)((rows + form - 1) / form) * tiles;
    auto kernel = form == 1 ? PackDelta<1, 8> : form == 2 ? PackDelta<2, 2> : PackDelta<4, 1>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((units * 32 + 255) / 256)), dim3(256), 0, STREAM, rows, tiles, splits, (const uint8_t *)partial->ptr,
        partial->strideBytes, slabBytes, alpha, alphaPtr, M(*delta), M(*deltaTileScale));
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

extern "C" int ts2_backprop_row_tile_normalize_lolu_t(int32_t len, int32_t lenRound, const ts2_mat *gate, const ts2_mat *vals, float valsScale,
    const ts2_mat *valsSrcTileScale, const ts2_mat *grad, const ts2_mat *gradGate, const ts2_mat *gradVals, const ts2_mat *gradGateT,
    const ts2_mat *gradValsT, void *stream)
{
    if (!gate || !vals || !valsSrcTileScale || !grad || !gradGate || !gradVals || !gradGateT || !gradValsT) {
        return TS2_ERR_NULL;
    }
    int dim = grad->x;
    if (dim % TILE || lenRound % 128 || lenRound < len || !MatOk(gate, len, dim, 2) || !MatOk(vals, len, dim, 2) || !MatOk(grad, len, dim, 2) ||
        !MatOk(gradGate, lenRound, dim, 1) || !MatOk(gradVals, lenRound, dim, 1) || !MatOk(gradGateT, dim, lenRound, 1) ||
        !MatOk(gradValsT, dim, lenRound, 1) || !MatOk(valsSrcTileScale, dim / TILE, len, 4)) {
        return TS2_ERR_SHAPE;
    }
    if (!Aligned16(gate->ptr, gate->strideBytes) || !Aligned16(vals->ptr, vals->strideBytes) || !Aligned16(grad->ptr, grad->strideBytes) ||
        !Aligned16(gradGateT->ptr, gradGateT->strideBytes) || !Aligned16(gradValsT->ptr, gradValsT->strideBytes) ||
        (((uintptr_t)gradGate->ptr | gradGate->strideBytes | (uintptr_t)gradVals->ptr | gradVals->strideBytes) & 7)) {
        return TS2_ERR_ALIGN;
    }
    hipLaunchKernelGGL(BackpropLoLU8T, dim3(dim / TILE, lenRound / 128), dim3(256), 0, STREAM, len, lenRound, M(*gate), M(*vals), valsScale,
        M(*valsSrcTileScale), M(*grad), M(*gradGate), M(*gradVals), M(*gradGateT), M(*gradValsT));
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}
