// Kernels around the layer stack: label embedding, final soft-max / loss gradient and 16-bit transposed copies for the
// final layer's bf16 products (the reference runs them in fp16: src/gpt/compute/gpu_final.cuh:223-296, gpu_embedding.cuh:126-218).
#include "vec.h"
#include "internal.h"

namespace
{
// state0[t] = sum over labels of +-E[label] * scale (ComputeEmbedding, src/gpt/compute/cpu_transformer.cpp:76-100).  A row is a chain of
// three loads (its labels' range, a label, the label's matrix row) before it is written, and two more for every further label, so a workgroup
// takes ROWS rows and has the same label of all of them under way together: 65536 x 1024 of e4m3 99 -> 71 us inside a step (336 MB: 54 at the
// rate of a copy), 16384 x 512 of int8 10.9 -> 9.6, with four labels per row 20.7 -> 18.6.
template <class TEmb, int ROWS>
__global__ void __launch_bounds__(256) EmbedForward(int len, int lenRound, int dim, const int *labelPtr, const uint32_t *labels, const uint8_t *embed,
    int64_t ldEmb, float mult, const float *scalePtr, float *state, int64_t ldState)
{
    if ((int)threadIdx.x * 4 >= dim) { // (waves beyond a narrow row do not wait for its labels)
        return;
    }
    const int t0 = blockIdx.x * ROWS;
    const float s = mult * (scalePtr ? *scalePtr : 1.f);
    int from[ROWS], to[ROWS], most = 0;
    uint32_t one[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const bool live = t0 + r < len;
        from[r] = live ? labelPtr[t0 + r] : 0;
        to[r] = live ? labelPtr[t0 + r + 1] : 0;
        most = max(most, to[r] - from[r]);
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        one[r] = from[r] < to[r] ? labels[from[r]] : 0;
    }
    for (int col = threadIdx.x * 4; col < dim; col += 1024) {
        F4 acc[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            acc[r] = from[r] < to[r] ? Load4<TEmb>(embed + (int64_t)(one[r] & 0x7fffffffu) * ldEmb + col * TEmb::SIZE) : ZeroF4();
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (from[r] < to[r]) {
                acc[r] = ZeroF4() + acc[r] * ((one[r] & 0x80000000u) ? -s : s);
            }
        }
        for (int j = 1; j < most; ++j) {
            auto has = [&](int r) { return ROWS == 1 || from[r] + j < to[r]; };
            uint32_t label[ROWS];
            F4 v[ROWS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                label[r] = has(r) ? labels[from[r] + j] : 0;
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                v[r] = has(r) ? Load4<TEmb>(embed + (int64_t)(label[r] & 0x7fffffffu) * ldEmb + col * TEmb::SIZE) : ZeroF4();
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                if (has(r)) {
                    acc[r] = acc[r] + v[r] * ((label[r] & 0x80000000u) ? -s : s);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (t0 + r < lenRound) {
                Store4<TF32>((uint8_t *)state + (int64_t)(t0 + r) * ldState + col * 4, acc[r]);
            }
        }
    }
}

// deltaLabel[label] += +-grad[t]  (src/gpt/compute/cpu_transformer.cpp:182-197); fp32 atomics, delta cleared by the caller.  The memory is
// the model's own device memory, where the hardware's fp32 add applies: plain atomicAdd compiles to a compare-and-swap loop
__global__ void __launch_bounds__(256) EmbedBackward(int len, int dim, const int *labelPtr, const uint32_t *labels, const float *grad, int64_t ldGrad,
    float *delta, int64_t ldDelta)
{
    int t = blockIdx.x;
    for (int k = labelPtr[t]; k < labelPtr[t + 1]; ++k) {
        uint32_t label = labels[k];
        float w = (label & 0x80000000u) ? -1.f : 1.f;
        label &= 0x7fffffffu;
        for (int col = threadIdx.x; col < dim; col += 256) {
            unsafeAtomicAdd(delta + (int64_t)label * ldDelta / 4 + col, grad[(int64_t)t * ldGrad / 4 + col] * w);
        }
    }
}

// The same for a delta of many labels, most of them named once or not at all: cleared and added to, each of its rows moves three times.  With a
// mark per label - the only term that names it, or LABEL_NONE, or LABEL_MANY - a row that one term makes is stored, and only the others are cleared.
// 65536 x 1024, a label per row 261 -> 115 us; 50305 labels of 2048 drawn by 32768 rows 267 -> 184.
constexpr int LABEL_NONE = -1, LABEL_MANY = -2;

__global__ void __launch_bounds__(256) LabelsNone(int labelCount, int *mark)
{
    const int label = blockIdx.x * 256 + threadIdx.x;
    if (label < labelCount) {
        mark[label] = LABEL_NONE;
    }
}

// any one of the terms stays (plain stores: counters would queue behind each other on a label that many rows share)
__global__ void __launch_bounds__(256) LabelsNamed(int len, const int *labelPtr, const uint32_t *labels, int *mark)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < len) {
        for (int k = labelPtr[t]; k < labelPtr[t + 1]; ++k) {
            mark[labels[k] & 0x7fffffffu] = k;
        }
    }
}

// every other term says so (a term that reads another's "many" instead of the winner says the same)
__global__ void __launch_bounds__(256) LabelsMany(int len, const int *labelPtr, const uint32_t *labels, int *mark)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < len) {
        for (int k = labelPtr[t]; k < labelPtr[t + 1]; ++k) {
            int *const m = mark + (labels[k] & 0x7fffffffu);
            if (*m != k) {
                *m = LABEL_MANY;
            }
        }
    }
}

// a wave per label
__global__ void __launch_bounds__(256) ClearLabels(int labelCount, int dim, const int *mark, float *delta, int64_t ldDelta)
{
    const int label = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (label < labelCount && mark[label] < 0) {
        for (int col = (threadIdx.x & 63) * 4; col < dim; col += 256) {
            Store4<TF32>((uint8_t *)delta + label * ldDelta + col * 4, ZeroF4());
        }
    }
}

// a wave per row
__global__ void __launch_bounds__(256) EmbedBackwardMarked(int len, int dim, const int *labelPtr, const uint32_t *labels, const int *mark,
    const float *grad, int64_t ldGrad, float *delta, int64_t ldDelta)
{
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= len) {
        return;
    }
    const uint8_t *const src = (const uint8_t *)grad + t * ldGrad;
    const int end = labelPtr[t + 1];
    for (int k = labelPtr[t]; k < end; ++k) {
        const uint32_t id = labels[k];
        const float w = (id & 0x80000000u) ? -1.f : 1.f;
        const int64_t label = id & 0x7fffffffu;
        uint8_t *const dst = (uint8_t *)delta + label * ldDelta;
        if (mark[label] == k) {
            for (int col = lane * 4; col < dim; col += 256) {
                Store4<TF32>(dst + col * 4, ZeroF4() + Load4<TF32>(src + col * 4) * w);
            }
        } else {
            for (int col = lane; col < dim; col += 64) {
                unsafeAtomicAdd((float *)dst + col, ((const float *)src)[col] * w);
            }
        }
    }
}

// SoftMax base 2 and its (onehot - p) gradient (src/gpt/compute/cpu_transformer.cpp:12-37,146-159).
// logits fp32 [row][vocab] are overwritten by probabilities, grad is bf16, zero in rows without a target; vocab is a multiple of 4.
//
// Bounded by HBM: a row is read once and held in registers, NCH chunks of four per lane, by W waves (one wave and no barrier for small
// vocabularies, up to sixteen for large ones); one exponential and seven other instructions per logit.  Against two passes by a workgroup
// of four waves, repeated on one batch: 4096 x 1024 12.2 -> 7.3 us, x 8192 67 -> 51, x 16384 165 -> 140, 777 x 50304 91 -> 81 (one
// workgroup per CU: four rounds, the last of nine rows; twice the registers per lane and two workgroups to a CU spilled).
template <int W, int NCH>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W, 4) FinalProbabilities(int rows, int vocab, float *logits, int64_t ldLogits,
    const float *bias, const int *target, float gradMult, bf16_t *grad, int64_t ldGrad)
{
    __shared__ float redM[W], redS[W];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int t = W == 1 ? blockIdx.x * 4 + wave : blockIdx.x, first = W == 1 ? lane : threadIdx.x;
    if (t >= rows) { // (one wave per row: a whole wave, and no barrier below)
        return;
    }
    float *row = (float *)((uint8_t *)logits + (int64_t)t * ldLogits);
    bf16_t *grow = (bf16_t *)((uint8_t *)grad + (int64_t)t * ldGrad);
    const int tg = target[t];
    float4 x[NCH];
    float m = -1e30f, least = 1e30f; // the row's largest logit with its bias, the lane's smallest
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int k = (i * 64 * W + first) * 4;
        x[i] = k < vocab ? *(const float4 *)(row + k) : make_float4(-1e30f, -1e30f, -1e30f, -1e30f);
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int k = (i * 64 * W + first) * 4;
        if (k < vocab) {
            const float4 b = *(const float4 *)(bias + k);
            x[i] = make_float4(x[i].x + b.x, x[i].y + b.y, x[i].z + b.z, x[i].w + b.w);
            least = fminf(least, fminf(fminf(x[i].x, x[i].y), fminf(x[i].z, x[i].w)));
        }
        m = fmaxf(m, fmaxf(fmaxf(x[i].x, x[i].y), fmaxf(x[i].z, x[i].w)));
    }
    m = WaveMax(m);
    if (W > 1) {
        if (lane == 0) {
            redM[wave] = m;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            m = fmaxf(m, redM[w]);
        }
    }
    // A logit is the exponential's argument as it is while the largest leaves room for the sum, and relative to the largest otherwise: a
    // subtraction rounds (relative to 64 below the largest, rms error of a probability 7.6e-7 instead of 6e-8).  The hardware's exponential
    // returns zero below 2^-126; a wave that reaches there takes exp2f, which goes on to 2^-149 at five instructions more.
    m = fabsf(m) <= 64 ? 0.f : m;
    float sum = 0;
    int plain = __builtin_amdgcn_readfirstlane((int)__all(least - m >= -125)), wide = plain ^ 1;
    // loops of one trip or none, not branches: a join would cost registers
    asm volatile("" : "+s"(plain), "+s"(wide));
#pragma unroll 1
    for (int r = 0; r < plain; ++r) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) { // (chunks beyond the vocabulary hold -1e30: weight zero)
            x[i] = make_float4(__builtin_amdgcn_exp2f(x[i].x - m), __builtin_amdgcn_exp2f(x[i].y - m), __builtin_amdgcn_exp2f(x[i].z - m),
                __builtin_amdgcn_exp2f(x[i].w - m));
            sum += (x[i].x + x[i].y) + (x[i].z + x[i].w);
        }
    }
#pragma unroll 1
    for (int r = 0; __builtin_expect(r < wide, 0); ++r) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            x[i] = make_float4(exp2f(x[i].x - m), exp2f(x[i].y - m), exp2f(x[i].z - m), exp2f(x[i].w - m));
            sum += (x[i].x + x[i].y) + (x[i].z + x[i].w);
        }
    }
    sum = WaveSum(sum);
    if (W > 1) {
        if (lane == 0) {
            redS[wave] = sum;
        }
        __syncthreads();
        sum = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            sum += redS[w];
        }
    }
    const float scale = 1 / sum, neg = -gradMult;
    const uint32_t live = tg < 0 ? 0u : ~0u; // (zero in a row without a target, whatever its probabilities are)
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int k = (i * 64 * W + first) * 4;
        if (k < vocab) {
            const float p[4] = {x[i].x * scale, x[i].y * scale, x[i].z * scale, x[i].w * scale};
            *(float4 *)(row + k) = make_float4(p[0], p[1], p[2], p[3]);
            float g[4] = {p[0] * neg, p[1] * neg, p[2] * neg, p[3] * neg};
            if ((unsigned)(tg - k) < 4u) { // the target's chunk (no chunk of a row without one)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    g[e] = e == tg - k ? (1 - p[e]) * gradMult : g[e];
                }
            }
            *(uint2 *)(grow + k) = make_uint2(PackBf16x2(g[0], g[1]) & live, PackBf16x2(g[2], g[3]) & live);
        }
    }
}

// The same for vocabularies that do not fit the registers of sixteen waves: one workgroup per row, two passes with 16-byte accesses; the
// first finds the maximum and the sum together (the sum is rescaled whenever a lane's maximum grows), the second, served by the caches,
// writes.
__global__ void __launch_bounds__(256) FinalProbabilitiesTwoPass(int vocab, float *logits, int64_t ldLogits, const float *bias, const int *target,
    float gradMult, bf16_t *grad, int64_t ldGrad)
{
    __shared__ float redM[4], redS[4];
    int t = blockIdx.x;
    int tid = threadIdx.x;
    float *row = (float *)((uint8_t *)logits + (int64_t)t * ldLogits);
    bf16_t *grow = (bf16_t *)((uint8_t *)grad + (int64_t)t * ldGrad);
    int tg = target[t];
    if (tg < 0) {
        for (int k = tid * 4; k < vocab; k += 1024) {
            *(uint2 *)(grow + k) = make_uint2(0, 0);
        }
    }
    // lane-local reference m (the running maximum of the logits with their bias where it exceeds 64, which leaves room for the sum, else 0) and
    // sum of 2^(x + bias - m)
    float m = 0, sum = 0;
    for (int k0 = tid * 4; k0 < vocab; k0 += 4096) {
        float4 x[4], bv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int k = k0 + i * 1024;
            bool in = k < vocab;
            x[i] = in ? *(const float4 *)(row + k) : make_float4(-1e30f, -1e30f, -1e30f, -1e30f);
            bv[i] = in ? *(const float4 *)(bias + k) : make_float4(0, 0, 0, 0);
        }
        float mNew = m;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = make_float4(x[i].x + bv[i].x, x[i].y + bv[i].y, x[i].z + bv[i].z, x[i].w + bv[i].w);
            mNew = fmaxf(mNew, fmaxf(fmaxf(x[i].x, x[i].y), fmaxf(x[i].z, x[i].w)));
        }
        if (mNew > 64) {
            sum *= exp2f(m - mNew);
            m = mNew;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            sum += (exp2f(x[i].x - m) + exp2f(x[i].y - m)) + (exp2f(x[i].z - m) + exp2f(x[i].w - m));
        }
    }
    float mx = WaveMax(m);
    if ((tid & 63) == 0) {
        redM[tid >> 6] = mx;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(redM[0], redM[1]), fmaxf(redM[2], redM[3]));
    sum = WaveSum(sum * exp2f(m - mx));
    if ((tid & 63) == 0) {
        redS[tid >> 6] = sum;
    }
    __syncthreads();
    float scale = 1 / ((redS[0] + redS[1]) + (redS[2] + redS[3]));
    for (int k0 = tid * 4; k0 < vocab; k0 += 4096) {
        float4 x[4], bv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int k = k0 + i * 1024;
            bool in = k < vocab;
            x[i] = in ? *(const float4 *)(row + k) : make_float4(0, 0, 0, 0);
            bv[i] = in ? *(const float4 *)(bias + k) : make_float4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int k = k0 + i * 1024;
            if (k >= vocab) {
                continue;
            }
            float p[4] = {exp2f(x[i].x + bv[i].x - mx) * scale, exp2f(x[i].y + bv[i].y - mx) * scale, exp2f(x[i].z + bv[i].z - mx) * scale,
                exp2f(x[i].w + bv[i].w - mx) * scale};
            *(float4 *)(row + k) = make_float4(p[0], p[1], p[2], p[3]);
            if (tg >= 0) {
                float g[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    g[e] = ((k + e == tg ? 1.f : 0.f) - p[e]) * gradMult;
                }
                *(uint2 *)(grow + k) = make_uint2(PackBf16x2(g[0], g[1]), PackBf16x2(g[2], g[3]));
            }
        }
    }
}

// dst[x][t] = bf16(src[t][x]) for t < rows, 0 up to rowsRound; 64x64 tiles through LDS
template <class TSrc>
__global__ void __launch_bounds__(256) TransposeToBf16(int rows, int rowsRound, int cols, const uint8_t *src, int64_t ldSrc, uint8_t *dst, int64_t ldDst)
{
    __shared__ float tile[64][65];
    int x0 = blockIdx.x * 64, t0 = blockIdx.y * 64;
    int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 64; r += 4) {
        int t = t0 + r, x = x0 + tx;
        float v = 0;
        if (t < rows && x < cols) {
            const uint8_t *p = src + (int64_t)t * ldSrc + (int64_t)x * TSrc::SIZE;
            if (TSrc::SIZE == 2) {
                v = Bf16ToFloat(*(const bf16_t *)p);
            } else if (std::is_same<TSrc, TI8>::value) {
                v = (float)*(const int8_t *)p;
            } else {
                v = __builtin_amdgcn_cvt_f32_fp8((int)*p, 0);
            }
        }
        tile[r][tx] = v;
    }
    __syncthreads();
    for (int r = ty; r < 64; r += 4) {
        int x = x0 + r, t = t0 + tx;
        if (x < cols && t < rowsRound) {
            *(bf16_t *)(dst + (int64_t)x * ldDst + (int64_t)t * 2) = FloatToBf16(tile[tx][r]);
        }
    }
}

// dst[x][t] = src[t][x] for 2-byte elements, zeros for rows <= t < rowsRound; 64x64 tiles, 16-byte loads and stores.
// cols and rowsRound are multiples of 8, rows of both matrices 16-byte aligned.
__global__ void __launch_bounds__(256) Transpose16(int rows, int rowsRound, int cols, const uint8_t *src, int64_t ldSrc, uint8_t *dst, int64_t ldDst)
{
    constexpr int PITCH = 66; // 2-byte elements per LDS row: column reads of neighbouring lanes fall into different banks
    __shared__ __attribute__((aligned(16))) uint16_t tile[64 * PITCH];
    int x0 = blockIdx.x * 64, t0 = blockIdx.y * 64;
    int tid = threadIdx.x;
    int lc = tid & 7, lr = tid >> 3; // 8 lanes x 16 bytes per row, 32 rows per pass
    v4i raw[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int t = t0 + lr + 32 * k, x = x0 + lc * 8;
        raw[k] = (t < rows && x < cols) ? *(const v4i *)(src + (int64_t)t * ldSrc + (int64_t)x * 2) : (v4i){0, 0, 0, 0};
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        uint32_t *d = (uint32_t *)(tile + (lr + 32 * k) * PITCH + lc * 8);
        d[0] = (uint32_t)raw[k][0];
        d[1] = (uint32_t)raw[k][1];
        d[2] = (uint32_t)raw[k][2];
        d[3] = (uint32_t)raw[k][3];
    }
    __syncthreads();
    // thread -> destination row x (64 of them), 8 consecutive t (8 blocks): 2 units per thread
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        int u = tid + 256 * k;
        int tb = u & 7, xr = u >> 3;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t lo = tile[(tb * 8 + 2 * e) * PITCH + xr];
            uint32_t hi = tile[(tb * 8 + 2 * e + 1) * PITCH + xr];
            w[e] = lo | (hi << 16);
        }
        int x = x0 + xr, t = t0 + tb * 8;
        if (x < cols && t < rowsRound) {
            *(uint4 *)(dst + (int64_t)x * ldDst + (int64_t)t * 2) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

__global__ void ZeroBytes(uint8_t *p, int64_t ld, int rowBytes)
{
    uint8_t *row = p + (int64_t)blockIdx.x * ld;
    for (int x = threadIdx.x * 4; x < rowBytes; x += blockDim.x * 4) {
        *(uint32_t *)(row + x) = 0;
    }
}
// The same for IEEE-half logits (the reference keeps its logit window in half, src/gpt/compute/gpu_final.cuh:173-189): eight values
// per 16-byte load, no probabilities kept
__global__ void __launch_bounds__(256) FinalSoftmaxGradHalf(int vocab, const _Float16 *logits, int64_t ldLogits, const float *bias, const int *target,
    float gradMult, bf16_t *grad, int64_t ldGrad, float *lossSum)
{
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    __shared__ float redM[4], redS[4];
    int t = blockIdx.x;
    int tid = threadIdx.x;
    const _Float16 *row = (const _Float16 *)((const uint8_t *)logits + (int64_t)t * ldLogits);
    bf16_t *grow = (bf16_t *)((uint8_t *)grad + (int64_t)t * ldGrad);
    int tg = target[t];
    if (tg < 0) {
        for (int k = tid * 8; k < vocab; k += 2048) {
            *(uint4 *)(grow + k) = make_uint4(0, 0, 0, 0);
        }
        return;
    }
    float m = 0, sum = 0;
    for (int k0 = tid * 8; k0 < vocab; k0 += 4096) {
        float x[2][8], bv[2][8];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            int k = k0 + i * 2048;
            bool in = k < vocab;
            v8h h = in ? *(const v8h *)(row + k) : (v8h)(_Float16)-60000.f;
            float4 b0 = in ? *(const float4 *)(bias + k) : make_float4(0, 0, 0, 0);
            float4 b1 = in ? *(const float4 *)(bias + k + 4) : make_float4(0, 0, 0, 0);
            const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[i][e] = (float)h[e];
                bv[i][e] = bb[e];
            }
        }
        float mNew = m;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                mNew = fmaxf(mNew, x[i][e]);
            }
        }
        sum *= exp2f(m - mNew);
        m = mNew;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sum += exp2f(x[i][e] + bv[i][e] - m);
            }
        }
    }
    float mx = WaveMax(m);
    if ((tid & 63) == 0) {
        redM[tid >> 6] = mx;
    }
    __syncthreads();
    mx = fmaxf(fmaxf(redM[0], redM[1]), fmaxf(redM[2], redM[3]));
    sum = WaveSum(sum * exp2f(m - mx));
    if ((tid & 63) == 0) {
        redS[tid >> 6] = sum;
    }
    __syncthreads();
    float scale = 1 / ((redS[0] + redS[1]) + (redS[2] + redS[3]));
    for (int k = tid * 8; k < vocab; k += 2048) {
        v8h h = *(const v8h *)(row + k); // second read of the row: served by L2
        float4 b0 = *(const float4 *)(bias + k), b1 = *(const float4 *)(bias + k + 4);
        const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
        float g[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float pr = exp2f((float)h[e] + bb[e] - mx) * scale;
            g[e] = ((k + e == tg ? 1.f : 0.f) - pr) * gradMult;
            if (k + e == tg && lossSum) {
                atomicAdd(lossSum, logf(pr));
            }
        }
        *(uint4 *)(grow + k) = make_uint4(PackBf16x2(g[0], g[1]), PackBf16x2(g[2], g[3]), PackBf16x2(g[4], g[5]), PackBf16x2(g[6], g[7]));
    }
}
// The same for rows of at most ROW_ROUNDS * 8192 logits, with the row read once and one exponential per logit: a workgroup of 1024
// threads walks rows with a grid stride and a thread keeps its logits in registers.  It takes its own maximum first (packed half
// max), replaces every logit by 2^(logit + bias - own reference) as a half (a number in [0, 1] with 11 significant bits, more than
// the bf16 gradient keeps) while summing in fp32, and after the workgroup reduction the gradient is that half times one per-thread
// factor.  The next row's loads are in flight during all of this.  Arithmetic per logit: two conversions, two adds, one v_exp_f32,
// one sum, one multiply - the two-pass kernel above is bound by its VALU work (two exponentials per logit), not by memory.
constexpr int ROW_ROUNDS = 7; // up to 57344 logits; 2 x 28 registers of row data per thread

__global__ void __launch_bounds__(1024) FinalSoftmaxGradHalfRow(int rows, int vocab, const _Float16 *logits, int64_t ldLogits, const float *bias,
    const int *target, float gradMult, bf16_t *grad, int64_t ldGrad, float *lossSum)
{
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    __shared__ float redM[16], redS[16];
    const int tid = threadIdx.x;
    v8h cur[ROW_ROUNDS], nxt[ROW_ROUNDS];
    auto prefetch = [&](int t) {
        const _Float16 *row = (const _Float16 *)((const uint8_t *)logits + (int64_t)t * ldLogits);
#pragma unroll
        for (int i = 0; i < ROW_ROUNDS; ++i) {
            int k = tid * 8 + i * 8192;
            nxt[i] = k < vocab ? *(const v8h *)(row + k) : (v8h)(_Float16)-60000.f;
        }
    };
    int t = blockIdx.x;
    if (t < rows) {
        prefetch(t);
    }
    // a thread meets the same columns in every row: the largest bias among them, added to its reference, keeps the halves in [0, 1]
    float biasTop = 0;
#pragma unroll
    for (int i = 0; i < ROW_ROUNDS; ++i) {
        int k = tid * 8 + i * 8192;
        if (k < vocab) {
            float4 b0 = *(const float4 *)(bias + k), b1 = *(const float4 *)(bias + k + 4);
            biasTop = fmaxf(fmaxf(fmaxf(biasTop, fmaxf(b0.x, b0.y)), fmaxf(b0.z, b0.w)), fmaxf(fmaxf(b1.x, b1.y), fmaxf(b1.z, b1.w)));
        }
    }
    float loss = 0; // of the thread that met the rows' labels: one atomic per workgroup, not one per row (13 ns each on one address)
    for (; t < rows; t += gridDim.x) {
#pragma unroll
        for (int i = 0; i < ROW_ROUNDS; ++i) {
            cur[i] = nxt[i];
        }
        if (t + (int)gridDim.x < rows) {
            prefetch(t + gridDim.x);
        }
        bf16_t *grow = (bf16_t *)((uint8_t *)grad + (int64_t)t * ldGrad);
        const int tg = target[t];
        if (tg < 0) { // (workgroup-uniform) no label: zero gradient
            for (int k = tid * 8; k < vocab; k += 8192) {
                *(uint4 *)(grow + k) = make_uint4(0, 0, 0, 0);
            }
            continue;
        }
        // own reference: the largest logit (not below 0, as in the two-pass kernel) plus the largest bias of the thread's columns
        v8h hm = cur[0];
#pragma unroll
        for (int i = 1; i < ROW_ROUNDS; ++i) {
            hm = __builtin_elementwise_max(hm, cur[i]);
        }
        float m = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            m = fmaxf(m, (float)hm[e]);
        }
        m += biasTop;
        float sum = 0;
#pragma unroll
        for (int i = 0; i < ROW_ROUNDS; ++i) {
            int k = tid * 8 + i * 8192;
            if (k < vocab) {
                float4 b0 = *(const float4 *)(bias + k), b1 = *(const float4 *)(bias + k + 4);
                const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
                v8h ex;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float w = __builtin_amdgcn_exp2f((float)cur[i][e] + (bb[e] - m)); // hardware exp2: below 2^-126 flushed to zero
                    sum += w;
                    ex[e] = (_Float16)w;
                }
                cur[i] = ex;
            }
        }
        float mx = WaveMax(m);
        if ((tid & 63) == 0) {
            redM[tid >> 6] = mx;
        }
        __syncthreads();
        mx = redM[0];
#pragma unroll
        for (int w = 1; w < 16; ++w) {
            mx = fmaxf(mx, redM[w]);
        }
        const float own = __builtin_amdgcn_exp2f(m - mx); // own reference -> row reference
        sum = WaveSum(sum * own);
        if ((tid & 63) == 0) {
            redS[tid >> 6] = sum;
        }
        __syncthreads();
        float total = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            total += redS[w];
        }
        const float scale = own / total;       // half -> probability
        const float negScale = -scale * gradMult; // half -> gradient of a logit that is not the label
#pragma unroll
        for (int i = 0; i < ROW_ROUNDS; ++i) {
            int k = tid * 8 + i * 8192;
            if (k < vocab) {
                float g[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    g[e] = (float)cur[i][e] * negScale;
                }
                if ((unsigned)(tg - k) < 8u) { // the label's chunk (one thread of the workgroup)
                    float pr = 0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        pr = e == tg - k ? (float)cur[i][e] * scale : pr;
                    }
                    const float gt = (1.f - pr) * gradMult;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        g[e] = e == tg - k ? gt : g[e];
                    }
                    loss += logf(pr);
                }
                *(uint4 *)(grow + k) = make_uint4(PackBf16x2(g[0], g[1]), PackBf16x2(g[2], g[3]), PackBf16x2(g[4], g[5]), PackBf16x2(g[6], g[7]));
            }
        }
        __syncthreads(); // the reduction slots are free again
    }
    if (lossSum) {
        loss = WaveSum(loss);
        if ((tid & 63) == 0) {
            redS[tid >> 6] = loss;
        }
        __syncthreads();
        if (tid == 0) {
            float total = 0;
            for (int w = 0; w < 16; ++w) {
                total += redS[w];
            }
            if (total != 0) {
                unsafeAtomicAdd(lossSum, total);
            }
        }
    }
}

// Vocabularies up to 2048: one wave per row, the row in its registers (NCH chunks of 512 halves), waves walk rows with the grid's stride,
// the next row's loads in flight.  Per logit one exponential in fp32, the arithmetic of the two-pass kernel but for the reference, which
// counts the bias.  A workgroup adds its
// rows' loss once: the per-row atomic on one address alone took 13 ns a row (16384 x 1024 logits: 213 us, now 24; 65536 x 128: 834 us).
template <int NCH>
__global__ void __launch_bounds__(256) FinalSoftmaxGradHalfWave(int rows, int vocab, const _Float16 *logits, int64_t ldLogits, const float *bias,
    const int *target, float gradMult, bf16_t *grad, int64_t ldGrad, float *lossSum)
{
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    __shared__ float red[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int stride = gridDim.x * 4;
    float bv[NCH][8];
    bool in[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int k = (i * 64 + lane) * 8;
        in[i] = k < vocab;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            bv[i][e] = in[i] ? bias[k + e] : 0.f;
        }
    }
    v8h nxt[NCH];
    int tgNext = -1;
    auto prefetch = [&](int t) {
        const _Float16 *row = (const _Float16 *)((const uint8_t *)logits + (int64_t)t * ldLogits);
        tgNext = target[t];
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            nxt[i] = in[i] ? *(const v8h *)(row + (i * 64 + lane) * 8) : (v8h)(_Float16)-60000.f;
        }
    };
    int t = blockIdx.x * 4 + wave;
    if (t < rows) {
        prefetch(t);
    }
    float loss = 0;
    for (; t < rows; t += stride) {
        v8h cur[NCH];
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            cur[i] = nxt[i];
        }
        const int tg = tgNext;
        if (t + stride < rows) {
            prefetch(t + stride);
        }
        bf16_t *grow = (bf16_t *)((uint8_t *)grad + (int64_t)t * ldGrad);
        if (tg < 0) { // (uniform over the wave) no label: zero gradient
#pragma unroll
            for (int i = 0; i < NCH; ++i) {
                if (in[i]) {
                    *(uint4 *)(grow + (i * 64 + lane) * 8) = make_uint4(0, 0, 0, 0);
                }
            }
            continue;
        }
        float m = 0;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                m = fmaxf(m, (float)cur[i][e] + bv[i][e]); // (with its bias: no bias overflows the exponential)
            }
        }
        m = WaveMax(m);
        float p[NCH][8], sum = 0;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                p[i][e] = in[i] ? exp2f((float)cur[i][e] + bv[i][e] - m) : 0.f;
                sum += p[i][e];
            }
        }
        const float scale = 1 / WaveSum(sum);
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int k = (i * 64 + lane) * 8;
            float g[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pr = p[i][e] * scale;
                g[e] = ((k + e == tg ? 1.f : 0.f) - pr) * gradMult;
                if (k + e == tg) {
                    loss += logf(pr);
                }
            }
            if (in[i]) {
                *(uint4 *)(grow + k) = make_uint4(PackBf16x2(g[0], g[1]), PackBf16x2(g[2], g[3]), PackBf16x2(g[4], g[5]), PackBf16x2(g[6], g[7]));
            }
        }
    }
    loss = WaveSum(loss);
    if (lane == 0) {
        red[wave] = loss;
    }
    __syncthreads();
    if (threadIdx.x == 0 && lossSum) {
        const float total = (red[0] + red[1]) + (red[2] + red[3]);
        if (total != 0) {
            unsafeAtomicAdd(lossSum, total);
        }
    }
}
} // namespace

#define STREAM ((hipStream_t)stream)

int Ts2EmbedForward(int len, int lenRound, int dim, const int *labelPtr, const uint32_t *labels, const ts2_mat *embed, int embType, float mult,
    const float *scalePtr, const ts2_mat *state, void *stream)
{
    // more rows than keep every CU's waves busy anyway, and then the more rows the better while the rows are short: 8192 x 512 with one, two and
    // four rows to a workgroup 6.0, 6.1, 6.5 us, 16384 x 512 10.4, 9.6, 10.2, 65536 x 256 25.4, 20.7, 18.4 (four labels: 52.4, 43.8, 39.5)
    const int per = lenRound >= 32768 ? 4 : lenRound >= 12288 ? 2 : 1;
#define LAUNCH_E(T, N)                                                                                                                     \
    hipLaunchKernelGGL((EmbedForward<T, N>), dim3((lenRound + N - 1) / N), dim3(256), 0, STREAM, len, lenRound, dim, labelPtr, labels,      \
        (const uint8_t *)embed->ptr, embed->strideBytes, mult, scalePtr, (float *)state->ptr, state->strideBytes)
#define LAUNCH_ROWS(T)                                                                                                                     \
    if (per == 4) {                                                                                                                        \
        LAUNCH_E(T, 4);                                                                                                                    \
    } else if (per == 2) {                                                                                                                 \
        LAUNCH_E(T, 2);                                                                                                                    \
    } else {                                                                                                                               \
        LAUNCH_E(T, 1);                                                                                                                    \
    }
    if (embType == TS2_I8) {
        LAUNCH_ROWS(TI8)
    } else if (embType == TS2_E4M3) {
        LAUNCH_ROWS(TE4M3)
#undef LAUNCH_ROWS
#undef LAUNCH_E
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

// Where the marks pay: five launches instead of two, and waves instead of workgroups on the rows that share a label.  Measured over 16385 to 131073
// labels, 256 to 4096 columns and a quarter to four times as many rows as labels, with labels drawn evenly (e), by Zipf's law (z) and as the sixth power
// of an even number (p, 16 % of the rows name one label); time with marks over time without, e z p:
//   elements   65537 x 512 (2^25), 65536 rows 0.75 0.94 1.01; 50305 x 1024 (2^25.6), 32768 rows 0.72 0.97 1.03, 50000 rows 0.74 0.95 1.02; 65537 x 1024 (2^26),
//              32768 rows 0.74 0.97 1.00, 65536 rows 0.72 0.92 0.98; 131073 x 2048, 131072 rows 0.70 0.88 0.88
//   rows       65537 x 1024, 16385 rows 0.84 1.04 1.12, 28672 rows 0.76 0.98 1.03; 50305 x 1536, 25000 rows 0.75 0.96 1.04, 32768 rows 0.70 0.93 0.99
//   labels     40961 x 1536, 32768 rows 0.71 0.92 1.02, 50305 as above; 32769 x 2048, 32768 rows 0.73 1.00 1.02; 16385 x 4096, 16384 rows 0.74 1.07 1.11
//   rows to labels  98305 x 768, a third 0.80 0.94 1.02, half 0.73 0.92 0.99; 131073 x 512, a quarter 0.79 1.01 1.04, half 0.67 0.94 0.98; 65537 x 1024, 1.4 0.80 0.92
//              0.98, twice 0.89 0.93 0.98 but 1.03 where each is named twice
static bool MarkLabels(int len, int dim, int labelCount)
{
    return (int64_t)labelCount * dim >= (int64_t)7 << 23 && len >= 30720 && labelCount >= 45056 && (int64_t)len * 16 >= (int64_t)labelCount * 7 &&
           (int64_t)len * 2 <= (int64_t)labelCount * 3;
}

int Ts2EmbedBackward(int len, int dim, const int *labelPtr, const uint32_t *labels, const ts2_mat *grad, const ts2_mat *delta, int labelCount,
    int *mark, void *stream)
{
    if (mark && MarkLabels(len, dim, labelCount)) {
        const dim3 terms((len + 255) / 256);
        hipLaunchKernelGGL(LabelsNone, dim3((labelCount + 255) / 256), dim3(256), 0, STREAM, labelCount, mark);
        hipLaunchKernelGGL(LabelsNamed, terms, dim3(256), 0, STREAM, len, labelPtr, labels, mark);
        hipLaunchKernelGGL(LabelsMany, terms, dim3(256), 0, STREAM, len, labelPtr, labels, mark);
        hipLaunchKernelGGL(ClearLabels, dim3((labelCount + 3) / 4), dim3(256), 0, STREAM, labelCount, dim, mark, (float *)delta->ptr, delta->strideBytes);
        hipLaunchKernelGGL(EmbedBackwardMarked, dim3((len + 3) / 4), dim3(256), 0, STREAM, len, dim, labelPtr, labels, mark, (const float *)grad->ptr,
            grad->strideBytes, (float *)delta->ptr, delta->strideBytes);
        TS2_CHECK_LAUNCH();
        return TS2_OK;
    }
    hipLaunchKernelGGL(ZeroBytes, dim3(labelCount), dim3(256), 0, STREAM, (uint8_t *)delta->ptr, delta->strideBytes, dim * 4);
    TS2_CHECK_LAUNCH();
    hipLaunchKernelGGL(EmbedBackward, dim3(len), dim3(256), 0, STREAM, len, dim, labelPtr, labels, (const float *)grad->ptr, grad->strideBytes,
        (float *)delta->ptr, delta->strideBytes);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2FinalSoftmaxGradHalf(int rows, int vocab, const ts2_mat *logits, const float *bias, const int *target, float gradMult, const ts2_mat *grad,
    float *lossSum, void *stream)
{
    if (vocab % 8 || (logits->strideBytes & 15) || (grad->strideBytes & 15) || ((uintptr_t)logits->ptr & 15) || ((uintptr_t)grad->ptr & 15) ||
        ((uintptr_t)bias & 15)) {
        return TS2_ERR_ALIGN;
    }
    if (vocab <= 2048) {
        // eight workgroups of four waves per CU at most: each walks several rows and adds one loss
        const int wgs = (rows + 3) / 4 < 2048 ? (rows + 3) / 4 : 2048;
#define LAUNCH_SW(N)                                                                                                                       \
    hipLaunchKernelGGL((FinalSoftmaxGradHalfWave<N>), dim3(wgs), dim3(256), 0, STREAM, rows, vocab, (const _Float16 *)logits->ptr,          \
        logits->strideBytes, bias, target, gradMult, (bf16_t *)grad->ptr, grad->strideBytes, lossSum)
        switch ((vocab + 511) / 512) {
        case 1: LAUNCH_SW(1); break;
        case 2: LAUNCH_SW(2); break;
        case 3: LAUNCH_SW(3); break;
        default: LAUNCH_SW(4); break;
        }
#undef LAUNCH_SW
    } else if (vocab <= ROW_ROUNDS * 8192) {
        const int wgs = rows < 512 ? rows : 512; // one workgroup of 16 waves per CU is resident (registers); two per CU in the queue
        hipLaunchKernelGGL(FinalSoftmaxGradHalfRow, dim3(wgs), dim3(1024), 0, STREAM, rows, vocab, (const _Float16 *)logits->ptr,
            logits->strideBytes, bias, target, gradMult, (bf16_t *)grad->ptr, grad->strideBytes, lossSum);
    } else {
        hipLaunchKernelGGL(FinalSoftmaxGradHalf, dim3(rows), dim3(256), 0, STREAM, vocab, (const _Float16 *)logits->ptr, logits->strideBytes, bias,
            target, gradMult, (bf16_t *)grad->ptr, grad->strideBytes, lossSum);
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2FinalProbabilities(int rows, int vocab, const ts2_mat *logits, const float *bias, const int *target, float gradMult, const ts2_mat *grad,
    void *stream)
{
#define LAUNCH_P(W, N)                                                                                                                     \
    hipLaunchKernelGGL((FinalProbabilities<W, N>), dim3(W == 1 ? (rows + 3) / 4 : rows), dim3(W == 1 ? 256 : 64 * W), 0, STREAM, rows, vocab, \
        (float *)logits->ptr, logits->strideBytes, bias, target, gradMult, (bf16_t *)grad->ptr, grad->strideBytes)
    // of 256 logits: one float4 per lane of a wave.  (2048 logits in four waves, not one: 64 rows 4.4 -> 3.1 us, 4096 rows 15.9 -> 14.4)
    const int chunks = (vocab + 255) / 256;
    if (chunks <= 2) {
        LAUNCH_P(1, 2);
    } else if (chunks <= 4) {
        LAUNCH_P(1, 4);
    } else if (chunks <= 8) {
        LAUNCH_P(4, 2);
    } else if (chunks <= 16) {
        LAUNCH_P(4, 4);
    } else if (chunks <= 32) {
        LAUNCH_P(4, 8);
    } else if (chunks <= 64) {
        LAUNCH_P(8, 8);
    } else if (chunks <= 104) {
        LAUNCH_P(8, 13);
    } else if (chunks <= 208) {
        LAUNCH_P(16, 13);
    } else {
        hipLaunchKernelGGL(FinalProbabilitiesTwoPass, dim3(rows), dim3(256), 0, STREAM, vocab, (float *)logits->ptr, logits->strideBytes, bias, target,
            gradMult, (bf16_t *)grad->ptr, grad->strideBytes);
    }
#undef LAUNCH_P
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

// dst[t][x] = bf16(src[t][x]) for 8-bit src (exact), rows <= t < rowsRound zero; a lane converts 8 consecutive elements
template <class TSrc>
__global__ void __launch_bounds__(256) RowsToBf16(int rows, int rowsRound, int cols8, const uint8_t *src, int64_t ldSrc, uint8_t *dst, int64_t ldDst)
{
    const long total = (long)rowsRound * cols8;
    for (long u = (long)blockIdx.x * 256 + threadIdx.x; u < total; u += (long)gridDim.x * 256) {
        const int t = (int)(u / cols8), c = (int)(u % cols8);
        uint32_t out[4] = {0, 0, 0, 0};
        if (t < rows) {
            const uint2 in = *(const uint2 *)(src + (int64_t)t * ldSrc + c * 8);
            const uint32_t w[2] = {in.x, in.y};
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                float lo, hi;
                if (std::is_same<TSrc, TI8>::value) {
                    lo = (float)(int8_t)(w[e >> 2] >> (8 * (e & 3)));
                    hi = (float)(int8_t)(w[e >> 2] >> (8 * ((e + 1) & 3)));
                } else {
                    lo = (e & 3) == 0 ? __builtin_amdgcn_cvt_f32_fp8((int)w[e >> 2], 0) : __builtin_amdgcn_cvt_f32_fp8((int)w[e >> 2], 2);
                    hi = (e & 3) == 0 ? __builtin_amdgcn_cvt_f32_fp8((int)w[e >> 2], 1) : __builtin_amdgcn_cvt_f32_fp8((int)w[e >> 2], 3);
                }
                out[e >> 1] = PackBf16x2(lo, hi);
            }
        }
        *(uint4 *)(dst + (int64_t)t * ldDst + c * 16) = make_uint4(out[0], out[1], out[2], out[3]);
    }
}

int Ts2RowsToBf16(int rows, int rowsRound, int cols, const ts2_mat *src, int srcType, const ts2_mat *dst, void *stream)
{
    if ((cols & 7) || (src->strideBytes & 7) || (dst->strideBytes & 15) || ((uintptr_t)src->ptr & 7) || ((uintptr_t)dst->ptr & 15)) {
        return TS2_ERR_ALIGN;
    }
    const long total = (long)rowsRound * (cols / 8);
    const dim3 grid((unsigned)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192));
    if (srcType == TS2_I8) {
        hipLaunchKernelGGL((RowsToBf16<TI8>), grid, dim3(256), 0, STREAM, rows, rowsRound, cols / 8, (const uint8_t *)src->ptr, src->strideBytes,
            (uint8_t *)dst->ptr, dst->strideBytes);
    } else if (srcType == TS2_E4M3) {
        hipLaunchKernelGGL((RowsToBf16<TE4M3>), grid, dim3(256), 0, STREAM, rows, rowsRound, cols / 8, (const uint8_t *)src->ptr, src->strideBytes,
            (uint8_t *)dst->ptr, dst->strideBytes);
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2TransposeToBf16(int rows, int rowsRound, int cols, const ts2_mat *src, int srcType, const ts2_mat *dst, void *stream)
{
    dim3 grid((cols + 63) / 64, (rowsRound + 63) / 64);
    const uint8_t *s = (const uint8_t *)src->ptr;
    uint8_t *d = (uint8_t *)dst->ptr;
    if (srcType == TS2_I8) {
        hipLaunchKernelGGL((TransposeToBf16<TI8>), grid, dim3(256), 0, STREAM, rows, rowsRound, cols, s, src->strideBytes, d, dst->strideBytes);
    } else if (srcType == TS2_E4M3) {
        hipLaunchKernelGGL((TransposeToBf16<TE4M3>), grid, dim3(256), 0, STREAM, rows, rowsRound, cols, s, src->strideBytes, d, dst->strideBytes);
    } else if (srcType == TS2_BF16) {
        if (cols % 8 == 0 && rowsRound % 8 == 0 && src->strideBytes % 16 == 0 && dst->strideBytes % 16 == 0 && (uintptr_t)s % 16 == 0 &&
            (uintptr_t)d % 16 == 0) {
            hipLaunchKernelGGL(Transpose16, grid, dim3(256), 0, STREAM, rows, rowsRound, cols, s, src->strideBytes, d, dst->strideBytes);
        } else {
            hipLaunchKernelGGL((TransposeToBf16<TBF16>), grid, dim3(256), 0, STREAM, rows, rowsRound, cols, s, src->strideBytes, d, dst->strideBytes);
        }
    } else {
        return TS2_ERR_UNSUPPORTED;
    }
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

__global__ void FillFloatsKernel(float *p, int n, float v)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

int Ts2FillFloats(float *p, int n, float v, void *stream)
{
    hipLaunchKernelGGL(FillFloatsKernel, dim3((n + 255) / 256), dim3(256), 0, STREAM, p, n, v);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}

int Ts2ZeroRows(const ts2_mat *m, int rows, int rowBytes, void *stream)
{
    hipLaunchKernelGGL(ZeroBytes, dim3(rows), dim3(256), 0, STREAM, (uint8_t *)m->ptr, m->strideBytes, rowBytes);
    TS2_CHECK_LAUNCH();
    return TS2_OK;
}
