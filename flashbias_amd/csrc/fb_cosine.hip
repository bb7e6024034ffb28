// The elementwise part of a cosine-attention window block (2_Vision_Transformer/swin_transformer_v2.py:155-207)
// around the attention kernels: forward, the packed projection (tokens, 3, H, d) becomes
// q = q / |q| * scale_h and k = k / |k| in the attention's 16-bit type (and v, where the projection has another
// type); backward, the attention's gradients become that of the packed projection and of the per-head logit scale,
// scale_h = exp(min(logit_scale_h, 4.6052)).
//
// Memory-bound: one pass over q and k in each direction (backward: q, k, dq, dk in, both gradients out), 16 bytes per
// lane and tensor, a head's row spread over d / 8 neighbouring lanes whose sums meet by lane exchanges.  Every thread
// keeps its head and channels for all the tokens it walks, so the scale is read once and the logit scale's gradient
// is one running sum per thread; its last step is a small kernel of one workgroup per head, in a fixed order.
// As tensor operations the same work took about 40 passes over tensors of that size (16 x 64 windows of 256 tokens, 16
// heads of 32 channels, bf16, forward + backward: 7.4 of the module's 12.7 ms).
//
// Rounding (fb_cosine.fp32 == 0): the type of the packed projection is also the type that tensor operations compute in,
// which round the norm, the quotient and the product to it one after the other; these kernels do the same, so that q and
// k are those of the tensor operations.  Under autocast (fb_cosine.fp32 != 0) the projection has 16 bits while tensor
// operations keep norm, quotient, exponential and product in fp32 and round once, and so do these kernels: with the
// roundings in between, scaled q would be off by 2.9e-3 instead of 1.7e-3 of its norm, on cosines that the scale
// multiplies by 10 and more.  The backward rounds its results only.
#include "flashbias.h"
#include "fb_kernels.h"
#include "fb_unit.h"

namespace fb {

struct F32 {}; // 32-bit floats, beside BF16 and F16

template <class T>
struct Io { // 8 consecutive elements of a 16-bit type
    static __device__ __forceinline__ void load(const void *p, int64_t i, float (&x)[8]) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t *>(static_cast<const uint16_t *>(p) + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[2 * e] = T::to_float((uint16_t)(w[e] & 0xffffu));
            x[2 * e + 1] = T::to_float((uint16_t)(w[e] >> 16));
        }
    }
    static __device__ __forceinline__ void store(void *p, int64_t i, const float (&x)[8]) {
        *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(p) + i) =
            u32x4_t{T::pack2(x[0], x[1]), T::pack2(x[2], x[3]), T::pack2(x[4], x[5]), T::pack2(x[6], x[7])};
    }
    static __device__ __forceinline__ float round(float x) { return T::to_float(T::from_float(x)); }
    static __device__ __forceinline__ float load1(const void *p, int64_t i) { return T::to_float(static_cast<const uint16_t *>(p)[i]); }
    static __device__ __forceinline__ void store1(void *p, int64_t i, float x) { static_cast<uint16_t *>(p)[i] = T::from_float(x); }
};
template <>
struct Io<F32> {
    static __device__ __forceinline__ void load(const void *p, int64_t i, float (&x)[8]) {
        const f32x4_t *w = reinterpret_cast<const f32x4_t *>(static_cast<const float *>(p) + i);
        const f32x4_t a = w[0], b = w[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = a[e];
            x[4 + e] = b[e];
        }
    }
    static __device__ __forceinline__ void store(void *p, int64_t i, const float (&x)[8]) {
        f32x4_t *w = reinterpret_cast<f32x4_t *>(static_cast<float *>(p) + i);
        w[0] = f32x4_t{x[0], x[1], x[2], x[3]};
        w[1] = f32x4_t{x[4], x[5], x[6], x[7]};
    }
    static __device__ __forceinline__ float round(float x) { return x; }
    static __device__ __forceinline__ float load1(const void *p, int64_t i) { return static_cast<const float *>(p)[i]; }
    static __device__ __forceinline__ void store1(void *p, int64_t i, float x) { static_cast<float *>(p)[i] = x; }
};

struct CosineArgs {
    const void *x, *logit_scale;
    void *q, *k, *v;
    const void *dq, *dk, *dv;
    void *dx, *dlogit_scale;
    float *partial;
    int64_t tokens, grad_ss;
    int H, d;
    int sweep; // tokens per step of the grid
};

__device__ __forceinline__ float sum_over(float x, int lanes) { // over aligned groups of `lanes` (a power of two)
    for (int m = 1; m < lanes; m <<= 1) x += __shfl_xor(x, m, 64);
    return x;
}

// FP32: nothing is rounded in between (the bound of the clamp stays a number of the parameter's type).
template <class X, bool FP32>
__device__ __forceinline__ float step(float x) {
    return FP32 ? x : Io<X>::round(x);
}

template <class SC, bool FP32>
__device__ __forceinline__ float logit_scale_of(const CosineArgs &a, int h) {
    const float l = Io<SC>::load1(a.logit_scale, h);
    return step<SC, FP32>(expf(fminf(l, Io<SC>::round(kLogitMax))));
}

// The unit vector of the lane group's row, rounded as the tensor operations round it; returns what it is divided by.
template <class IN, bool FP32>
__device__ __forceinline__ float normalise(float (&x)[8], int lanes, float &norm) {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf(x[e], x[e], s);
    norm = step<IN, FP32>(__builtin_sqrtf(sum_over(s, lanes)));
    const float denom = fmaxf(norm, step<IN, FP32>(kNormEps));
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = step<IN, FP32>(x[e] / denom);
    return denom;
}

// The product with the scale is formed in the wider of the two types.
template <class IN, class SC, bool FP32>
__device__ __forceinline__ float times_scale(float x, float s) {
    return __is_same(IN, SC) ? step<IN, FP32>(x * s) : x * s;
}

template <class IN, class OUT, class SC, bool FP32>
__global__ __launch_bounds__(256) void cosine_fwd_kernel(const CosineArgs a) {
    const int lanes = a.d / 8, chunks = a.H * lanes;
    const int idx = blockIdx.x * 256 + threadIdx.x, col = idx % chunks, first = idx / chunks;
    if (first >= a.sweep) return;
    const int h = col / lanes;
    const float s = logit_scale_of<SC, FP32>(a, h);
    const int64_t row = (int64_t)a.H * a.d;
    for (int64_t t = first; t < a.tokens; t += a.sweep) {
        float q[8], k[8], v[8], norm;
        Io<IN>::load(a.x, 3 * row * t + 8 * col, q);
        Io<IN>::load(a.x, 3 * row * t + row + 8 * col, k);
        if (a.v) Io<IN>::load(a.x, 3 * row * t + 2 * row + 8 * col, v);
        normalise<IN, FP32>(q, lanes, norm);
        normalise<IN, FP32>(k, lanes, norm);
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = times_scale<IN, SC, FP32>(q[e], s);
        Io<OUT>::store(a.q, row * t + 8 * col, q);
        Io<OUT>::store(a.k, row * t + 8 * col, k);
        if (a.v) Io<OUT>::store(a.v, row * t + 8 * col, v);
    }
}

// d/dx of x / |x| applied to the gradient g of the unit vector n: (g - n (n . g)) / |x|.
__device__ __forceinline__ void project(float (&g)[8], const float (&n)[8], int lanes, float norm, float denom) {
    float dot = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(g[e], n[e], dot);
    dot = sum_over(dot, lanes);
    if (norm < denom) dot = 0.f; // (a row of zeros: the clamped denominator is a constant)
    const float inv = 1.f / denom;
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = (g[e] - n[e] * dot) * inv;
}

template <class IN, class OUT, class SC, bool FP32>
__global__ __launch_bounds__(256) void cosine_bwd_kernel(const CosineArgs a) {
    const int lanes = a.d / 8, chunks = a.H * lanes;
    const int idx = blockIdx.x * 256 + threadIdx.x, col = idx % chunks, first = idx / chunks;
    if (first >= a.sweep) return;
    const int h = col / lanes;
    const float s = logit_scale_of<SC, FP32>(a, h);
    const int64_t row = (int64_t)a.H * a.d;
    float sum = 0.f;
    for (int64_t t = first; t < a.tokens; t += a.sweep) {
        const int64_t at = 3 * row * t + 8 * col, from = a.grad_ss * t + 8 * col;
        float q[8], k[8], gq[8], gk[8], qn, kn;
        Io<IN>::load(a.x, at, q);
        Io<IN>::load(a.x, at + row, k);
        Io<OUT>::load(a.dq, from, gq);
        Io<OUT>::load(a.dk, from, gk);
        if (a.dv) {
            float gv[8];
            Io<OUT>::load(a.dv, from, gv);
            Io<IN>::store(a.dx, at + 2 * row, gv);
        }
        const float dq = normalise<IN, FP32>(q, lanes, qn), dk = normalise<IN, FP32>(k, lanes, kn);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sum = __builtin_fmaf(gq[e], q[e], sum);
            gq[e] *= s;
        }
        project(gq, q, lanes, qn, dq);
        project(gk, k, lanes, kn, dk);
        Io<IN>::store(a.dx, at, gq); // (may be where dq and dk were read from)
        Io<IN>::store(a.dx, at + row, gk);
    }
    sum = sum_over(sum, lanes);
    if (col % lanes == 0) a.partial[(int64_t)h * a.sweep + first] = sum;
}

template <class SC, bool FP32>
__global__ __launch_bounds__(256) void cosine_scale_grad_kernel(const CosineArgs a) {
    __shared__ float part[256];
    const int h = blockIdx.x, tid = threadIdx.x;
    float s = 0.f;
    for (int i = tid; i < a.sweep; i += 256) s += a.partial[(int64_t)h * a.sweep + i];
    part[tid] = s;
    for (int n = 128; n > 0; n >>= 1) {
        __syncthreads();
        if (tid < n) part[tid] += part[tid + n];
    }
    if (tid == 0) {
        const bool inside = Io<SC>::load1(a.logit_scale, h) <= Io<SC>::round(kLogitMax);
        Io<SC>::store1(a.dlogit_scale, h, inside ? part[0] * logit_scale_of<SC, FP32>(a, h) : 0.f);
    }
}

// Workgroups: enough for every thread to have one token, at most eight per compute unit (all the waves it holds),
// which then walk the tokens.
static int cosine_blocks(int64_t tokens, int chunks) {
    const int64_t all = (tokens * chunks + 255) / 256, most = 8 * (int64_t)num_cus(), least = (chunks + 255) / 256;
    return (int)(all < least ? least : all < most ? all : most < least ? least : most);
}

int64_t cosine_sweep(int64_t tokens, int H, int d) {
    const int chunks = H * (d / 8);
    return (int64_t)cosine_blocks(tokens, chunks) * 256 / chunks;
}

template <class IN, class OUT, class SC, bool FP32>
static hipError_t launch_cosine_t(const CosineArgs &a, bool backward, hipStream_t stream) {
    const int blocks = cosine_blocks(a.tokens, a.H * (a.d / 8));
    if (!backward) return launch_flat(cosine_fwd_kernel<IN, OUT, SC, FP32>, blocks, 256, 0, stream, a);
    const hipError_t e = launch_flat(cosine_bwd_kernel<IN, OUT, SC, FP32>, blocks, 256, 0, stream, a);
    if (e != hipSuccess) return e;
    return launch_flat(cosine_scale_grad_kernel<SC, FP32>, a.H, 256, 0, stream, a);
}

template <class IN, class OUT, class SC>
static hipError_t launch_cosine_p(const CosineArgs &a, bool fp32, bool backward, hipStream_t stream) {
    return fp32 ? launch_cosine_t<IN, OUT, SC, true>(a, backward, stream) : launch_cosine_t<IN, OUT, SC, false>(a, backward, stream);
}

template <class IN, class OUT>
static hipError_t launch_cosine_s(const CosineArgs &a, int scale_type, bool fp32, bool backward, hipStream_t stream) {
    switch (scale_type) {
    case FB_F16: return launch_cosine_p<IN, OUT, F16>(a, fp32, backward, stream);
    case FB_BF16: return launch_cosine_p<IN, OUT, BF16>(a, fp32, backward, stream);
    default: return launch_cosine_p<IN, OUT, F32>(a, fp32, backward, stream);
    }
}

hipError_t launch_cosine(const fb_cosine *p, bool fp32, bool backward, hipStream_t stream) {
    CosineArgs a;
    a.x = p->qkv;
    a.logit_scale = p->logit_scale;
    a.q = p->q;
    a.k = p->k;
    a.v = p->v;
    a.dq = p->dq;
    a.dk = p->dk;
    a.dv = p->dv;
    a.dx = p->dqkv;
    a.dlogit_scale = p->dlogit_scale;
    a.partial = p->partial;
    a.tokens = p->tokens;
    a.grad_ss = p->grad_stride;
    a.H = p->H;
    a.d = p->d;
    a.sweep = (int)cosine_sweep(p->tokens, p->H, p->d);
    const bool bf16 = p->dtype == FB_BF16;
    switch (p->in_dtype) {
    case FB_F16: return bf16 ? launch_cosine_s<F16, BF16>(a, p->scale_dtype, fp32, backward, stream) : launch_cosine_s<F16, F16>(a, p->scale_dtype, fp32, backward, stream);
    case FB_BF16: return bf16 ? launch_cosine_s<BF16, BF16>(a, p->scale_dtype, fp32, backward, stream) : launch_cosine_s<BF16, F16>(a, p->scale_dtype, fp32, backward, stream);
    default: return bf16 ? launch_cosine_s<F32, BF16>(a, p->scale_dtype, fp32, backward, stream) : launch_cosine_s<F32, F16>(a, p->scale_dtype, fp32, backward, stream);
    }
}

// The logit scale's gradient from `shares` partial sums a head (the ring backward's).
hipError_t launch_cosine_scale_grad(const fb_cosine *p, int shares, hipStream_t stream) {
    CosineArgs a = {};
    a.logit_scale = p->logit_scale;
    a.dlogit_scale = p->dlogit_scale;
    a.partial = p->partial;
    a.sweep = shares;
    switch (p->scale_dtype) {
    case FB_F16: return launch_flat(cosine_scale_grad_kernel<F16, false>, p->H, 256, 0, stream, a);
    case FB_BF16: return launch_flat(cosine_scale_grad_kernel<BF16, false>, p->H, 256, 0, stream, a);
    default: return launch_flat(cosine_scale_grad_kernel<F32, false>, p->H, 256, 0, stream, a);
    }
}

} // namespace fb
