// The rows of a cosine-attention window block (2_Vision_Transformer/swin_transformer_v2.py:155-207) inside the attention kernels:
// q / |q| * scale_h and k / |k| in the 16-bit type, 16-byte chunks of eight channels, with the roundings of fb_cosine.hip one after
// the other (norm, quotient, product), so that the attention sees the bits that the separate pass would have stored.
//
// A pass of its own reads and writes q and k (forward), and reads q, k, dq, dk and writes dq, dk (backward): 225 and 357 us at 16 x 64
// windows of 256 tokens, 16 heads, bf16, bound by memory.  In the window forward it is 41 us of vector work (498 -> 539), in the ring
// backward 133 (867 -> 1000): training step of the block 3641 -> 3205 us; windows of 64 tokens 918 -> 880, of 144 (256 x 16) 647 -> 593;
// small grids, which lose two launches, 64 x 4 windows of 144 98 -> 81, 64 x 8 of 256 196 -> 153.
// There is no smallest grid: the ring kernel takes a (window, head) pair a workgroup, where the general kernels take two or four for windows of
// more than 128 tokens, but that is less than the passes and launches around them.  Normalisation, forward, backward and its normalisation,
// separate / inside, us, rank 16: 16 windows x 2 heads of 64 tokens 21.0 / 17.7, of 144 27.0 / 25.9, of 256 31.4 / 28.5; 16 x 4 21.5 / 17.9, 29.4 / 26.3,
// 34.2 / 29.4; 16 x 8 23.2 / 18.4, 35.1 / 27.2, 39.4 / 31.9; 32 x 4 24.0 / 18.3, 36.9 / 26.8, 43.0 / 31.3; with masks 16 x 4 31.1 / 19.8, 50.2 / 30.2, 54.2 / 34.8.
// Behind only at 4 x 2 without a mask, 25.1 / 25.8 and 26.4 / 28.1 (64 tokens 19.8 / 17.5), in graphs; an eager step of that size is 190 to 260 us of host.
#pragma once
#include "fb_device.h"

namespace fb {

constexpr float kLogitMax = 4.6052f; // (swin_transformer_v2.py:180: log of 100)
constexpr float kNormEps = 1e-12f;   // (torch.nn.functional.normalize)

// The logit scale of a window block: one value per head, in the element type `type` (fb_dtype).
struct LogitScale {
    const void *ptr; // null: the call is no cosine attention
    int type;
};

template <class SC>
__device__ __forceinline__ float scale_from(uint16_t x) { // (rounded to the parameter's type, the clamp's bound too)
    const float l = fminf(SC::to_float(x), SC::to_float(SC::from_float(kLogitMax)));
    return SC::to_float(SC::from_float(expf(l)));
}
__device__ __forceinline__ float scale_of_head(const LogitScale &s, int h) { // (h wave-uniform, and so the result, in a scalar register)
    float x;
    if (s.type == 2) {
        x = expf(fminf(static_cast<const float *>(s.ptr)[h], kLogitMax));
    } else {
        const uint16_t w = static_cast<const uint16_t *>(s.ptr)[h];
        x = s.type == 1 ? scale_from<BF16>(w) : scale_from<F16>(w);
    }
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x)));
}

template <class T>
__device__ __forceinline__ float round16(float x) { return T::to_float(T::from_float(x)); }

template <class T>
__device__ __forceinline__ void chunk_floats(u32x4_t w, float (&x)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x[2 * e] = T::to_float((uint16_t)(w[e] & 0xffffu));
        x[2 * e + 1] = T::to_float((uint16_t)(w[e] >> 16));
    }
}
template <class T>
__device__ __forceinline__ float chunk_squares(u32x4_t w) {
    float x[8], s = 0.f;
    chunk_floats<T>(w, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf(x[e], x[e], s);
    return s;
}

// What a row is divided by: max(|row|, eps).  The quotients, to be rounded to 16 bits, are formed from one reciprocal of the row (a
// division takes about ten instructions a value).  bf16: x and the denominator d have 8 significant bits, a tie t of the rounding 9, so
// x - t d is a multiple of its last place and x / d at least 2^-17 of itself away from t, while x * (1 / d) is within 2^-22 of it: the
// product rounds as the quotient does.  fp16 (11 and 12 bits, 2^-23): corrected by its own remainder, which rounds it to fp32 as a
// division does.  Where the denominator is infinite they are x * 0, as x / inf.
struct RowNorm {
    float norm, inv, denom; // (denom: 1 where it is infinite)
    template <class T>
    static __device__ __forceinline__ RowNorm of(float squares) {
        RowNorm r;
        r.norm = round16<T>(__builtin_sqrtf(squares));
        r.inv = 1.f / fmaxf(r.norm, round16<T>(kNormEps));
        r.template finish<T>();
        return r;
    }
    template <class T>
    __device__ __forceinline__ void finish() { // denom from norm
        denom = fmaxf(norm, round16<T>(kNormEps));
        denom = denom == INFINITY ? 1.f : denom;
    }
    template <class T>
    __device__ __forceinline__ float quotient(float x) const {
        const float q = x * inv;
        if constexpr (T::kWideRange) return q;
        return __builtin_fmaf(__builtin_fmaf(-denom, q, x), inv, q);
    }
};

// The unit vector's eight channels, as stored (k), and times the scale (q).
template <class T>
__device__ __forceinline__ u32x4_t chunk_unit(u32x4_t w, const RowNorm &r) {
    float x[8];
    chunk_floats<T>(w, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = T::pack2(r.template quotient<T>(x[2 * e]), r.template quotient<T>(x[2 * e + 1]));
    return w;
}
template <class T>
__device__ __forceinline__ u32x4_t chunk_times(u32x4_t w, float s) {
    float x[8];
    chunk_floats<T>(w, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = T::pack2(x[2 * e] * s, x[2 * e + 1] * s);
    return w;
}

// x of this lane + x of lane ^ 32.
__device__ __forceinline__ float half_wave_sum(float x) {
    float lo = x, hi = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
    return lo + hi;
}
// The sum over aligned groups of four lanes, (0 + 1) + (2 + 3).
__device__ __forceinline__ float quad_sum(float x) {
    x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true)); // lane ^ 1
    x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true)); // lane ^ 2
    return x;
}

// A row of 32 channels held by the lanes (c, 0) and (c, 1) as an MFMA operand (chunks 2 t + g): its unit vector.
template <class T>
__device__ __forceinline__ RowNorm unit_operand(u32x4_t (&x)[2]) {
    const float s0 = half_wave_sum(chunk_squares<T>(x[0])), s1 = half_wave_sum(chunk_squares<T>(x[1]));
    const RowNorm r = RowNorm::of<T>(s0 + s1);
    x[0] = chunk_unit<T>(x[0], r);
    x[1] = chunk_unit<T>(x[1], r);
    return r;
}

} // namespace fb
