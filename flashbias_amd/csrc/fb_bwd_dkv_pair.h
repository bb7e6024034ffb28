// dk, dv and dk_bias for head dims 65 ... 128 in one pass (aligned tensors, rank up to 32, no mask or a vector mask).
// Included by fb_bwd_dkv.hip after the general kernel, whose arithmetic it shares (lane = key, register = query).
//
// At these head dims the accumulators of dv and [dk | dk_bias] and the operands K, K_b, V of 32 keys do not fit one wave of
// 256 registers beside anything else, and two passes compute S and P twice (44 products a 32 x 32 block instead of
// 35).  Here two waves share a block of 32 keys: wave w < 4 forms S and P and sums dv (K, K_b and dv in registers, 17
// products), hands P over in fp32 through LDS, and wave w + 4 forms dP and dS and sums [dk | dk_bias] (V and dk in
// registers, 18 products) one block of queries later.  Both are on one SIMD, in different phases by construction.
//
// Blocks of 32 queries run through a ring of four LDS stages: the second waves' block, the first waves', the one that has
// landed and the one on its way; one barrier a block.
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKR_, int MASK_, bool FOLD_>
struct DkvPairCfg {
    static constexpr int NKD = 8, NKR = NKR_, NK = NKD + NKR_, NDV = 4, MB = 4 + (NKR_ > 0 ? 1 : 0);
    static constexpr bool FOLD = FOLD_, VMASK = MASK_ == kVectorMask;
    static_assert(MASK_ != kMatrixMask && !(FOLD_ && VMASK) && NKR_ <= 2, "");
    static constexpr int NWAVES = 8, NTHREADS = 64 * NWAVES, BN = 128, BMQ = 32;
    static constexpr int ROWCH = 16, CPR = 2 * (NKR > 0 ? NKR : 1);
    // a stage, bytes: Q and dO rows of 256, Q_b rows of 32 or 64, lse * log2(e) and -delta
    static constexpr int SQ = BMQ * 256, SQB = NKR > 0 ? BMQ * CPR * 16 : 0, STAGE = 2 * SQ + SQB + 8 * BMQ, NSTAGE = 4;
    static constexpr int P = NSTAGE * STAGE, LDS_BYTES = P + 4 * 2 * 4096; // two blocks of P for each pair
    static_assert(LDS_BYTES <= 160 * 1024, "");
    static __device__ __forceinline__ bool low_parts(const BwdArgs &a) { return FOLD_ && NKR_ == 1 && a.r <= 8 && a.scale != 1.f; }
};

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_dkv_pair_kernel(const BwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = lds_addr_of(smem);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), pair = wave & 3;

    // (one workgroup serves `group` consecutive batch entries of its (head, key tile), as the general kernel does)
    const int group = a.group > 1 ? a.group : 1;
    const int nbg = (a.B + group - 1) / group;
    int bgh, tile_n;
    work_order(blockIdx.x, a.ntiles_n, a.ntiles_n * nbg * a.H, a.causal, bgh, tile_n);
    const int bg = bgh / a.H, h = bgh % a.H;
    const int n0 = tile_n * C::BN, wk0 = n0 + 32 * pair;

    // clear the stages once: the zero padding of the channel dimension is never rewritten
    for (int i = threadIdx.x; i < C::P / 16; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem)[i] = u32x4_t{0u, 0u, 0u, 0u};
    __syncthreads();

    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e; // the scores are in units of 1 / scale when folded
    const int blk0 = a.causal ? n0 / C::BMQ : 0, nblk = (a.Lq + C::BMQ - 1) / C::BMQ; // causal: the first block that sees a key
    f32x16_t acc_b; // the second waves' dk_bias, summed over the group
#pragma unroll
    for (int v = 0; v < 16; ++v) acc_b[v] = 0.f;

    for (int bi = 0; bi < group; ++bi) {
        const int b = __builtin_amdgcn_readfirstlane(bg * group + bi);
        if (b >= a.B) break;
        int tid_again = threadIdx.x; // (opaque: what derives from the lane id is recomputed per entry, not kept in registers)
        asm volatile("" : "+v"(tid_again));
        const int lane = tid_again & 63, c = lane & 31, g = lane >> 5;
        const int bh = b * a.H + h, key = wk0 + c;

        // ---- copies: per block and wave one instruction (four rows) of Q and one of dO; waves 0 (1) Q_b, waves 4 and 5
        // the statistics
        TileDma<C::BMQ, C::ROWCH, C::NWAVES, false> cq, cd;
        DenseCopy<C::BMQ, C::CPR> cb;
        cq.init(a.q.ptr + b * a.q.sb + h * a.q.sh, a.q.ss, a.d, C::ROWCH, nullptr, 0, 0, wave, lane, blk0 * C::BMQ);
        cd.init(a.dout.ptr + b * a.dout.sb + h * a.dout.sh, a.dout.ss, a.d, C::ROWCH, nullptr, 0, 0, wave, lane, blk0 * C::BMQ);
        if constexpr (C::NKR > 0) cb.init(a.qb.ptr + b * a.qb.sb + h * a.qb.sh, a.qb.ss, a.r, C::low_parts(a), wave, lane, blk0 * C::BMQ);
        const float *stat = a.delta + ((wave == 4 ? (int64_t)a.B * a.H : 0) + bh) * a.Lq; // lse * log2(e), -delta
        constexpr int QB_WAVES = C::NKR > 0 ? decltype(cb)::NINST : 0;
        auto issue = [&](int blk) { // (in sequence)
            const uint32_t at = lds0 + ((blk - blk0) & 3) * C::STAGE;
            const int r0 = blk * C::BMQ;
            cq.issue(at, r0, a.Lq, a.q.ss, 0, C::ROWCH);
            cd.issue(at + C::SQ, r0, a.Lq, a.dout.ss, 0, C::ROWCH);
            if constexpr (C::NKR > 0) cb.issue(at + 2 * C::SQ, r0, a.Lq);
            if ((wave == 4 || wave == 5) && lane < C::BMQ)
                lds_dma4(stat + min(r0 + lane, a.Lq - 1), at + 2 * C::SQ + C::SQB + (wave - 4) * 4 * C::BMQ);
        };
        auto landed = [&](bool newest_may_fly) { // this wave's copies, but for the newest block's
            if (!newest_may_fly)
                wait_vmcnt<0>();
            else if (wave < QB_WAVES || wave == 4 || wave == 5)
                wait_vmcnt<3>();
            else
                wait_vmcnt<2>();
        };
        // One turn of the ring: blk + 2 is requested, `work` runs, blk + 1 has landed for everyone.
        auto turn = [&](int blk, auto work) {
            if (blk + 2 < nblk) issue(blk + 2);
            work();
            landed(blk + 2 < nblk);
            barrier_lds();
        };
        if (blk0 < nblk) issue(blk0);
        if (blk0 + 1 < nblk) issue(blk0 + 1);

        const bool real = wk0 < a.Lk;
        const uint32_t pbuf = C::P + pair * 8192 + lane * 16;
        if (wave < 4) {
            // ---- S, P and dv
            u32x4_t kr[C::NK]; // B operand of S: this lane's key
            const uint16_t *kbase = a.k.ptr + b * a.k.sb + h * a.k.sh;
#pragma unroll
            for (int t = 0; t < C::NKD; ++t) kr[t] = load_chunk<true>(kbase, a.k.ss, key, a.Lk, 16 * t + 8 * g, a.d);
            if constexpr (C::NKR > 0) {
                const uint16_t *kbbase = a.kb.ptr + b * a.kb.sb + h * a.kb.sh;
                const bool low = C::low_parts(a) && g == 1;
#pragma unroll
                for (int t = 0; t < C::NKR; ++t) {
                    u32x4_t x = load_chunk<true>(kbbase, a.kb.ss, key, a.Lk, low ? 0 : 16 * t + 8 * g, a.r);
                    if (C::FOLD && a.scale != 1.f) x = fold_scale_chunk<T>(x, 1.f / a.scale, C::low_parts(a), low);
                    kr[C::NKD + t] = x;
                }
            }
            float mkey = 0.f; // vector mask: the value of this lane's key
            if constexpr (C::VMASK) {
                const int64_t at = mask_offset(a.mask, b, h) + min(key, a.Lk - 1);
                mkey = a.mask.is_f32 ? reinterpret_cast<const float *>(a.mask.ptr)[at] : T::to_float(reinterpret_cast<const uint16_t *>(a.mask.ptr)[at]);
            }
            f32x16_t acc[C::NDV];
#pragma unroll
            for (int n = 0; n < C::NDV; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
            landed(blk0 + 1 < nblk);
            barrier_lds();
#pragma unroll 1
            for (int blk = blk0; blk <= nblk; ++blk)
                turn(blk, [&]() {
                    const int r0 = blk * C::BMQ;
                    if (blk == nblk || !real || (a.causal && wk0 > r0 + 31)) return;
                    const uint8_t *st = smem + ((blk - blk0) & 3) * C::STAGE;
                    TileAddr16 ta(lds_addr_of(st), c, g);
                    asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                    f32x16_t s;
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[v] = 0.f;
                    __builtin_amdgcn_s_setprio(1);
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) s = T::mfma(ta.load_row(t, 0), kr[t], s);
                    // the softmax scale multiplies the fp32 q k^T accumulator before the bias steps
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[v] = C::VMASK ? __builtin_fmaf(s[v], a.scale, mkey) : s[v] * a.scale;
                    }
                    if constexpr (C::NKR > 0) {
#pragma unroll
                        for (int t = 0; t < C::NKR; ++t)
                            s = T::mfma(*reinterpret_cast<const u32x4_t *>(st + 2 * C::SQ + lean_row_addr<C::CPR>(c, 2 * t + g)), kr[C::NKD + t], s);
                    }
                    __builtin_amdgcn_s_setprio(0);
                    // (bitwise on purpose, as in the dq kernel: no scalar block between the last MFMA and the branch)
                    const bool edge = (wk0 + 32 > a.Lk) | (r0 + 32 > a.Lq) | ((a.causal != 0) & (wk0 + 31 > r0));
                    if (edge) {
                        int query0 = r0 + 4 * g;
                        asm volatile("" : "+v"(query0)); // (computed here, not kept in registers across the loop)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int query = query0 + 8 * (v >> 2) + (v & 3);
                            if (key >= a.Lk || query >= a.Lq || (a.causal && key > query)) s[v] = -INFINITY;
                        }
                    }
                    asm volatile("s_nop 11" : "+v"(s)); // (fb_bwd_win.hip: wait states across the branch above)
                    const float *lse2 = reinterpret_cast<const float *>(st + 2 * C::SQ + C::SQB) + 4 * g;
                    u32x4_t pp[2];
#pragma unroll
                    for (int j = 0; j < 4; ++j) { // register v <-> query r0 + 8 (v / 4) + 4 g + v % 4
                        const f32x4_t l = *reinterpret_cast<const f32x4_t *>(lse2 + 8 * j);
                        f32x4_t p;
#pragma unroll
                        for (int e = 0; e < 4; ++e) p[e] = fast_exp2(__builtin_fmaf(s[4 * j + e], to_log2, -l[e]));
                        *reinterpret_cast<f32x4_t *>(smem + pbuf + (blk & 1) * 4096 + j * 1024) = p;
                        pp[j >> 1][2 * (j & 1)] = T::pack2(p[0], p[1]);
                        pp[j >> 1][2 * (j & 1) + 1] = T::pack2(p[2], p[3]);
                    }
                    __builtin_amdgcn_s_setprio(1);
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int n = 0; n < C::NDV; ++n) acc[n] = T::mfma(ta.load_tr(n, C::SQ + 16 * 256 * t), pp[t], acc[n]);
                    __builtin_amdgcn_s_setprio(0);
                });
            const bool ok = key < a.Lk;
            uint16_t *row = const_cast<uint16_t *>(a.dv.ptr) + b * a.dv.sb + h * a.dv.sh + (int64_t)(ok ? key : 0) * a.dv.ss;
#pragma unroll
            for (int n = 0; n < C::NDV; ++n) {
                asm volatile("s_nop 11" : "+v"(acc[n]));
                store_acc_rows<T, true>(row + 32 * n, ok, a.dv.vec_ok, acc[n], 1.f, a.d - 32 * n, g);
            }
        } else {
            // ---- dP, dS and [dk | dk_bias], one block behind
            u32x4_t vr[C::NKD]; // B operand of dP
            const uint16_t *vbase = a.v.ptr + b * a.v.sb + h * a.v.sh;
#pragma unroll
            for (int t = 0; t < C::NKD; ++t) vr[t] = load_chunk<true>(vbase, a.v.ss, key, a.Lk, 16 * t + 8 * g, a.d);
            f32x16_t acc[4];
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
            landed(blk0 + 1 < nblk);
            barrier_lds();
#pragma unroll 1
            for (int next = blk0; next <= nblk; ++next)
                turn(next, [&]() {
                    const int blk = next - 1;
                    if (blk < blk0 || !real || (a.causal && wk0 > blk * C::BMQ + 31)) return;
                    const uint8_t *st = smem + ((blk - blk0) & 3) * C::STAGE;
                    TileAddr16 ta(lds_addr_of(st), c, g);
                    asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                    f32x16_t dp; // -delta is the initial value
                    const float *negd = reinterpret_cast<const float *>(st + 2 * C::SQ + C::SQB) + C::BMQ + 4 * g;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(negd + 8 * j);
#pragma unroll
                        for (int e = 0; e < 4; ++e) dp[4 * j + e] = x[e];
                    }
                    __builtin_amdgcn_s_setprio(1);
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) dp = T::mfma(ta.load_row(t, C::SQ), vr[t], dp);
                    __builtin_amdgcn_s_setprio(0);
                    u32x4_t ds[2];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t p = *reinterpret_cast<const f32x4_t *>(smem + pbuf + (blk & 1) * 4096 + j * 1024);
                        ds[j >> 1][2 * (j & 1)] = T::pack2(p[0] * dp[4 * j], p[1] * dp[4 * j + 1]);
                        ds[j >> 1][2 * (j & 1) + 1] = T::pack2(p[2] * dp[4 * j + 2], p[3] * dp[4 * j + 3]);
                    }
                    __builtin_amdgcn_s_setprio(1);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
#pragma unroll
                        for (int n = 0; n < 4; ++n) acc[n] = T::mfma(ta.load_tr(n, 16 * 256 * t), ds[t], acc[n]);
                        if constexpr (C::NKR > 0) acc_b = T::mfma(dense_read_a_tr<C::CPR>(st + 2 * C::SQ, 16 * t, c, g), ds[t], acc_b);
                    }
                    __builtin_amdgcn_s_setprio(0);
                });
            const bool ok = key < a.Lk;
            uint16_t *row = const_cast<uint16_t *>(a.dk.ptr) + b * a.dk.sb + h * a.dk.sh + (int64_t)(ok ? key : 0) * a.dk.ss;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                asm volatile("s_nop 11" : "+v"(acc[n]));
                store_acc_rows<T, true>(row + 32 * n, ok, a.dk.vec_ok, acc[n], a.scale, a.d - 32 * n, g);
            }
        }
    }
    if constexpr (C::NKR > 0) {
        if (wave >= 4 && a.dkb.ptr) { // (null: the caller does not want the factor gradients)
            const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
            const int key = wk0 + (lane & 31);
            const bool ok = key < a.Lk;
            asm volatile("s_nop 11" : "+v"(acc_b));
            uint16_t *row = const_cast<uint16_t *>(a.dkb.ptr) + bg * a.dkb.sb + h * a.dkb.sh + (int64_t)(ok ? key : 0) * a.dkb.ss;
            store_acc_rows<T, true>(row, ok, a.dkb.vec_ok, acc_b, 1.f, a.r, lane >> 5);
        }
    }
}

template <class T, int NKR, int MASK, bool FOLD>
static hipError_t launch_dkv_pair(const BwdArgs &a0, hipStream_t stream) {
    typedef DkvPairCfg<T, NKR, MASK, FOLD> C;
    BwdArgs a = a0;
    a.ntiles_n = (a.Lk + C::BN - 1) / C::BN;
    auto kern = bwd_dkv_pair_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    const int group = a.group > 1 ? a.group : 1;
    return launch_flat(kern, (int64_t)a.ntiles_n * ((a.B + group - 1) / group) * a.H, C::NTHREADS, C::LDS_BYTES, stream, a);
}

} // namespace fb
