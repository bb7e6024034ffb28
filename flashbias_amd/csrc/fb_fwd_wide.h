// Forward for head dims 33 ... 128 on aligned tensors (rank up to 32, no mask or a vector mask).  Included by fb_fwd.hip
// after the general kernel, whose arithmetic it shares (one query per lane, S^T = [K | K_b] [Q | Q_b]^T, online softmax
// against a lagging reference point, O^T += V^T P^T, P from registers).
//
// What differs is how tiles reach the matrix cores.  At these head dims the general kernel's loader, which takes K and V
// through registers and transposes V on the way into LDS, is what a tile's time goes into: the transposing stores meet
// in few banks, its stage takes about 40 registers (at head dim 128 the kernel spilled at 256), and K fragments are
// requested one MFMA ahead.  Here global_load_lds copies [K], [K_b] and [V] row-major into two stages, one tile ahead,
// V^T fragments come from transposing LDS reads, and no register holds a tile.
//
// Left to itself the compiler asks for two K fragments and waits for them, once a contraction step: at head dim 128 nine times a
// tile of 64 keys, whose 34 products take 1088 cycles.  Here the order is fixed: fragments two steps ahead of their
// products, the first columns of V with the last of them, addresses from two registers (240 -> 212 of them at head dim
// 128, 147 -> 134 at 64).  us, before and after: causal B4 H32 L=4096 d128 r8 625 -> 610, B2 H8 L=1500 d128 r16 37.0 -> 35.0, B1 H4 L=999
// d128 27.1 -> 24.8; d64 causal B2 H8 L=4096 r8 68.3 -> 62.0, r2 as 16 B2 H16 L=2048 45.2 -> 40.8, B1 H4 L=1000 r32 19.7 -> 18.8, B4 H16
// L=2048 r8 92.6 -> 89.3.  What is left is products and exponentials of two waves that overlap in part.  Not kept: four waves a SIMD
// at head dim 64 (spills: causal 64 -> 78, masked 44 -> 84).
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKD_, int NKR_, int NDV_, int MASK_, bool FOLD_, int SPLIT_>
struct FwdWideCfg {
    static constexpr int NKD = NKD_, NKR = NKR_, NDV = NDV_, NK = NKD_ + NKR_;
    static constexpr bool VMASK = MASK_ == kVectorMask, FOLD = FOLD_;
    static_assert(MASK_ != kMatrixMask && !(FOLD_ && VMASK), "");
    static constexpr int SPLIT = SPLIT_, NWAVES = 4, NTHREADS = 64 * NWAVES * SPLIT; // (NWAVES: of a group)
    static constexpr int BM = 32 * NWAVES;
    static constexpr int KBLK = 2, BN = 32 * KBLK;
    static constexpr int ROWCH = 2 * NKD, CPR = 2 * NKR; // 16-byte chunks per row of K and V, of K_b
    static constexpr int SK = BN * ROWCH * 8, SKB = BN * CPR * 8, SM = VMASK ? 2 * BN : 0;
    static constexpr int STAGE = 2 * SK + SKB + SM; // elements: K, V, K_b, fp32 vector mask
    static constexpr int LDS_BYTES = 2 * STAGE * 2 * SPLIT;
    static_assert(LDS_BYTES <= 160 * 1024 && (SPLIT == 1 || LDS_BYTES >= NDV_ * 16384 + 4 * 512), "");
    // head dim <= 64: three workgroups per compute unit (168 registers, 3 x 40 KB)
    static constexpr int WAVES_EU = NKD <= 4 && SPLIT == 1 ? 3 : 2;
    // Exponentials before another wave's products.  us, against the products first: causal B4 H32 L=4096 d128 629 -> 610, fp16 d64
    // r16 8 x 8 x (1000 x 1500) with a padding mask 44.6 -> 43.9; without a mask at head dim 64 neither (causal B2 H8 L=4096
    // 62.0, products first 63.7, exponentials first 66.3).
    static constexpr bool EXP_FIRST = NKD > 4 || VMASK;
    static __device__ __forceinline__ bool low_parts(const FwdArgs &a) { return FOLD_ && NKR_ == 1 && a.r <= 8 && a.scale != 1.f; }
};

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void fwd_wide_kernel(const FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int grp = C::SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8); // takes its share of the tiles of keys, in stages of its own
    uint16_t *stage0 = reinterpret_cast<uint16_t *>(smem) + grp * 2 * C::STAGE;
    const int tid = threadIdx.x & (64 * C::NWAVES - 1), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, g = lane >> 5;

    const int total = a.ntiles_m * a.B * a.H;
    int bh, tile_m;
    work_order(blockIdx.x, a.ntiles_m, total, a.causal, bh, tile_m);
    if (a.causal) tile_m = a.ntiles_m - 1 - tile_m; // the last query tile sees the most keys
    const int b = bh / a.H, h = bh % a.H;
    const int m0 = tile_m * C::BM, wq0 = m0 + wave * 32;
    const int query = wq0 + c;

    const uint16_t *qbase = a.q.ptr + b * a.q.sb + h * a.q.sh;
    const uint16_t *kbase = a.k.ptr + b * a.k.sb + h * a.k.sh;
    const uint16_t *vbase = a.v.ptr + b * a.v.sb + h * a.v.sh;

    int k_end = a.Lk;
    if (a.causal && m0 + C::BM < k_end) k_end = m0 + C::BM;
    const int ntiles = (k_end + C::BN - 1) / C::BN, walk = (ntiles + C::SPLIT - 1) / C::SPLIT, tile0 = grp * walk;

    u32x4_t qr[C::NK];
#pragma unroll
    for (int t = 0; t < C::NKD; ++t) qr[t] = load_chunk<true>(qbase, a.q.ss, query, a.Lq, 16 * t + 8 * g, a.d);
    DenseCopy<C::BN, C::NKR ? C::CPR : 2> kbd; // K_b rows, one copy instruction of the first waves per tile
    if constexpr (C::NKR > 0) {
        const uint16_t *qbbase = a.qb.ptr + b * a.qb.sb + h * a.qb.sh;
        const bool low = C::low_parts(a) && g == 1;
#pragma unroll
        for (int t = 0; t < C::NKR; ++t) {
            u32x4_t x = load_chunk<true>(qbbase, a.qb.ss, query, a.Lq, low ? 0 : 16 * t + 8 * g, a.r);
            if (C::FOLD && a.scale != 1.f) x = fold_scale_chunk<T>(x, 1.f / a.scale, C::low_parts(a), low);
            qr[C::NKD + t] = x;
        }
        kbd.init(a.kb.ptr + b * a.kb.sb + h * a.kb.sh, a.kb.ss, a.r, C::low_parts(a), wave, lane, tile0 * C::BN);
    }
    f32x16_t acc_o[C::NDV];
#pragma unroll
    for (int n = 0; n < C::NDV; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc_o[n][v] = 0.f;
    float m_ref = -INFINITY, m2 = 0.f, l_run = 0.f; // (as in fwd_body)
    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e;
    const float lag = 8.0f / to_log2;

    {   // clear the stages once: the zero padding of the channel dimension is never rewritten
        u32x4_t *z = reinterpret_cast<u32x4_t *>(smem);
        for (int i = threadIdx.x; i < C::LDS_BYTES / 16; i += C::NTHREADS) z[i] = u32x4_t{0u, 0u, 0u, 0u};
    }
    __syncthreads();

    TileDma<C::BN, C::ROWCH, C::NWAVES, false> kd, vd;
    kd.init(kbase, a.k.ss, a.d, C::ROWCH, nullptr, 0, 0, wave, lane, tile0 * C::BN);
    vd.init(vbase, a.v.ss, a.d, C::ROWCH, nullptr, 0, 0, wave, lane, tile0 * C::BN);
    auto issue = [&](int buf, int n0) {
        const uint32_t base = lds_addr_of(stage0 + buf * C::STAGE);
        kd.issue(base, n0, a.Lk, a.k.ss, 0, C::ROWCH);
        if constexpr (C::NKR > 0) kbd.issue(base + 4 * C::SK, n0, a.Lk);
        vd.issue_or_zero(base + 2 * C::SK, n0, a.Lk, a.v.ss);
    };
    // Vector mask: thread `tid` carries the value of key n0 + tid of the tile that follows.
    float mkey = 0.f;
    auto load_vmask = [&](int n0) {
        const int key = min(n0 + (tid & (C::BN - 1)), a.Lk - 1); // (past the end: the score is set to -inf below)
        const uint8_t *mbase = reinterpret_cast<const uint8_t *>(a.mask.ptr) + mask_offset(a.mask, b, h) * (a.mask.is_f32 ? 4 : 2);
        mkey = a.mask.is_f32 ? reinterpret_cast<const float *>(mbase)[key] : T::to_float(reinterpret_cast<const uint16_t *>(mbase)[key]);
    };
    auto store_vmask = [&](int buf) {
        if (tid < C::BN) reinterpret_cast<float *>(stage0 + buf * C::STAGE + 2 * C::SK + C::SKB)[tid] = mkey;
    };
    if (C::SPLIT == 1 || tile0 < ntiles) {
        issue(0, tile0 * C::BN);
        if constexpr (C::VMASK) {
            load_vmask(tile0 * C::BN);
            store_vmask(0);
        }
    }
    wait_vmcnt<0>();
    barrier_lds();

    for (int it = 0; it < walk; ++it) {
        const int cur = it & 1, n0 = (tile0 + it) * C::BN;
        const bool more = it + 1 < walk && (C::SPLIT == 1 || tile0 + it + 1 < ntiles);
        if (more) {
            issue(cur ^ 1, n0 + C::BN);
            if constexpr (C::VMASK) load_vmask(n0 + C::BN);
        }
        const uint16_t *sK = stage0 + cur * C::STAGE, *sV = sK + C::SK;
        const uint8_t *sKb = reinterpret_cast<const uint8_t *>(sV + C::SK);
        // (a tile hidden from every query of this wave: so are all later ones, but the copies and barriers go on)
        if (!(a.causal && n0 > wq0 + 31) && wq0 < a.Lq && (C::SPLIT == 1 || tile0 + it < ntiles)) {
            if constexpr (C::EXP_FIRST) __builtin_amdgcn_s_setprio(0);
            f32x16_t s[C::KBLK];
#pragma unroll
            for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                for (int v = 0; v < 16; ++v) s[kb][v] = 0.f;
            // Fragments are requested two contraction steps ahead, beside the products; those of the first 16 keys of V with the
            // last ones.
            TileAddr<C::ROWCH> ta(lds_addr_of(sK), c, g);
            asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
            u32x4_t kf[C::NK][C::KBLK], vt[C::NDV];
            auto request = [&](int t) {
#pragma unroll
                for (int kb = 0; kb < C::KBLK; ++kb)
                    kf[t][kb] = t < C::NKD ? ta.load_row(t, kb * 32 * C::ROWCH * 16)
                                           : *reinterpret_cast<const u32x4_t *>(sKb + lean_row_addr<C::CPR ? C::CPR : 2>(c, 2 * (t - C::NKD) + g) + kb * 32 * C::CPR * 16);
            };
            auto columns = [&](int key) {
#pragma unroll
                for (int n = 0; n < C::NDV; ++n) vt[n] = ta.load_tr(n, 2 * C::SK + key * C::ROWCH * 16);
            };
            // the softmax scale multiplies the fp32 q k^T accumulator before the bias steps (:246-256)
            auto scale_scores = [&]() {
#pragma unroll
                for (int kb = 0; kb < C::KBLK; ++kb) {
                    const float *sM = reinterpret_cast<const float *>(sV + C::SK + C::SKB) + kb * 32 + 4 * g;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        f32x4_t x;
                        if constexpr (C::VMASK) x = *reinterpret_cast<const f32x4_t *>(sM + 8 * j);
#pragma unroll
                        for (int e = 0; e < 4; ++e) s[kb][4 * j + e] = C::VMASK ? __builtin_fmaf(s[kb][4 * j + e], a.scale, x[e]) : s[kb][4 * j + e] * a.scale;
                    }
                }
            };
            request(0);
            request(1);
            FB_HOLD;
#pragma unroll
            for (int t = 0; t < C::NK; ++t) {
                if (!C::FOLD && t == C::NKD) scale_scores();
                if (t + 2 < C::NK)
                    request(t + 2);
                else if (t + 2 == C::NK)
                    columns(0);
#pragma unroll
                for (int kb = 0; kb < C::KBLK; ++kb) s[kb] = T::mfma(kf[t][kb], qr[t], s[kb]);
                if (!C::FOLD && t == C::NKD - 1) {
                    mix<C::KBLK * C::NKD, 1, 0>();
                    FB_HOLD;
                }
            }
            if constexpr (!C::FOLD && C::NKR == 0) scale_scores();
            if constexpr (C::FOLD) {
                mix<C::KBLK * C::NK, 1, 0>();
                FB_HOLD;
            }
            // (bitwise on purpose, as in the dq kernel: no scalar block between the last MFMA and the branch)
            const bool edge = (n0 + C::BN > a.Lk) | ((a.causal != 0) & (n0 + C::BN - 1 > wq0));
            if (edge) {
                int key0 = n0 + 4 * g;
                asm volatile("" : "+v"(key0)); // (computed here, not kept in registers across the loop)
#pragma unroll
                for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int key = key0 + kb * 32 + 8 * (v >> 2) + (v & 3);
                        if (key >= a.Lk || (a.causal && key > query)) s[kb][v] = -INFINITY;
                    }
            }
            if constexpr (C::EXP_FIRST) __builtin_amdgcn_s_setprio(1);
            float mx = s[0][0];
#pragma unroll
            for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                for (int v = (kb == 0 ? 1 : 0); v < 16; ++v) mx = fmaxf(mx, s[kb][v]);
            mx = half_wave_max(mx);
            const bool grow = mx > m_ref + lag; // also true for the first finite score of a row
            if (__any(grow)) {
                const float m_new = grow ? mx : m_ref;
                const float alpha = grow ? fast_exp2((m_ref - m_new) * to_log2) : 1.f; // exp2(-inf) = 0
                l_run *= alpha;
#pragma unroll
                for (int n = 0; n < C::NDV; ++n)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc_o[n][v] *= alpha;
                m_ref = m_new;
                m2 = reference_log2<T>(m_new, to_log2);
            }
#pragma unroll
            for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    u32x4_t pb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float p0 = fast_exp2(__builtin_fmaf(s[kb][8 * t + 2 * e], to_log2, -m2));
                        const float p1 = fast_exp2(__builtin_fmaf(s[kb][8 * t + 2 * e + 1], to_log2, -m2));
                        pb[e] = T::pack2(p0, p1);
                        l_run += p0 + p1;
                    }
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) acc_o[n] = T::mfma(vt[n], pb, acc_o[n]);
                    if (2 * kb + t + 1 < 2 * C::KBLK) columns(kb * 32 + 16 * t + 16);
                }
        }
        if constexpr (C::VMASK) {
            if (more) store_vmask(cur ^ 1);
        }
        wait_vmcnt<0>(); // the next tile has landed
        barrier_lds();
    }

    if constexpr (C::SPLIT == 2) { // the second group's sums to the first one's (the stages are free: the loop ends with a barrier)
        uint8_t *ex = smem + wave * 4096;
        float *em = reinterpret_cast<float *>(smem + C::NDV * 16384 + wave * 512) + lane;
#pragma unroll
        for (int n = 0; n < C::NDV; ++n) asm volatile("s_nop 11" : "+v"(acc_o[n]));
        if (grp == 1) {
#pragma unroll
            for (int n = 0; n < C::NDV; ++n) lds_put_block(ex + n * 16384, acc_o[n], lane);
            em[0] = m_ref;
            em[64] = l_run;
        }
        barrier_lds();
        if (grp == 1) return;
        float mine, other;
        join_references(m_ref, em[0], to_log2, mine, other);
        l_run = l_run * mine + em[64] * other;
#pragma unroll
        for (int n = 0; n < C::NDV; ++n) {
#pragma unroll
            for (int v = 0; v < 16; ++v) acc_o[n][v] *= mine;
            lds_add_block(ex + n * 16384, acc_o[n], lane, other);
        }
    }
    uint16_t *obase = const_cast<uint16_t *>(a.o.ptr) + b * a.o.sb + h * a.o.sh;
    int q = query;
    asm volatile("" : "+v"(q)); // (keeps the address arithmetic below the key loop)
    const float l = l_run + __shfl_xor(l_run, 32, 64);
    const float inv = 1.f / l;
    const bool ok = q < a.Lq;
    if (ok && g == 0) a.lse[(int64_t)bh * a.Lq + q] = m_ref * (C::FOLD ? a.scale : 1.f) + __builtin_amdgcn_logf(l) * kLn2;
    uint16_t *orow = obase + (int64_t)(ok ? q : 0) * a.o.ss;
#pragma unroll
    for (int n = 0; n < C::NDV; ++n) store_acc_rows<T, true>(orow + 32 * n, ok, true, acc_o[n], inv, a.d - 32 * n, g);
}

template <class T, int NKD, int NKR, int NDV, int MASK, bool FOLD, int SPLIT>
static hipError_t launch_fwd_wide_split(const FwdArgs &a0, hipStream_t stream) {
    typedef FwdWideCfg<T, NKD, NKR, NDV, MASK, FOLD, SPLIT> C;
    FwdArgs a = a0;
    a.ntiles_m = (a.Lq + C::BM - 1) / C::BM;
    auto kern = fwd_wide_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    const int64_t total = (int64_t)a.ntiles_m * a.B * a.H;
    return launch_flat(kern, total, C::NTHREADS, C::LDS_BYTES, stream, a);
}

// Two groups of waves, which split the keys and join their sums in LDS: up to one workgroup a compute unit, under a causal mask, where a launch
// lasts as long as its longest workgroup, up to two if that one is long. us, one group / two, rank 8: head dim 64, 64 workgroups (B1 H8) of 1000
// keys 19.1 / 16.8, causal 19.3 / 16.8, padded 22.8 / 18.9; 192 of 1500 27.6 / 23.9, of 3000 (B2 H4) 48.1 / 37.4; 256 of 1024 (B2 H16) 20.1 / 18.3, of 4096
// (B1 H8) 59.8 / 49.4; of 512 keys (B1 H8) 11.6 / 11.1, of 256 7.66 / 7.75; 384 of 1500 (B1 H32) 37.4 / 43.2, causal 27.9 / 25.9, of 700 causal 16.7 / 21.0;
// 512 causal of 2048 36.8 / 36.3, of 8192 128.6 / 105.7; head dim 128, 64 of 1000 26.2 / 24.0, 256 of 4096 86.7 / 78.0, 512 causal of 8192 196 / 158.
inline bool wide_split(const FwdArgs &a) {
    const int64_t wgs = (int64_t)a.B * a.H * ((a.Lq + 127) / 128);
    return a.Lk >= 512 && wgs <= (a.causal && a.Lk >= 1024 ? 2 : 1) * (int64_t)num_cus();
}

template <class T, int NKD, int NKR, int NDV, int MASK, bool FOLD>
static hipError_t launch_fwd_wide(const FwdArgs &a, hipStream_t stream) {
    return wide_split(a) ? launch_fwd_wide_split<T, NKD, NKR, NDV, MASK, FOLD, 2>(a, stream) : launch_fwd_wide_split<T, NKD, NKR, NDV, MASK, FOLD, 1>(a, stream);
}

} // namespace fb
