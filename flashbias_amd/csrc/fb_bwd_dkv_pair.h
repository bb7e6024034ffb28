// dk, dv and dk_bias for head dims 65 ... 128 in one pass (aligned tensors, rank up to 32, no mask or a vector mask).
// Included by fb_bwd_dkv.hip after the general kernel, whose arithmetic it shares (lane = key, register = query).
//
// At these head dims the accumulators of dv and [dk | dk_bias] and the operands K, K_b, V of 32 keys do not fit one wave of
// 256 registers beside anything else, and two passes compute S and P twice (44 products a 32 x 32 block instead of
// 35).  Here two waves share a block of 32 keys: wave w < 4 forms S and P and sums dv (K, K_b and dv in registers, 17
// products), hands P over in fp32 through LDS, and wave w + 4 forms dP and dS and sums [dk | dk_bias] (V and dk in
// registers, 18 products) one step of queries later.  Both are on one SIMD.
//
// Causal B4 H32 L=4096 d128 r8: 1.72 ms in two passes, 1.34 here (B2 H8 L=4096 without a mask 0.40 -> 0.29, B1 H8 L=1000 0.114 ->
// 0.048).  The matrix pipe is busy for half of the time at a clock of 1.7 GHz (two passes: a third at 2.0): the card's power is
// what is left, and steps of 32 queries, row fragments loaded a block ahead or an order slot by slot changed nothing more.
//
// Steps of 64 queries run through a ring of three LDS stages: the second waves' step, the first waves' and the one on its
// way.  Two barriers a step: the second waves take the last step's P into registers before the first one, the first
// waves write this step's after it, so one buffer serves.
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKR_, int MASK_, bool FOLD_>
struct DkvPairCfg {
    static constexpr int NKD = 8, NKR = NKR_, NK = NKD + NKR_, NDV = 4, MB = 4 + (NKR_ > 0 ? 1 : 0);
    static constexpr bool FOLD = FOLD_, VMASK = MASK_ == kVectorMask;
    static_assert(MASK_ != kMatrixMask && !(FOLD_ && VMASK) && NKR_ <= 2, "");
    static constexpr int NWAVES = 8, NTHREADS = 64 * NWAVES, BN = 128, BMQ = 64;
    static constexpr int ROWCH = 16, CPR = 2 * (NKR > 0 ? NKR : 1);
    // a stage, bytes: Q and dO rows of 256, Q_b rows of 32 or 64, lse * log2(e) and -delta
    static constexpr int SQ = BMQ * 256, SQB = NKR > 0 ? BMQ * CPR * 16 : 0, STAGE = 2 * SQ + SQB + 8 * BMQ, NSTAGE = 3;
    static constexpr int P = NSTAGE * STAGE, LDS_BYTES = P + 4 * 2 * 4096; // P: two blocks of each pair
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
    const int step0 = a.causal ? n0 / C::BMQ : 0, nsteps = (a.Lq + C::BMQ - 1) / C::BMQ; // causal: the first step that sees a key
    auto walk = [&](auto first_tag) { // (two copies of the loop: the second waves' registers are not the first ones')
    constexpr bool FIRST = decltype(first_tag)::value;
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

        // ---- copies: per step every wave issues five: eight rows of Q, eight of dO, and Q_b (the first waves) or a row of
        // the statistics (the others: lse * log2(e) the even, -delta the odd ones).  Past the end: the last step again.
        const int crow = 8 * wave + (lane >> 4); // (and crow + 4: the swizzle of the chunks differs)
        uint32_t chunk[2];
        uint64_t lanes_on[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            chunk[j] = (lane & 15) ^ swz_of<C::ROWCH>(crow + 4 * j);
            lanes_on[j] = __builtin_amdgcn_ballot_w64((int)chunk[j] * 8 < a.d);
        }
        const uint32_t qpitch = (uint32_t)(a.q.ss * 2), dpitch = (uint32_t)(a.dout.ss * 2), bpitch = C::NKR > 0 ? (uint32_t)(a.qb.ss * 2) : 0u;
        const uint8_t *qbase = reinterpret_cast<const uint8_t *>(a.q.ptr + b * a.q.sb + h * a.q.sh);
        const uint8_t *dbase = reinterpret_cast<const uint8_t *>(a.dout.ptr + b * a.dout.sb + h * a.dout.sh);
        const uint8_t *bbase = C::NKR > 0 ? reinterpret_cast<const uint8_t *>(a.qb.ptr + b * a.qb.sb + h * a.qb.sh) : nullptr;
        constexpr int QB_WAVES = C::NKR > 0 ? C::BMQ * C::CPR / 64 : 0;
        int brow, bch; // (a rank of at most 8 folded with low parts: chunk 1 is a second copy of chunk 0)
        lean_copy_place<C::CPR>(lane, brow, bch);
        brow += (wave < QB_WAVES ? wave : 0) * (64 / C::CPR);
        if (C::low_parts(a) && bch == 1) bch = 0;
        const uint64_t lanes_b = __builtin_amdgcn_ballot_w64(bch * 8 < a.r);
        const float *stat = a.delta + (((wave & 1) == 0 ? (int64_t)a.B * a.H : 0) + bh) * a.Lq;
        auto issue_rows = [&](int step, int stage, const uint8_t *base, uint32_t pitch, uint32_t at) {
            const int r0 = min(step, nsteps - 1) * C::BMQ;
#pragma unroll
            for (int j = 0; j < 2; ++j) // (a ragged last step: rows past the end are the last one again)
                lds_dma16_lanes((uint32_t)min(crow + 4 * j, a.Lq - 1 - r0) * pitch + chunk[j] * 16, base + (int64_t)r0 * pitch,
                                lds0 + stage * C::STAGE + at + (2 * wave + j) * 1024, lanes_on[j]);
        };
        auto issue_rest = [&](int step, int stage) {
            const uint32_t at = lds0 + stage * C::STAGE + 2 * C::SQ;
            const int r0 = min(step, nsteps - 1) * C::BMQ;
            if (wave < QB_WAVES)
                lds_dma16_lanes((uint32_t)min(brow, a.Lq - 1 - r0) * bpitch + bch * 16, bbase + (int64_t)r0 * bpitch, at + wave * 1024, lanes_b);
            else
                lds_dma4(stat + min(r0 + lane, a.Lq - 1), at + C::SQB + (wave & 1) * 4 * C::BMQ);
        };
        auto issue_q = [&](int step, int stage) { issue_rows(step, stage, qbase, qpitch, 0); };
        auto issue_do = [&](int step, int stage) { issue_rows(step, stage, dbase, dpitch, C::SQ); };
        auto after = [](int stage) { return stage + 1 == C::NSTAGE ? 0 : stage + 1; };
        if (step0 < nsteps) {
            issue_q(step0, 0);
            issue_do(step0, 0);
            issue_rest(step0, 0);
        }

        const uint32_t pbuf = C::P + pair * 8192 + lane * 16;
        if constexpr (FIRST) {
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
            wait_vmcnt<0>();
            barrier_lds();
            int stage = 0;
            // (blocks that a causal mask hides from this wave alone are computed with everything masked: a way round them
            // cost 250 bytes of scratch)
#pragma unroll 1
            for (int step = step0; step < nsteps; ++step) {
                const uint8_t *st = smem + stage * C::STAGE;
                TileAddr16 ta(lds_addr_of(st), c, g);
                asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                const int nxt = after(stage), r0 = step * C::BMQ;
                // LDS reads are requested a phase ahead of their use, one or two beside every product: a wave issues one every
                // 16 cycles at best, and left to itself the compiler saves the registers and waits for each by itself.
                u32x4_t qa[C::NK];
                auto rows = [&](int i) {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) qa[t] = ta.load_row(t, 8192 * i);
                    if constexpr (C::NKR > 0) {
#pragma unroll
                        for (int t = 0; t < C::NKR; ++t)
                            qa[C::NKD + t] = *reinterpret_cast<const u32x4_t *>(st + 2 * C::SQ + i * 32 * C::CPR * 16 + lean_row_addr<C::CPR>(c, 2 * t + g));
                    }
                };
                const float *lse2 = reinterpret_cast<const float *>(st + 2 * C::SQ + C::SQB) + 4 * g;
                f32x4_t l[4];
                auto lses = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) l[j] = *reinterpret_cast<const f32x4_t *>(lse2 + 32 * i + 8 * j);
                };
                auto products = [&](f32x16_t &s, int t0, int t1) {
#pragma unroll
                    for (int t = t0; t < t1; ++t) s = T::mfma(qa[t], kr[t], s);
                };
                auto scaled = [&](f32x16_t &s) { // the softmax scale multiplies the fp32 q k^T accumulator before the bias steps
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[v] = C::VMASK ? __builtin_fmaf(s[v], a.scale, mkey) : s[v] * a.scale;
                    }
                };
                auto hide = [&](f32x16_t &s, int q0) {
                    // (keys past the end stay: their columns end in no other and are not stored.  Hidden, they cost the wave that holds some of them its every step
                    // and the launch of a small grid as much: fb_bwd_dkv_mid.h, step of B1 H8 L=1000 d64 70.1 -> 64.1 us.)
                    // (bitwise on purpose, as in the dq kernel: no scalar block between the last MFMA and the branch)
                    const bool edge = (q0 + 32 > a.Lq) | ((a.causal != 0) & (wk0 + 31 > q0));
                    if (edge) {
                        int query0 = q0 + 4 * g;
                        asm volatile("" : "+v"(query0)); // (computed here, not kept in registers across the loop)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int query = query0 + 8 * (v >> 2) + (v & 3);
                            if (query >= a.Lq || (a.causal && key > query)) s[v] = -INFINITY;
                        }
                    }
                    asm volatile("s_nop 11" : "+v"(s)); // (fb_bwd_win.hip: wait states across the branch above)
                };
                u32x4_t pp[2];
                auto exps = [&](const f32x16_t &s, int i, int j) { // register v <-> query r0 + 32 i + 8 (v / 4) + 4 g + v % 4
                    f32x4_t p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) p[e] = fast_exp2(__builtin_fmaf(s[4 * j + e], to_log2, -l[j][e]));
                    *reinterpret_cast<f32x4_t *>(smem + pbuf + i * 4096 + j * 1024) = p;
                    pp[j >> 1][2 * (j & 1)] = T::pack2(p[0], p[1]);
                    pp[j >> 1][2 * (j & 1) + 1] = T::pack2(p[2], p[3]);
                };
                u32x4_t dot[2][C::NDV];
                auto columns = [&](int i, int t) {
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) dot[t][n] = ta.load_tr(n, C::SQ + 8192 * i + 16 * 256 * t);
                };
                auto sums = [&](int t) {
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) acc[n] = T::mfma(dot[t][n], pp[t], acc[n]);
                };
                f32x16_t s0, s1;
#pragma unroll
                for (int v = 0; v < 16; ++v) s0[v] = s1[v] = 0.f;
                rows(0);
                issue_q(step + 1, nxt);
                FB_HOLD;
                __builtin_amdgcn_s_setprio(1);
                products(s0, 0, C::NKD);
                const u32x4_t fac0 = qa[C::NK - 1], fac1 = qa[C::NK - 2]; // (the first block's factor rows, for after the scale)
                rows(1);
                lses(0);
                mix<8, 2, 0>();
                FB_HOLD;
                scaled(s0);
                if constexpr (C::NKR == 2) s0 = T::mfma(fac1, kr[C::NK - 2], s0);
                if constexpr (C::NKR > 0) s0 = T::mfma(fac0, kr[C::NK - 1], s0);
                issue_do(step + 1, nxt);
                issue_rest(step + 1, nxt);
                FB_HOLD;
                barrier_lds(); // the second waves have taken the last step's P
                hide(s0, r0);
                products(s1, 0, C::NKD);
                columns(0, 0);
                exps(s0, 0, 0);
                exps(s0, 0, 1);
                mix<8, 1, 3>();
                FB_HOLD;
                scaled(s1);
                products(s1, C::NKD, C::NK);
                FB_HOLD;
                sums(0);
                columns(0, 1);
                exps(s0, 0, 2);
                exps(s0, 0, 3);
                mix<4, 2, 5>();
                FB_HOLD;
                lses(1);
                hide(s1, r0 + 32);
                sums(1);
                columns(1, 0);
                exps(s1, 1, 0);
                exps(s1, 1, 1);
                mix<4, 2, 5>();
                FB_HOLD;
                sums(0);
                columns(1, 1);
                exps(s1, 1, 2);
                exps(s1, 1, 3);
                mix<4, 2, 5>();
                FB_HOLD;
                sums(1);
                __builtin_amdgcn_s_setprio(0);
                wait_vmcnt<0>();
                barrier_lds();
                stage = nxt;
            }
            barrier_lds(); // (the second waves' last step)
            barrier_lds();
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
            wait_vmcnt<0>();
            barrier_lds();
            int stage = 0;
            // (the first waves' first step)
            if (step0 < nsteps) {
                issue_q(step0 + 1, 1);
                issue_do(step0 + 1, 1);
                issue_rest(step0 + 1, 1);
            }
            barrier_lds();
            wait_vmcnt<0>();
            barrier_lds();
#pragma unroll 1
            for (int step = step0; step < nsteps; ++step) {
                const uint8_t *st = smem + stage * C::STAGE;
                TileAddr16 ta(lds_addr_of(st), c, g);
                asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                const int nxt = after(stage), nxt2 = after(nxt); // (the first waves are one step ahead, the copies two)
                f32x4_t p[2][4];
                auto load_p = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) p[i][j] = *reinterpret_cast<const f32x4_t *>(smem + pbuf + i * 4096 + j * 1024);
                };
                u32x4_t da[C::NKD];
                auto rows = [&](int i) {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) da[t] = ta.load_row(t, C::SQ + 8192 * i);
                };
                f32x16_t dp; // -delta is the initial value
                const float *negd = reinterpret_cast<const float *>(st + 2 * C::SQ + C::SQB) + C::BMQ + 4 * g;
                auto deltas = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(negd + 32 * i + 8 * j);
#pragma unroll
                        for (int e = 0; e < 4; ++e) dp[4 * j + e] = x[e];
                    }
                };
                auto products = [&]() {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) dp = T::mfma(da[t], vr[t], dp);
                };
                u32x4_t ds[2], qt[2][C::MB];
                auto columns = [&](int i, int t) {
#pragma unroll
                    for (int n = 0; n < 4; ++n) qt[t][n] = ta.load_tr(n, 8192 * i + 16 * 256 * t);
                    if constexpr (C::NKR > 0) qt[t][4] = dense_read_a_tr<C::CPR>(st + 2 * C::SQ, 32 * i + 16 * t, c, g);
                };
                auto scale_p = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        ds[j >> 1][2 * (j & 1)] = T::pack2(p[i][j][0] * dp[4 * j], p[i][j][1] * dp[4 * j + 1]);
                        ds[j >> 1][2 * (j & 1) + 1] = T::pack2(p[i][j][2] * dp[4 * j + 2], p[i][j][3] * dp[4 * j + 3]);
                    }
                };
                auto sums = [&](int t) {
#pragma unroll
                    for (int n = 0; n < 4; ++n) acc[n] = T::mfma(qt[t][n], ds[t], acc[n]);
                    if constexpr (C::NKR > 0) acc_b = T::mfma(qt[t][4], ds[t], acc_b);
                };
                rows(0);
                deltas(0);
                issue_q(step + 2, nxt2);
                FB_HOLD;
                __builtin_amdgcn_s_setprio(1);
                products();
                load_p(0);
                load_p(1);
                columns(0, 0);
                mix<8, 2, 0>();
                FB_HOLD;
                issue_do(step + 2, nxt2);
                issue_rest(step + 2, nxt2);
                FB_HOLD;
                barrier_lds(); // (P is in registers)
                scale_p(0);
                FB_HOLD;
                sums(0);
                columns(0, 1);
                mix<C::MB, 2, 0>();
                FB_HOLD;
                sums(1);
                rows(1);
                deltas(1);
                mix<C::MB, 2, 0>();
                FB_HOLD;
                products();
                columns(1, 0);
                mix<8, 1, 0>();
                FB_HOLD;
                scale_p(1);
                FB_HOLD;
                sums(0);
                columns(1, 1);
                mix<C::MB, 2, 0>();
                FB_HOLD;
                sums(1);
                __builtin_amdgcn_s_setprio(0);
                wait_vmcnt<0>();
                barrier_lds();
                stage = nxt;
            }
            const bool ok = key < a.Lk;
            uint16_t *row = const_cast<uint16_t *>(a.dk.ptr) + b * a.dk.sb + h * a.dk.sh + (int64_t)(ok ? key : 0) * a.dk.ss;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                asm volatile("s_nop 11" : "+v"(acc[n]));
                store_acc_rows<T, true>(row + 32 * n, ok, a.dk.vec_ok, acc[n], a.scale, a.d - 32 * n, g);
            }
        }
    }
    if constexpr (C::NKR > 0 && !FIRST) {
        if (a.dkb.ptr) { // (null: the caller does not want the factor gradients)
            const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
            const int key = wk0 + (lane & 31);
            const bool ok = key < a.Lk;
            asm volatile("s_nop 11" : "+v"(acc_b));
            uint16_t *row = const_cast<uint16_t *>(a.dkb.ptr) + bg * a.dkb.sb + h * a.dkb.sh + (int64_t)(ok ? key : 0) * a.dkb.ss;
            store_acc_rows<T, true>(row, ok, a.dkb.vec_ok, acc_b, 1.f, a.r, lane >> 5);
        }
    }
    };
    if (wave < 4)
        walk(std::true_type{});
    else
        walk(std::false_type{});
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
