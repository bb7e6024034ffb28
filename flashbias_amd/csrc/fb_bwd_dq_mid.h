// dq and dq_bias for head dims 17 ... 64 (aligned tensors, rank up to 32, no mask): one query block a wave.  Included by
// fb_bwd_dq.hip after the general kernel; the arithmetic is that of the general kernel, operation by operation (lane = query,
// register = key; the same bits where one group of waves walks all keys).
//
// Head dims above 32: as in the dk/dv kernel for them (fb_bwd_dkv_mid.h) the reads of a phase are requested beside the products of
// the phase before; left to itself the compiler waits for each where it is used.  Head dim 32: tiles of dense 64-byte rows take half
// the copy instructions of the general kernel's padded ones (its copies are a tenth of its cycles), and without dq_bias 121 to
// 127 registers leave four waves a SIMD instead of two with two query blocks each.  The vector unit and the matrix pipe
// together bound both.
//
// General kernel against this one, training step, us, bf16: d64 without dq_bias, r2 as 16, causal B2 H16 L=2048 158 -> 144; d64 r8 causal
// B2 H8 L=4096 281 -> 259; d64 r16 B4 H16 L=2048 391 -> 379; d64 r32 B1 H4 L=1000 94 -> 88; d32 r2 as 16 without dq_bias, causal B1 H50
// L=4096 412 -> 399, L=8192 1428 -> 1397, B2 H32 L=3000 304 -> 294; d32 r32 768 x 4 rows of 768 2080 -> 2045, 301 x 4 of 301 229 -> 221.
// With a vector mask it was behind (its values a tile at a time in the stage: fp16 d64 8 x 8 x (1000 x 1500) 194 -> 196, d32 r8 157.8 ->
// 158.3), so those stay with the general kernel.
//
// SPLIT: on small grids a second group of four waves takes the second half of the keys for the same queries, in stages of its own,
// and hands its sums over in LDS (mid_split).
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKD_, int NKR_, bool FOLD_, bool BG_, int SPLIT_ = 1>
struct DqMidCfg {
    static constexpr int NKD = NKD_, NKR = NKR_, NK = NKD + NKR_, NDQ = NKD / 2;
    static_assert(NKD_ == 2 || NKD_ == 4, "");
    static constexpr bool FOLD = FOLD_, BG = BG_ && NKR_ > 0;
    static_assert(NKR_ <= 2, "");
    static constexpr int SPLIT = SPLIT_, NWAVES = 4, NTHREADS = 64 * NWAVES * SPLIT, BM = 32 * NWAVES, BN = 64; // (NWAVES: of a group)
    static constexpr int ROWCH = 2 * NKD, RB = 16 * ROWCH; // chunks and bytes of a K or V row
    static constexpr int CPR = 2 * (NKR > 0 ? NKR : 1);
    static constexpr int NI = NKD / 2; // copy instructions per wave, tensor and tile
    // a stage, bytes: K, V, K_b rows of 32 or 64
    static constexpr int SK = BN * RB, SKB = NKR > 0 ? BN * CPR * 16 : 0, STAGE = 2 * SK + SKB;
    static constexpr int LDS_BYTES = 2 * STAGE * SPLIT;
    // (head dim 32: 121-127 registers without dq_bias at ranks up to 16; at rank 32 129-135, with it 139-155)
    static constexpr int WAVES_EU = NKD == 4 || SPLIT == 2 ? 2 : BG || NKR == 2 ? 3 : 4;
    static_assert(WAVES_EU * LDS_BYTES / SPLIT <= 160 * 1024 && (SPLIT == 1 || LDS_BYTES >= (NDQ + 1) * 4 * 4096), "");
    static constexpr bool ORDERED = NKD == 4; // two waves a SIMD: the order is fixed phase by phase
    static __device__ __forceinline__ bool low_parts(const BwdArgs &a) { return FOLD_ && NKR_ == 1 && a.r <= 8 && a.scale != 1.f; }
};

template <class T, class C>
__device__ __forceinline__ void bwd_dq_mid_body(const BwdArgs &a, int wg) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int grp = C::SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8); // takes its share of the tiles of keys, in stages of its own
    uint8_t *const stages = smem + grp * 2 * C::STAGE;
    const uint32_t lds0 = lds_addr_of(stages);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & (64 * C::NWAVES - 1)) >> 6);

    // (one workgroup serves `group` consecutive batch entries of its (head, query tile), as the general kernel does)
    const int group = a.group > 1 ? a.group : 1;
    const int nbg = (a.B + group - 1) / group;
    int bgh, tile_m;
    work_order(wg, a.ntiles_m, a.ntiles_m * nbg * a.H, a.causal, bgh, tile_m);
    if (a.causal) tile_m = a.ntiles_m - 1 - tile_m; // the last query tile sees the most keys
    const int bg = bgh / a.H, h = bgh % a.H;
    const int m0 = tile_m * C::BM, wq0 = m0 + 32 * wave;

    // clear the stages once: the zero padding of the channel dimension is never rewritten
    for (int i = threadIdx.x; i < C::LDS_BYTES / 16; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem)[i] = u32x4_t{0u, 0u, 0u, 0u};
    __syncthreads();

    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e; // the scores are in units of 1 / scale when folded
    int k_end = a.Lk;
    if (a.causal && m0 + C::BM < k_end) k_end = m0 + C::BM; // keys past the last query are hidden
    const int ntiles = (k_end + C::BN - 1) / C::BN, walk = (ntiles + C::SPLIT - 1) / C::SPLIT, tile0 = grp * walk;
    f32x16_t acc_b; // dq_bias, summed over the group
#pragma unroll
    for (int v = 0; v < 16; ++v) acc_b[v] = 0.f;
    u32x4_t qbr[C::NKR > 0 ? C::NKR : 1]; // (outlives a batch entry when the batch shares the factor)

    for (int bi = 0; bi < group; ++bi) {
        const int b = __builtin_amdgcn_readfirstlane(bg * group + bi);
        if (b >= a.B) break;
        int tid_again = threadIdx.x; // (opaque: what derives from the lane id is recomputed per entry, not kept in registers)
        asm volatile("" : "+v"(tid_again));
        const int lane = tid_again & 63, c = lane & 31, g = lane >> 5;
        const int bh = b * a.H + h, query = wq0 + c;

        // ---- copies: per tile every wave issues sixteen rows of K and of V, the first waves K_b
        int crow, cch;
        if constexpr (C::NKD == 4) {
            crow = 16 * wave + (lane >> 3); // (and crow + 8, whose chunks the swizzle moves by two places)
            cch = (lane & 7) ^ swz_of<8>(crow);
        } else {
            lean_copy_place<4>(lane, crow, cch);
            crow += 16 * wave;
        }
        uint64_t lanes_on[C::NI];
#pragma unroll
        for (int j = 0; j < C::NI; ++j) lanes_on[j] = __builtin_amdgcn_ballot_w64((cch ^ (2 * j)) * 8 < a.d);
        const uint32_t kpitch = (uint32_t)(a.k.ss * 2), vpitch = (uint32_t)(a.v.ss * 2), bpitch = C::NKR > 0 ? (uint32_t)(a.kb.ss * 2) : 0u;
        const uint8_t *kbase = reinterpret_cast<const uint8_t *>(a.k.ptr + b * a.k.sb + h * a.k.sh);
        const uint8_t *vbase = reinterpret_cast<const uint8_t *>(a.v.ptr + b * a.v.sb + h * a.v.sh);
        const uint8_t *bbase = C::NKR > 0 ? reinterpret_cast<const uint8_t *>(a.kb.ptr + b * a.kb.sb + h * a.kb.sh) : nullptr;
        constexpr int KB_WAVES = C::NKR > 0 ? C::BN * C::CPR / 64 : 0;
        int brow, bch; // (a rank of at most 8 folded with low parts: chunk 1 is a second copy of chunk 0)
        lean_copy_place<C::CPR>(lane, brow, bch);
        brow += (wave < KB_WAVES ? wave : 0) * (64 / C::CPR);
        if (C::low_parts(a) && bch == 1) bch = 0;
        const uint64_t lanes_b = __builtin_amdgcn_ballot_w64(bch * 8 < a.r);
        auto issue = [&](int n0, int stage) {
            const int last = a.Lk - 1 - n0; // (a ragged last tile: rows past the end are the last one again)
            const uint32_t at = lds0 + stage * C::STAGE;
#pragma unroll
            for (int j = 0; j < C::NI; ++j) {
                const uint32_t row = (uint32_t)min(crow + 8 * j, last), ch = (uint32_t)(cch ^ (2 * j)) * 16;
                lds_dma16_lanes(row * kpitch + ch, kbase + (int64_t)n0 * kpitch, at + (C::NI * wave + j) * 1024, lanes_on[j]);
                lds_dma16_lanes(row * vpitch + ch, vbase + (int64_t)n0 * vpitch, at + C::SK + (C::NI * wave + j) * 1024, lanes_on[j]);
            }
            if (wave < KB_WAVES) lds_dma16_lanes((uint32_t)min(brow, last) * bpitch + bch * 16, bbase + (int64_t)n0 * bpitch, at + 2 * C::SK + wave * 1024, lanes_b);
        };
        if (C::SPLIT == 1 || tile0 < ntiles) issue(tile0 * C::BN, 0);

        // ---- query-side operands
        u32x4_t qr[C::NKD], dor[1][C::NKD];
        const uint16_t *qbase = a.q.ptr + b * a.q.sb + h * a.q.sh, *dobase = a.dout.ptr + b * a.dout.sb + h * a.dout.sh;
#pragma unroll
        for (int t = 0; t < C::NKD; ++t) {
            qr[t] = load_chunk<true>(qbase, a.q.ss, query, a.Lq, 16 * t + 8 * g, a.d);
            dor[0][t] = load_chunk<true>(dobase, a.dout.ss, query, a.Lq, 16 * t + 8 * g, a.d);
        }
        if constexpr (C::NKR > 0) {
            if (bi == 0 || a.qb.sb != 0) {
                const uint16_t *qbbase = a.qb.ptr + b * a.qb.sb + h * a.qb.sh;
                const bool low = C::low_parts(a) && g == 1;
#pragma unroll
                for (int t = 0; t < C::NKR; ++t) {
                    qbr[t] = load_chunk<true>(qbbase, a.qb.ss, query, a.Lq, low ? 0 : 16 * t + 8 * g, a.r);
                    if (C::FOLD && a.scale != 1.f) qbr[t] = fold_scale_chunk<T>(qbr[t], 1.f / a.scale, C::low_parts(a), low);
                }
            }
        }
        float nd, lse2;
        dq_row_stats<T, C::NKD, true>(a, dor[0], b, h, bh, query, g, nd, lse2);
        f32x16_t negd, acc[C::NDQ];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            negd[v] = nd;
#pragma unroll
            for (int n = 0; n < C::NDQ; ++n) acc[n][v] = 0.f;
        }
        wait_vmcnt<0>();
        barrier_lds();

#pragma unroll 1
        for (int it = 0; it < walk; ++it) {
            const int stage = it & 1, n0 = (tile0 + it) * C::BN;
            if (it + 1 < walk && (C::SPLIT == 1 || tile0 + it + 1 < ntiles)) issue(n0 + C::BN, stage ^ 1);
            if (!(a.causal && n0 > wq0 + 31) && wq0 < a.Lq && (C::SPLIT == 1 || tile0 + it < ntiles)) {
                const uint8_t *st = stages + stage * C::STAGE;
                TileAddr<C::ROWCH> ta(lds_addr_of(st), c, g);
                if constexpr (C::ORDERED) asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                u32x4_t ka[C::NK], va[C::NKD];
                auto rows = [&](int i) {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) {
                        ka[t] = ta.load_row(t, 32 * C::RB * i);
                        va[t] = ta.load_row(t, C::SK + 32 * C::RB * i);
                    }
#pragma unroll
                    for (int t = 0; t < C::NKR; ++t)
                        ka[C::NKD + t] = *reinterpret_cast<const u32x4_t *>(st + 2 * C::SK + i * 32 * C::CPR * 16 + lean_row_addr<C::CPR>(c, 2 * t + g));
                };
                u32x4_t kt[C::NDQ + 1];
                auto columns = [&](int i, int t) {
#pragma unroll
                    for (int n = 0; n < C::NDQ; ++n) kt[n] = ta.load_tr(n, 32 * C::RB * i + 16 * C::RB * t);
                    if constexpr (C::BG) kt[C::NDQ] = dense_read_a_tr<C::CPR>(st + 2 * C::SK, 32 * i + 16 * t, c, g);
                };
                u32x4_t dsp[2];
                auto sums = [&](int t) {
#pragma unroll
                    for (int n = 0; n < C::NDQ; ++n) acc[n] = T::mfma(kt[n], dsp[t], acc[n]);
                    if constexpr (C::BG) acc_b = T::mfma(kt[C::NDQ], dsp[t], acc_b);
                };
                rows(0);
                if constexpr (C::ORDERED) FB_HOLD;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    // ---- q k^T and q_b k_b^T: two chains joined by the FMA that applies the softmax scale to the first (:638-641);
                    // folded, one chain
                    f32x16_t s, sb, dp = negd;
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[v] = sb[v] = 0.f;
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) {
                        s = T::mfma(ka[t], qr[t], s);
                        dp = T::mfma(va[t], dor[0][t], dp);
                    }
#pragma unroll
                    for (int t = 0; t < C::NKR; ++t) {
                        if constexpr (C::FOLD)
                            s = T::mfma(ka[C::NKD + t], qbr[t], s);
                        else
                            sb = T::mfma(ka[C::NKD + t], qbr[t], sb);
                    }
                    columns(i, 0);
                    if constexpr (C::ORDERED) {
                        mix<2 * C::NKD + C::NKR, 1, 0>();
                        FB_HOLD;
                    }
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[v] = C::NKR > 0 ? __builtin_fmaf(s[v], a.scale, sb[v]) : s[v] * a.scale;
                    }
                    // (bitwise on purpose, as in the general kernel: no scalar block between the last MFMA and the branch)
                    const bool edge = (n0 + 32 * i + 32 > a.Lk) | ((a.causal != 0) & (n0 + 32 * i + 31 > wq0));
                    if (edge) {
                        int key0 = n0 + 32 * i + 4 * g;
                        asm volatile("" : "+v"(key0)); // (computed here, not kept in 16 registers across the loop)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int key = key0 + 8 * (v >> 2) + (v & 3);
                            if (key >= a.Lk || (a.causal && key > query)) s[v] = -INFINITY;
                        }
                    }
                    if (C::ORDERED) asm volatile("s_nop 11" : "+v"(s)); // (fb_bwd_win.hip: wait states across the branch above)
                    if (i == 0) {
                        rows(1);
                        if constexpr (C::ORDERED) FB_HOLD;
                    }
#pragma unroll
                    for (int v = 0; v < 16; v += 2) {
                        const float p0 = fast_exp2(__builtin_fmaf(s[v], to_log2, -lse2));
                        const float p1 = fast_exp2(__builtin_fmaf(s[v + 1], to_log2, -lse2));
                        dsp[v >> 3][(v & 7) >> 1] = T::pack2(p0 * dp[v], p1 * dp[v + 1]);
                    }
                    if constexpr (C::ORDERED) FB_HOLD;
                    // ---- [dQ | dQ_b]^T += [K | K_b]^T dS^T over this block's 32 keys
                    sums(0);
                    columns(i, 1);
                    if constexpr (C::ORDERED) {
                        mix<C::NDQ + (C::BG ? 1 : 0), 2, 0>();
                        FB_HOLD;
                    }
                    sums(1);
                    if constexpr (C::ORDERED) FB_HOLD;
                }
            }
            wait_vmcnt<0>(); // the next tile has landed
            barrier_lds();
        }

        if constexpr (C::SPLIT == 2) { // the second group's sums to the first one's (the stages are free: the loop ends with a barrier)
            uint8_t *ex = smem + wave * 4096;
#pragma unroll
            for (int n = 0; n < C::NDQ; ++n) asm volatile("s_nop 11" : "+v"(acc[n]));
            if constexpr (C::BG) asm volatile("s_nop 11" : "+v"(acc_b));
            if (grp == 1) {
#pragma unroll
                for (int n = 0; n < C::NDQ; ++n) lds_put_block(ex + n * 16384, acc[n], lane);
                if constexpr (C::BG) lds_put_block(ex + C::NDQ * 16384, acc_b, lane);
            }
            barrier_lds();
            if (grp == 1) return; // (one batch entry: launch_dq_mid)
#pragma unroll
            for (int n = 0; n < C::NDQ; ++n) lds_add_block(ex + n * 16384, acc[n], lane);
            if constexpr (C::BG) lds_add_block(ex + C::NDQ * 16384, acc_b, lane);
        }
        int q = wq0 + c;
        asm volatile("" : "+v"(q)); // (keeps the address arithmetic below the key loop)
        const bool ok = q < a.Lq;
        uint16_t *row = const_cast<uint16_t *>(a.dq.ptr) + b * a.dq.sb + h * a.dq.sh + (int64_t)(ok ? q : 0) * a.dq.ss;
#pragma unroll
        for (int n = 0; n < C::NDQ; ++n) {
            asm volatile("s_nop 11" : "+v"(acc[n]));
            store_acc_rows<T, true>(row + 32 * n, ok, a.dq.vec_ok, acc[n], a.scale, a.d - 32 * n, g);
        }
    }
    if constexpr (C::BG) {
        const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        const int q = wq0 + (lane & 31);
        const bool ok = q < a.Lq;
        asm volatile("s_nop 11" : "+v"(acc_b));
        uint16_t *row = const_cast<uint16_t *>(a.dqb.ptr) + bg * a.dqb.sb + h * a.dqb.sh + (int64_t)(ok ? q : 0) * a.dqb.ss;
        store_acc_rows<T, true>(row, ok, a.dqb.vec_ok, acc_b, 1.f, a.r, lane >> 5);
    }
}

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void bwd_dq_mid_kernel(const BwdArgs a) {
    bwd_dq_mid_body<T, C>(a, blockIdx.x);
}

template <class T, int NKD, int NKR, bool FOLD, bool BG, int SPLIT = 1>
static hipError_t launch_dq_mid_split(const BwdArgs &a0, hipStream_t stream) {
    typedef DqMidCfg<T, NKD, NKR, FOLD, BG, SPLIT> C;
    BwdArgs a = a0;
    a.ntiles_m = (a.Lq + C::BM - 1) / C::BM;
    auto kern = bwd_dq_mid_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    const int group = a.group > 1 ? a.group : 1;
    return launch_flat(kern, (int64_t)a.ntiles_m * ((a.B + group - 1) / group) * a.H, C::NTHREADS, C::LDS_BYTES, stream, a);
}

template <class T, int NKD, int NKR, bool FOLD, bool BG>
static hipError_t launch_dq_mid_bg(const BwdArgs &a, hipStream_t stream) {
    if (mid_split(a, a.Lq, a.Lk)) return launch_dq_mid_split<T, NKD, NKR, FOLD, BG, 2>(a, stream);
    return launch_dq_mid_split<T, NKD, NKR, FOLD, BG>(a, stream);
}

// Whether aligned calls without a mask take this kernel: 2 all, 1 those that want no dq_bias, 0 none (measured above).  Head dims above
// 32, and at head dim 32 ranks above 16 and calls that want no dq_bias; with it the general kernel's two query blocks a wave
// share enough to stay level at ranks up to 16, on grids where the walk is not split (B2 H4 L=8192 r16 training step 537 / 538, B8 H16 L=700 100 / 99.5).
constexpr int dq_mid_use(int nkd, int nkr) { return nkr > 2 ? 0 : nkd == 4 || (nkd == 2 && nkr == 2) ? 2 : nkd == 2 && nkr == 1 ? 1 : 0; }

template <class T, int NKD, int NKR, bool FOLD>
static hipError_t launch_dq_mid(const BwdArgs &a, hipStream_t stream) {
    if constexpr (NKR > 0 && dq_mid_use(NKD, NKR) == 2) {
        if (a.dqb.ptr) return launch_dq_mid_bg<T, NKD, NKR, FOLD, true>(a, stream);
    }
    if constexpr (NKR > 0 && dq_mid_use(NKD, NKR) == 1) {
        if (a.dqb.ptr) return launch_dq_mid_split<T, NKD, NKR, FOLD, true, 2>(a, stream); // (both_split)
    }
    return launch_dq_mid_bg<T, NKD, NKR, FOLD, false>(a, stream); // (no dq_bias wanted: without its products)
}

} // namespace fb
