// dk, dv and dk_bias for head dims 17 ... 64 (aligned tensors, rank up to 32, no mask or a vector mask).  Included by
// fb_bwd_dkv.hip after the pair kernel; the arithmetic is that of the general kernel, operation by operation (lane = key,
// register = query; the same bits where one group of waves walks all queries).
//
// Head dims above 32.  A 32 x 32 block takes 19 or 21 products (650 cycles), about 100 vector instructions (450) and 37 LDS reads.  Left to itself the
// compiler asks for each fragment where it is used and waits for it, sixteen times a block: 4000 cycles for a wave that has a SIMD
// to itself.  Here the reads of a phase are requested beside the products of the phase before, tiles of 128-byte rows and a dense
// region for Q_b take half the copy instructions, and two stages leave the reads' addresses in two registers.  What is left is
// two waves a SIMD (the accumulators and operands of 32 keys take 213 to 256 registers) that overlap their products and exponentials in
// part, and the copies (14 % without them, a fifth of it the clock).
//
// General kernel against this one, us: fp16 r16, 8 x 8 x (1000 x 1500) with a padding mask 118 -> 97 (training step 212 -> 190);
// bf16 r16 B4 H16 L=2048 217 -> 190 (step 409 -> 387); r8 causal B2 H8 L=4096 147 -> 119 (306 -> 276); r2 as 16 without dk_bias,
// causal B2 H16 L=2048 80 -> 59 (177 -> 156); r32 B1 H4 L=1000 54 -> 42 (106 -> 94).
//
// Head dim 32: three waves a SIMD (129 to 167 registers) cover for each other as in the general kernel; what counts is the dense
// rows of 64 bytes, three or four copy instructions a wave and step for six or seven (the copies were a tenth of the cycles).
// General kernel against this one, training step, us, bf16: r2 as 16 without dk_bias, causal B1 H50 L=4096 412 -> 399, L=8192 1448 ->
// 1416, B2 H32 L=3000 306 -> 293; r16 B2 H4 L=8192 567 -> 555, B8 H16 L=700 100 -> 95; r32 768 x 4 rows of 768 2139 -> 2097, 301 x
// 4 of 301 225 -> 213; r32 fp16 with a padding mask, 2 x 4 x (1000 x 3000) 170 -> 160.  Not kept: four waves without dk_bias (spills:
// 399 -> 409).
//
// SPLIT: on small grids a second group of four waves takes the second half of the queries for the same keys, in stages of its own,
// and hands its sums over in LDS (mid_split).  At 1 x 8 x 1000 one group takes 2.6 us for a step of 64 queries, most of it waiting.
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKD_, int NKR_, int MASK_, bool FOLD_, bool BG_, int SPLIT_ = 1>
struct DkvMidCfg {
    static constexpr int NKD = NKD_, NKR = NKR_, NK = NKD + NKR_, NDV = NKD / 2;
    static_assert(NKD_ == 2 || NKD_ == 4, "");
    static constexpr bool FOLD = FOLD_, VMASK = MASK_ == kVectorMask, BG = BG_ && NKR_ > 0;
    static_assert(MASK_ != kMatrixMask && !(FOLD_ && VMASK) && NKR_ <= 2, "");
    static constexpr int MB = NDV + (BG ? 1 : 0); // 32-row blocks of [dK | dK_b]^T
    static constexpr int SPLIT = SPLIT_, NWAVES = 4, NTHREADS = 64 * NWAVES * SPLIT, BN = 128, BMQ = 64; // (NWAVES: of a group)
    static constexpr int CPR = 2 * (NKR > 0 ? NKR : 1);
    static constexpr int ROWCH = 2 * NKD, RB = 16 * ROWCH; // chunks and bytes of a Q or dO row
    static constexpr int NI = NKD / 2; // copy instructions per wave, tensor and step
    // a stage, bytes: Q, dO, Q_b rows of 32 or 64, lse * log2(e) and -delta
    static constexpr int SQ = BMQ * RB, SQB = NKR > 0 ? BMQ * CPR * 16 : 0, STAGE = 2 * SQ + SQB + 8 * BMQ, NSTAGE = 2;
    static constexpr int LDS_BYTES = NSTAGE * STAGE * SPLIT;
    static constexpr int WAVES_EU = NKD == 4 || SPLIT == 2 ? 2 : 3;
    static_assert(WAVES_EU * LDS_BYTES / SPLIT <= 160 * 1024 && (SPLIT == 1 || LDS_BYTES >= 2 * NDV * 16384), "");
    // Rank above 16 with dk_bias at head dims above 32: the places of the copies are formed where they are used.  Kept, they spill (24
    // bytes), and a reload waits for the tile that has just been requested: training step, us, r32 causal B2 H8 L=4096 272 -> 265,
    // B4 H16 L=2048 405 -> 400, B1 H4 L=1000 87.3 -> 85.  The others have the registers (r2 as 16 causal B2 H16 L=2048 136.5 -> 138).
    static constexpr bool FRESH = NKD == 4 && BG && (NKR == 2 || SPLIT == 2);
    static constexpr bool ORDERED = NKD == 4; // two waves a SIMD: the order is fixed phase by phase
    static __device__ __forceinline__ bool low_parts(const BwdArgs &a) { return FOLD_ && NKR_ == 1 && a.r <= 8 && a.scale != 1.f; }
};

template <class T, class C>
__device__ __forceinline__ void bwd_dkv_mid_body(const BwdArgs &a, int wg) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int grp = C::SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8); // takes its share of the steps, in stages of its own
    uint8_t *const stages = smem + grp * C::NSTAGE * C::STAGE;
    const uint32_t lds0 = lds_addr_of(stages);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & (64 * C::NWAVES - 1)) >> 6);

    // (one workgroup serves `group` consecutive batch entries of its (head, key tile), as the general kernel does)
    const int group = a.group > 1 ? a.group : 1;
    const int nbg = (a.B + group - 1) / group;
    int bgh, tile_n;
    work_order(wg, a.ntiles_n, a.ntiles_n * nbg * a.H, a.causal, bgh, tile_n);
    const int bg = bgh / a.H, h = bgh % a.H;
    const int n0 = tile_n * C::BN, wk0 = n0 + 32 * wave;

    // clear the stages once: the zero padding of the channel dimension is never rewritten
    for (int i = threadIdx.x; i < C::LDS_BYTES / 16; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem)[i] = u32x4_t{0u, 0u, 0u, 0u};
    __syncthreads();

    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e; // the scores are in units of 1 / scale when folded
    const int nsteps = (a.Lq + C::BMQ - 1) / C::BMQ, seen = a.causal ? n0 / C::BMQ : 0; // causal: the first step that sees a key
    const int walk = (max(nsteps - seen, 0) + C::SPLIT - 1) / C::SPLIT, step0 = seen + grp * walk;
    f32x16_t acc_b; // dk_bias, summed over the group
#pragma unroll
    for (int v = 0; v < 16; ++v) acc_b[v] = 0.f;

    for (int bi = 0; bi < group; ++bi) {
        const int b = __builtin_amdgcn_readfirstlane(bg * group + bi);
        if (b >= a.B) break;
        int tid_again = threadIdx.x; // (opaque: what derives from the lane id is recomputed per entry, not kept in registers)
        asm volatile("" : "+v"(tid_again));
        const int lane = tid_again & 63, c = lane & 31, g = lane >> 5;
        const int bh = b * a.H + h, key = wk0 + c;

        // ---- copies: per step every wave issues sixteen rows of Q and of dO, the first waves Q_b, the last ones a row of the
        // statistics.
        auto row_place = [&](int lane, int &crow, int &cch) {
            if constexpr (C::NKD == 4) {
                crow = 16 * wave + (lane >> 3); // (and crow + 8, whose chunks the swizzle moves by two places)
                cch = (lane & 7) ^ swz_of<8>(crow);
            } else {
                lean_copy_place<4>(lane, crow, cch);
                crow += 16 * wave;
            }
        };
        int crow, cch;
        row_place(lane, crow, cch);
        uint64_t lanes_on[C::NI];
#pragma unroll
        for (int j = 0; j < C::NI; ++j) lanes_on[j] = __builtin_amdgcn_ballot_w64((cch ^ (2 * j)) * 8 < a.d);
        const uint32_t qpitch = (uint32_t)(a.q.ss * 2), dpitch = (uint32_t)(a.dout.ss * 2), bpitch = C::NKR > 0 ? (uint32_t)(a.qb.ss * 2) : 0u;
        const uint8_t *qbase = reinterpret_cast<const uint8_t *>(a.q.ptr + b * a.q.sb + h * a.q.sh);
        const uint8_t *dbase = reinterpret_cast<const uint8_t *>(a.dout.ptr + b * a.dout.sb + h * a.dout.sh);
        const uint8_t *bbase = C::NKR > 0 ? reinterpret_cast<const uint8_t *>(a.qb.ptr + b * a.qb.sb + h * a.qb.sh) : nullptr;
        constexpr int QB_WAVES = C::NKR > 0 ? C::BMQ * C::CPR / 64 : 0;
        // (a rank of at most 8 folded with low parts: chunk 1 is a second copy of chunk 0)
        auto factor_place = [&](int lane, int &brow, int &bch) {
            lean_copy_place<C::CPR>(lane, brow, bch);
            brow += (wave < QB_WAVES ? wave : 0) * (64 / C::CPR);
            if (C::low_parts(a) && bch == 1) bch = 0;
        };
        int brow, bch;
        factor_place(lane, brow, bch);
        const uint64_t lanes_b = __builtin_amdgcn_ballot_w64(bch * 8 < a.r);
        const float *stat = a.delta + (((wave & 1) == 0 ? (int64_t)a.B * a.H : 0) + bh) * a.Lq;
        auto issue = [&](int step, int stage) {
            const int r0 = step * C::BMQ, last = a.Lq - 1 - r0; // (a ragged last step: rows past the end are the last one again)
            const uint32_t at = lds0 + stage * C::STAGE;
            int l = lane; // (opaque: the places are formed here, not reloaded from scratch behind the copies)
            if constexpr (C::FRESH) {
                asm volatile("" : "+v"(l));
                row_place(l, crow, cch);
                factor_place(l, brow, bch);
            }
#pragma unroll
            for (int j = 0; j < C::NI; ++j) {
                const uint32_t row = (uint32_t)min(crow + 8 * j, last), ch = (uint32_t)(cch ^ (2 * j)) * 16;
                lds_dma16_lanes(row * qpitch + ch, qbase + (int64_t)r0 * qpitch, at + (C::NI * wave + j) * 1024, lanes_on[j]);
                lds_dma16_lanes(row * dpitch + ch, dbase + (int64_t)r0 * dpitch, at + C::SQ + (C::NI * wave + j) * 1024, lanes_on[j]);
            }
            if (wave < QB_WAVES) lds_dma16_lanes((uint32_t)min(brow, last) * bpitch + bch * 16, bbase + (int64_t)r0 * bpitch, at + 2 * C::SQ + wave * 1024, lanes_b);
            if (wave >= 2) lds_dma4(stat + min(r0 + l, a.Lq - 1), at + 2 * C::SQ + C::SQB + (wave & 1) * 4 * C::BMQ);
        };
        if (step0 < nsteps) issue(step0, 0);

        // ---- key-side operands
        u32x4_t kr[C::NK], vr[C::NKD];
        {
            const uint16_t *kbase = a.k.ptr + b * a.k.sb + h * a.k.sh, *vbase = a.v.ptr + b * a.v.sb + h * a.v.sh;
#pragma unroll
            for (int t = 0; t < C::NKD; ++t) {
                kr[t] = load_chunk<true>(kbase, a.k.ss, key, a.Lk, 16 * t + 8 * g, a.d);
                vr[t] = load_chunk<true>(vbase, a.v.ss, key, a.Lk, 16 * t + 8 * g, a.d);
            }
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
        }
        float mkey = 0.f; // vector mask: the value of this lane's key
        if constexpr (C::VMASK) {
            const int64_t at = mask_offset(a.mask, b, h) + min(key, a.Lk - 1);
            mkey = a.mask.is_f32 ? reinterpret_cast<const float *>(a.mask.ptr)[at] : T::to_float(reinterpret_cast<const uint16_t *>(a.mask.ptr)[at]);
        }
        f32x16_t acc_dv[C::NDV], acc_dk[C::NDV];
#pragma unroll
        for (int n = 0; n < C::NDV; ++n)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc_dv[n][v] = acc_dk[n][v] = 0.f;
        wait_vmcnt<0>();
        barrier_lds();

        int stage = 0;
#pragma unroll 1
        for (int step = step0; step < (C::SPLIT == 1 ? nsteps : step0 + walk); ++step) {
            const uint8_t *st = stages + stage * C::STAGE;
            if (step + 1 < nsteps && (C::SPLIT == 1 || step + 1 < step0 + walk)) issue(step + 1, stage ^ 1);
            const int r0 = step * C::BMQ;
            if (!(a.causal && wk0 > r0 + C::BMQ - 1) && wk0 < a.Lk && (C::SPLIT == 1 || step < nsteps)) {
                TileAddr<C::ROWCH> ta(lds_addr_of(st), c, g);
                if constexpr (C::ORDERED) asm volatile("" : "+v"(ta.row), "+v"(ta.tr));
                u32x4_t qa[C::NK], da[C::NKD];
                auto rows = [&](int i) {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) {
                        qa[t] = ta.load_row(t, 32 * C::RB * i);
                        da[t] = ta.load_row(t, C::SQ + 32 * C::RB * i);
                    }
#pragma unroll
                    for (int t = 0; t < C::NKR; ++t)
                        qa[C::NKD + t] = *reinterpret_cast<const u32x4_t *>(st + 2 * C::SQ + i * 32 * C::CPR * 16 + lean_row_addr<C::CPR>(c, 2 * t + g));
                };
                // register v <-> query r0 + 32 i + 8 (v / 4) + 4 g + v % 4
                const float *stats = reinterpret_cast<const float *>(st + 2 * C::SQ + C::SQB) + 4 * g;
                f32x16_t s, dp; // -delta is the initial value of dP
                f32x4_t l[4];
                auto deltas = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(stats + C::BMQ + 32 * i + 8 * j);
#pragma unroll
                        for (int e = 0; e < 4; ++e) dp[4 * j + e] = x[e];
                    }
                };
                auto lses = [&](int i) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) l[j] = *reinterpret_cast<const f32x4_t *>(stats + 32 * i + 8 * j);
                };
                u32x4_t dot[C::NDV], qt[C::MB];
                auto columns = [&](int i, int t) {
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) dot[n] = ta.load_tr(n, C::SQ + 32 * C::RB * i + 16 * C::RB * t);
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) qt[n] = ta.load_tr(n, 32 * C::RB * i + 16 * C::RB * t);
                    if constexpr (C::BG) qt[C::NDV] = dense_read_a_tr<C::CPR>(st + 2 * C::SQ, 32 * i + 16 * t, c, g);
                };
                u32x4_t pp[2], pds[2];
                auto sums = [&](int t) {
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) acc_dv[n] = T::mfma(dot[n], pp[t], acc_dv[n]);
#pragma unroll
                    for (int n = 0; n < C::NDV; ++n) acc_dk[n] = T::mfma(qt[n], pds[t], acc_dk[n]);
                    if constexpr (C::BG) acc_b = T::mfma(qt[C::NDV], pds[t], acc_b);
                };
                constexpr int NSUM = C::NDV + C::MB;
                rows(0);
                deltas(0);
                if constexpr (C::ORDERED) FB_HOLD;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int q0 = r0 + 32 * i;
                    // ---- S and dP; the statistics and the first half's columns come meanwhile
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) {
                        s = T::mfma(qa[t], kr[t], s);
                        dp = T::mfma(da[t], vr[t], dp);
                    }
                    u32x4_t fac[C::NKR > 0 ? C::NKR : 1]; // (the factor rows, for after the scale)
#pragma unroll
                    for (int t = 0; t < C::NKR; ++t) fac[t] = qa[C::NKD + t];
                    columns(i, 0);
                    lses(i);
                    if constexpr (C::ORDERED) {
                        mix<2 * C::NKD, 2, 0>();
                        FB_HOLD;
                    }
                    // the softmax scale multiplies the fp32 q k^T accumulator before the bias steps
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[v] = C::VMASK ? __builtin_fmaf(s[v], a.scale, mkey) : s[v] * a.scale;
                    }
#pragma unroll
                    for (int t = 0; t < C::NKR; ++t) s = T::mfma(fac[t], kr[C::NKD + t], s);
                    if constexpr (C::ORDERED) FB_HOLD;
                    // (keys past the end stay: their columns end in no other and are not stored.  Hidden, they cost the wave that holds some of them its every step
                    // and the launch of a small grid as much: step of B1 H8 L=2000 r16 74.0 -> 64.6 us, 1000 42.6 -> 38.4.)
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
                    if (i == 0) {
                        rows(1);
                        if constexpr (C::ORDERED) FB_HOLD;
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float p[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) p[e] = fast_exp2(__builtin_fmaf(s[4 * j + e], to_log2, -l[j][e]));
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            pp[j >> 1][2 * (j & 1) + e] = T::pack2(p[2 * e], p[2 * e + 1]);
                            pds[j >> 1][2 * (j & 1) + e] = T::pack2(p[2 * e] * dp[4 * j + 2 * e], p[2 * e + 1] * dp[4 * j + 2 * e + 1]);
                        }
                    }
                    if constexpr (C::ORDERED) FB_HOLD;
                    // ---- dV^T += dO^T P, [dK | dK_b]^T += [Q | Q_b]^T dS
                    sums(0);
                    columns(i, 1);
                    if constexpr (C::ORDERED) {
                        mix<NSUM, 2, 0>();
                        FB_HOLD;
                    }
                    sums(1);
                    if (i == 0) deltas(1);
                    if constexpr (C::ORDERED) {
                        mix<NSUM, 1, 0>();
                        FB_HOLD;
                    }
                }
            }
            wait_vmcnt<0>(); // the next step has landed
            barrier_lds();
            stage ^= 1;
        }

        if constexpr (C::SPLIT == 2) { // the second group's sums to the first one's (the stages are free: the loop ends with a barrier)
            uint8_t *ex = smem + wave * 4096;
#pragma unroll
            for (int n = 0; n < C::NDV; ++n) asm volatile("s_nop 11" : "+v"(acc_dv[n]), "+v"(acc_dk[n]));
            if constexpr (C::BG) asm volatile("s_nop 11" : "+v"(acc_b));
            if (grp == 1) {
#pragma unroll
                for (int n = 0; n < C::NDV; ++n) {
                    lds_put_block(ex + 2 * n * 16384, acc_dv[n], lane);
                    lds_put_block(ex + (2 * n + 1) * 16384, acc_dk[n], lane);
                }
            }
            barrier_lds();
            if (grp == 0) {
#pragma unroll
                for (int n = 0; n < C::NDV; ++n) {
                    lds_add_block(ex + 2 * n * 16384, acc_dv[n], lane);
                    lds_add_block(ex + (2 * n + 1) * 16384, acc_dk[n], lane);
                }
            }
            if constexpr (C::BG) { // (no room for a fifth block beside them)
                barrier_lds();
                if (grp == 1) lds_put_block(ex, acc_b, lane);
                barrier_lds();
                if (grp == 0) lds_add_block(ex, acc_b, lane);
            }
            if (grp == 1) return; // (one batch entry: launch_dkv_mid)
        }
        const bool ok = key < a.Lk;
        uint16_t *dvrow = const_cast<uint16_t *>(a.dv.ptr) + b * a.dv.sb + h * a.dv.sh + (int64_t)(ok ? key : 0) * a.dv.ss;
        uint16_t *dkrow = const_cast<uint16_t *>(a.dk.ptr) + b * a.dk.sb + h * a.dk.sh + (int64_t)(ok ? key : 0) * a.dk.ss;
#pragma unroll
        for (int n = 0; n < C::NDV; ++n) {
            asm volatile("s_nop 11" : "+v"(acc_dv[n]), "+v"(acc_dk[n]));
            store_acc_rows<T, true>(dvrow + 32 * n, ok, a.dv.vec_ok, acc_dv[n], 1.f, a.d - 32 * n, g);
            store_acc_rows<T, true>(dkrow + 32 * n, ok, a.dk.vec_ok, acc_dk[n], a.scale, a.d - 32 * n, g);
        }
    }
    if constexpr (C::BG) {
        const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        const int key = wk0 + (lane & 31);
        const bool ok = key < a.Lk;
        asm volatile("s_nop 11" : "+v"(acc_b));
        uint16_t *row = const_cast<uint16_t *>(a.dkb.ptr) + bg * a.dkb.sb + h * a.dkb.sh + (int64_t)(ok ? key : 0) * a.dkb.ss;
        store_acc_rows<T, true>(row, ok, a.dkb.vec_ok, acc_b, 1.f, a.r, lane >> 5);
    }
}

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void bwd_dkv_mid_kernel(const BwdArgs a) {
    bwd_dkv_mid_body<T, C>(a, blockIdx.x);
}

template <class T, int NKD, int NKR, int MASK, bool FOLD, bool BG, int SPLIT = 1>
static hipError_t launch_dkv_mid_split(const BwdArgs &a0, hipStream_t stream) {
    typedef DkvMidCfg<T, NKD, NKR, MASK, FOLD, BG, SPLIT> C;
    BwdArgs a = a0;
    a.ntiles_n = (a.Lk + C::BN - 1) / C::BN;
    auto kern = bwd_dkv_mid_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    const int group = a.group > 1 ? a.group : 1;
    return launch_flat(kern, (int64_t)a.ntiles_n * ((a.B + group - 1) / group) * a.H, C::NTHREADS, C::LDS_BYTES, stream, a);
}

template <class T, int NKD, int NKR, int MASK, bool FOLD, bool BG>
static hipError_t launch_dkv_mid_bg(const BwdArgs &a, hipStream_t stream) {
    if (mid_split(a, a.Lk, a.Lq)) return launch_dkv_mid_split<T, NKD, NKR, MASK, FOLD, BG, 2>(a, stream);
    return launch_dkv_mid_split<T, NKD, NKR, MASK, FOLD, BG>(a, stream);
}

// (no dk_bias wanted: without its products)
template <class T, int NKD, int NKR, int MASK, bool FOLD>
static hipError_t launch_dkv_mid(const BwdArgs &a, hipStream_t stream) {
    if constexpr (NKR > 0) {
        if (a.dkb.ptr) return launch_dkv_mid_bg<T, NKD, NKR, MASK, FOLD, true>(a, stream);
    }
    return launch_dkv_mid_bg<T, NKD, NKR, MASK, FOLD, false>(a, stream);
}

} // namespace fb
