// Forward for windows: head dim 32, Lq, Lk <= 256, rank up to 16, no mask or a 16-bit matrix mask, aligned tensors (the
// window attention of 2_Vision_Transformer/swin_transformer_v2.py:178-203).  The arithmetic is that of fwd_kernel: one
// query per lane, S^T = [K | K_b] [Q | Q_b]^T, online softmax against a lagging reference point, O^T += V^T P^T with P
// from registers.
//
// The general kernel gives a window a workgroup that holds half of the compute unit's registers, and spends its life in
// turn on the first tile's way from memory, eight 32-key blocks and the stores.  Here a window's K, K_b and V take 40 KB, a
// wave works on one block of 32 queries at a time in 128 registers, and four workgroups of four waves (mask: three) or two of
// eight share a compute unit: nothing is pipelined by hand, whatever one waits for the others fill.
#include "fb_kernels.h"
#include "fb_lean_tiles.h"

namespace fb {

// FOLD_: the scores are scale * (q k^T + q_b k_b^T) in one chain (no factors, or a scale of exactly 1).
// MASK_: a matrix mask, whose blocks the wave that uses them copies to LDS one ahead.
// NWAVES_: 4, or 8 for small grids of windows of more than 128 queries (launch_fwd_win_waves).
// PAIR_: two blocks of 32 keys at a time (eight waves, and four without a mask above 64 keys).
// COS_: q and k are rows of a cosine block's projection, normalised here (fb_unit.h): K where its copies have landed in LDS, by
// the wave that copied it, Q in the registers of the block that uses it.
template <class T, int NKR_, bool FOLD_, bool MASK_, int NWAVES_, bool PAIR_, bool COS_ = false>
struct FwdWinCfg {
    static constexpr bool FOLD = FOLD_, MASK = MASK_, COS = COS_;
    static_assert(FOLD_ || !COS_, "a cosine block's scale is 1");
    static constexpr int NKD = 2, NKR = NKR_, NK = NKD + NKR_;
    static constexpr int NWAVES = NWAVES_, NTHREADS = 64 * NWAVES, LK = 256;
    static constexpr bool ONE = 32 * NWAVES >= LK;     // one window a workgroup, one block of queries a wave: nothing is kept for the next
    static constexpr bool PAIR = PAIR_;
    static constexpr int TILE = PAIR ? 4096 : 2048;    // a wave's mask tile: 32 queries x 64 or 32 keys
    static constexpr int K = 0, V = K + LK * 64, KB = V + LK * 64, MT = KB + (NKR ? LK * 32 : 0), LDS_BYTES = MT + (MASK ? NWAVES * TILE : 0);
    static constexpr int WAVES_EU = !MASK || PAIR ? 4 : 3;
    static_assert(NWAVES == 4 || NWAVES == 8, "");
    static_assert(WAVES_EU * 4 / NWAVES * LDS_BYTES <= 160 * 1024, "");
};

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void fwd_win_kernel(const FwdArgs a, int walk) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = lds_addr_of(smem);
    const int lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    // a workgroup walks `walk` consecutive batch entries of its head
    if constexpr (C::ONE) walk = 1;
    const int nbg = (a.B + walk - 1) / walk;
    const int work = xcd_remap(blockIdx.x, nbg * a.H);
    const int bg = work / a.H, h = work % a.H;
    const int nqb = (a.Lq + 31) / 32, nkb = (a.Lk + 31) / 32;

    if constexpr (C::NKR > 0) { // (the channel padding of a rank below 16 is never written)
        for (int i = threadIdx.x; i < C::LK * 2; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem + C::KB)[i] = u32x4_t{0u, 0u, 0u, 0u};
        __syncthreads();
    }
    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e, lag = 8.f / to_log2;
    const uint32_t row_off[2] = {lds0 + lean_row_addr<4>(c, g), lds0 + lean_row_addr<4>(c, 2 + g)};
    const uint32_t col_off[2] = {lds0 + C::V + lean_tr_addr4(c, g, 0), lds0 + C::V + lean_tr_addr4(c, g, 1)};
    const uint32_t kb_row = lds0 + C::KB + lean_row_addr<2>(c, g);
    const uint32_t lds_m = lds0 + C::MT + wave * C::TILE;
    float cos_scale = 1.f;
    if constexpr (C::COS) cos_scale = scale_of_head(a.cosine, h);

    for (int bi = 0; bi < walk; ++bi) {
        const int b = __builtin_amdgcn_readfirstlane(bg * walk + bi);
        if (b >= a.B) break;
        {   // K and V: 16 rows a copy instruction, whole blocks of 32 keys (rows past the end: the last one again)
            const uint8_t *kbase = reinterpret_cast<const uint8_t *>(a.k.ptr + b * a.k.sb + h * a.k.sh);
            const uint8_t *vbase = reinterpret_cast<const uint8_t *>(a.v.ptr + b * a.v.sb + h * a.v.sh);
            int row, chunk;
            lean_copy_place<4>(lane, row, chunk);
#pragma unroll
            for (int j = 0; j < C::LK / 16 / C::NWAVES; ++j) {
                const int i = wave + C::NWAVES * j, r = min(16 * i + row, a.Lk - 1);
                if (i < 2 * nkb) {
                    lds_dma16_all((uint32_t)(r * (int)(a.k.ss * 2) + chunk * 16), kbase, lds0 + C::K + i * 1024);
                    lds_dma16_all((uint32_t)(r * (int)(a.v.ss * 2) + chunk * 16), vbase, lds0 + C::V + i * 1024);
                }
            }
            if constexpr (C::NKR > 0) {
                if (bi == 0 || a.kb.sb != 0) {
                    constexpr int ROWS = 32 * C::NWAVES; // a copy instruction of each wave
                    DenseCopy<ROWS, 2> cb;
                    cb.init(a.kb.ptr + b * a.kb.sb + h * a.kb.sh, a.kb.ss, a.r, false, wave, lane, 0);
                    cb.issue(lds0 + C::KB, 0, a.Lk);
                    // (only where it has rows: the copy's offsets count down from the half's first row, unsigned)
                    if (ROWS < C::LK && a.Lk > ROWS) cb.issue(lds0 + C::KB + ROWS * 32, ROWS, a.Lk);
                }
            }
        }
        const uint16_t *qbase = a.q.ptr + b * a.q.sb + h * a.q.sh, *qbbase = C::NKR > 0 ? a.qb.ptr + b * a.qb.sb + h * a.qb.sh : nullptr;
        u32x4_t qn[C::NK]; // the next block's query operand
        auto load_q = [&](int qb) {
            const int query = min(32 * qb + c, a.Lq - 1);
#pragma unroll
            for (int t = 0; t < C::NKD; ++t) qn[t] = *reinterpret_cast<const u32x4_t *>(qbase + (int64_t)query * a.q.ss + 16 * t + 8 * g);
            if constexpr (C::NKR > 0) qn[C::NKD] = load_chunk<true>(qbbase, a.qb.ss, query, a.Lq, 8 * g, a.r);
        };
        if (wave < nqb) load_q(wave);
        // Mask tile (queries 32 qb .., keys 32 kb ..) as 32 rows of 128 (pairs of blocks) or 64 bytes; rows and 16-byte chunks
        // past the end re-read the last ones.
        const uint8_t *mbase = nullptr;
        if constexpr (C::MASK) mbase = reinterpret_cast<const uint8_t *>(a.mask.ptr) + mask_offset(a.mask, b, h) * 2;
        auto copy_mask = [&](int qb, int kb) {
            constexpr int NI = C::TILE / 1024, ROWS = 32 / NI; // copy instructions and the rows of one
            int l = lane, row, chunk;
            if constexpr (C::PAIR) asm volatile("" : "+v"(l)); // (the addresses are formed here, not kept in registers)
            lean_copy_place<4>(l, row, chunk);
            if constexpr (C::PAIR) {
                row = l >> 3;
                chunk = (l & 7) ^ swz_of<8>(row); // (rows + 8: two places further)
            }
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int col = min(32 * kb + 8 * (C::PAIR && (j & 1) ? chunk ^ 2 : chunk), a.Lk - 8);
                lds_dma16_all((uint32_t)(min(32 * qb + ROWS * j + row, a.Lq - 1) * (int)(a.mask.sm * 2) + col * 2), mbase, lds_m + j * 1024);
            }
        };
        // This half-wave's four keys of the eight from 8 i on, in this lane's row of the tile.  (Chunks differ in address bits that are
        // XORed in; eight waves: from an opaque address, or each one's is kept and fp16 spills.)
        uint32_t mrow = lds_m + (C::PAIR ? 2 * swz_off<8>(c, 0) : lean_chunk_off<4>(c, 0)) + 8 * g;
        auto mask_run = [&](int i) { return *(const __attribute__((address_space(3))) u32x2_t *)(mrow ^ (uint32_t)(16 * i)); };
        if constexpr (C::MASK) {
            if (wave < nqb) copy_mask(wave, 0);
        }
        wait_vmcnt<0>();
        if constexpr (C::COS) { // a row of this wave's by 64 / ROWS lanes
            constexpr int ROWS = C::LK / C::NWAVES, LPR = 64 / ROWS, CH = 4 / LPR;
            int l = lane;
            asm volatile("" : "+v"(l)); // (formed here, not kept in registers across the blocks)
            const int row = 16 * (wave + C::NWAVES * (l / LPR / 16)) + (l / LPR & 15);
            if (row < 32 * nkb) {
                u32x4_t x[CH];
                float sq[CH];
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    x[j] = lds_load16(lds0 + C::K + lean_chunk_off<4>(row, CH * (l % LPR) + j));
                    sq[j] = chunk_squares<T>(x[j]);
                }
                float sum = sq[0] + sq[1];
                if constexpr (CH == 4)
                    sum += sq[2] + sq[3];
                else
                    sum += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0xB1, 0xf, 0xf, true)); // lane ^ 1
                const RowNorm r = RowNorm::of<T>(sum);
#pragma unroll
                for (int j = 0; j < CH; ++j)
                    *(__attribute__((address_space(3))) u32x4_t *)(lds0 + C::K + lean_chunk_off<4>(row, CH * (l % LPR) + j)) = chunk_unit<T>(x[j], r);
            }
        }
        if (a.Lk & 31) { // V past the end: zeros in place of the last row (lds_zero16), by the waves that copied there
            int l = lane, row, chunk, last = 2 * nkb - 2;
            asm volatile("" : "+v"(l), "+s"(last)); // (formed here: ahead of the loop they cost every window's start)
            lean_copy_place<4>(l, row, chunk);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int i = last + e;
                if ((i & (C::NWAVES - 1)) == wave) lds_zero16(lds0 + C::V + i * 1024, l, 16 * i + row >= a.Lk);
            }
        }
        barrier_lds();

#pragma unroll 1
        for (int qb = wave; qb < nqb; qb += C::NWAVES) {
            if (C::PAIR && !C::ONE && qb != wave) load_q(qb); // (a block ahead, as below, it takes registers that pairs of blocks need)
            u32x4_t q[C::NK];
#pragma unroll
            for (int t = 0; t < C::NK; ++t) q[t] = qn[t];
            if (!C::PAIR && qb + C::NWAVES < nqb) load_q(qb + C::NWAVES);
            if constexpr (C::COS) {
                u32x4_t x[2] = {q[0], q[1]};
                unit_operand<T>(x);
                q[0] = chunk_times<T>(x[0], cos_scale);
                q[1] = chunk_times<T>(x[1], cos_scale);
            }
            f32x16_t o;
#pragma unroll
            for (int v = 0; v < 16; ++v) o[v] = 0.f;
            float m_ref = -INFINITY, m2 = 0.f, l_run = 0.f, slack = lag;
            // N blocks of 32 keys from block kb on.  In pairs two at a time (one test of the reference point and one set of addresses for
            // 64 keys), the last of an odd number alone: 4096 x 16 windows of 256 tokens 1430 -> 1368 us, 128 x 16 of 144 28.3 -> 27.6,
            // of 256 48.5 -> 45.5.  Masked blocks alone with four waves: the copies of two would leave two workgroups a compute unit,
            // and masks loaded to registers a pair ahead cost more (1024 x 16 of 256 473 -> 635).  Up to 128 keys alone too: the
            // first pair always moves its reference point (64 x 16 of 64 tokens 7.5, in a pair 7.9, of 100 11.3 / 11.9, of 72 9.6 / 9.8,
            // of 128 equal, 256 x 16 of 100 36.0 / 36.6).
            auto group = [&](auto tag, int kb) __attribute__((always_inline)) {
                constexpr int N = decltype(tag)::value;
                const uint32_t at = kb * 2048;
                f32x16_t s[N];
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    f32x16_t sb;
                    if constexpr (C::MASK) {
                        if (n == 0) wait_vmcnt<0>();
                        if constexpr (C::PAIR) asm volatile("" : "+v"(mrow));
#pragma unroll
                        for (int j = 0; j < 4; ++j) { // register v <-> key 8 (v / 4) + 4 g + v % 4 of the block
                            const u32x2_t x = mask_run(4 * n + j);
#pragma unroll
                            for (int e = 0; e < 2; ++e) {
                                sb[4 * j + 2 * e] = T::to_float((uint16_t)(x[e] & 0xffffu));
                                sb[4 * j + 2 * e + 1] = T::to_float((uint16_t)(x[e] >> 16));
                            }
                        }
                        if (n == N - 1) {
                            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (they have left LDS: the tile after this one)
                            if (kb + N < nkb)
                                copy_mask(qb, kb + N);
                            else if (!C::ONE && qb + C::NWAVES < nqb)
                                copy_mask(qb + C::NWAVES, 0);
                        }
                    } else {
#pragma unroll
                        for (int v = 0; v < 16; ++v) sb[v] = 0.f;
                    }
                    // q k^T and q_b k_b^T: two chains joined by the FMA that applies the softmax scale to the first (:246-256),
                    // an additive mask the initial value of the second; folded, one chain
                    if constexpr (C::FOLD)
                        s[n] = sb;
                    else
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[n][v] = 0.f;
                    // (single blocks: the other chain's product between the two of q k^T; in pairs that spills)
                    if constexpr (!C::FOLD && C::NKR > 0 && !C::PAIR) {
                        s[n] = T::mfma(lds_load16(row_off[0] + C::K + at + n * 2048), q[0], s[n]);
                        sb = T::mfma(lds_load16(kb_row + kb * 1024 + n * 1024), q[C::NKD], sb);
                        s[n] = T::mfma(lds_load16(row_off[1] + C::K + at + n * 2048), q[1], s[n]);
                    } else {
#pragma unroll
                        for (int t = 0; t < C::NKD; ++t) s[n] = T::mfma(lds_load16(row_off[t] + C::K + at + n * 2048), q[t], s[n]);
                        if constexpr (C::NKR > 0) {
                            const u32x4_t kf = lds_load16(kb_row + kb * 1024 + n * 1024);
                            if constexpr (C::FOLD)
                                s[n] = T::mfma(kf, q[C::NKD], s[n]);
                            else
                                sb = T::mfma(kf, q[C::NKD], sb);
                        }
                    }
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[n][v] = __builtin_fmaf(s[n][v], a.scale, sb[v]);
                    }
                    // (the second block's fragments are not requested ahead of the first block's scores: that spills)
                    if constexpr (N > 1) __builtin_amdgcn_sched_barrier(0);
                }
                u32x4_t vt[2];
                if constexpr (N == 1) {
#pragma unroll
                    for (int t = 0; t < 2; ++t) vt[t] = lds_load_tr(col_off[0] + at + t * 1024, col_off[1] + at + t * 1024);
                }
                if (32 * (kb + N) > a.Lk) {
#pragma unroll
                    for (int n = 0; n < N; ++n) {
                        int key0 = 32 * (kb + n) + 4 * g;
                        asm volatile("" : "+v"(key0)); // (formed in the branch)
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            if (key0 + 8 * (v >> 2) + (v & 3) >= a.Lk) s[n][v] = -INFINITY;
                    }
                }
#pragma unroll
                for (int n = 0; n < N; ++n) asm volatile("s_nop 11" : "+v"(s[n])); // (fb_bwd_win.hip: wait states across the branch above)
                // The reference point of a row moves block by block.  After a block with an even number that moved it the next one
                // moves it without a lag, so that it is the maximum of 64 keys, as in fwd_kernel: the probability 1 is the one
                // that is not rounded.  Where no row of a pair is above its reference point by the lag neither block moves one,
                // and the test of both at once is all a pair needs; pairs that move it for 64 keys at a time round the
                // probabilities of the first block against the second's maximum (error of o against float64, 769 x 8 windows of
                // 144 tokens 2.203e-3 -> 2.217e-3, fp16 2048 x 8 of 64 2.558e-4 -> 2.596e-4).
                float mx[N];
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    mx[n] = s[n][0];
#pragma unroll
                    for (int v = 1; v < 16; ++v) mx[n] = fmaxf(mx[n], s[n][v]);
                }
                const float top = half_wave_max(N == 1 ? mx[0] : fmaxf(mx[0], mx[N - 1]));
                const bool above = top > m_ref + slack; // also true for the first finite score of a row
                const bool move = __any(above);
                if constexpr (N == 1) slack = above && !(kb & 1) ? 0.f : lag;
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    if (move) {
                        if (n > 0) asm volatile("s_nop 11" : "+v"(o)); // (the first block's products)
                        const float m = N == 1 ? top : half_wave_max(mx[n]);
                        const bool grow = N == 1 ? above : m > m_ref + slack;
                        if constexpr (N > 1) slack = grow && n == 0 ? 0.f : lag;
                        const float m_new = grow ? m : m_ref;
                        const float alpha = grow ? fast_exp2((m_ref - m_new) * to_log2) : 1.f; // exp2(-inf) = 0
                        l_run *= alpha;
#pragma unroll
                        for (int v = 0; v < 16; ++v) o[v] *= alpha;
                        m_ref = m_new;
                        m2 = reference_log2<T>(m_new, to_log2);
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        if constexpr (N > 1) vt[t] = lds_load_tr(col_off[0] + at + n * 2048 + t * 1024, col_off[1] + at + n * 2048 + t * 1024);
                        u32x4_t pb;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float p0 = fast_exp2(__builtin_fmaf(s[n][8 * t + 2 * e], to_log2, -m2));
                            const float p1 = fast_exp2(__builtin_fmaf(s[n][8 * t + 2 * e + 1], to_log2, -m2));
                            pb[e] = T::pack2(p0, p1);
                            l_run += p0 + p1;
                        }
                        o = T::mfma(vt[t], pb, o);
                    }
                }
                asm volatile("s_nop 11" : "+v"(o)); // (across the loop's branches)
            };
            if constexpr (!C::PAIR) {
#pragma unroll 1
                for (int kb = 0; kb < nkb; ++kb) group(std::integral_constant<int, 1>{}, kb);
            } else {
#pragma unroll 1
                for (int kb = 0; kb + 1 < nkb; kb += 2) group(std::integral_constant<int, 2>{}, kb);
                if (nkb & 1) group(std::integral_constant<int, 1>{}, nkb - 1);
            }
            const float l = l_run + __shfl_xor(l_run, 32, 64);
            const int query = 32 * qb + c;
            const bool ok = query < a.Lq;
            if (ok && g == 0) a.lse[((int64_t)b * a.H + h) * a.Lq + query] = m_ref * (C::FOLD ? a.scale : 1.f) + __builtin_amdgcn_logf(l) * kLn2;
            uint16_t *orow = const_cast<uint16_t *>(a.o.ptr) + b * a.o.sb + h * a.o.sh + (int64_t)(ok ? query : 0) * a.o.ss;
            store_acc_rows<T, true>(orow, ok, true, o, 1.f / l, a.d, g);
            if constexpr (C::ONE) break;
        }
        if (bi + 1 < walk) barrier_lds(); // everyone has read K and V
    }
}

template <class T, int NKR, bool FOLD, bool MASK, int NWAVES, bool PAIR, bool COS>
static hipError_t launch_fwd_win_cfg(const FwdArgs &a, hipStream_t stream) {
    typedef FwdWinCfg<T, NKR, FOLD, MASK, NWAVES, PAIR, COS> C;
    auto kern = fwd_win_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    int walk = 1;
    for (int w = C::ONE ? 1 : 8; w > 1; w /= 2)
        if ((int64_t)((a.B + w - 1) / w) * a.H >= 16 * (int64_t)num_cus()) {
            walk = w;
            break;
        }
    const int64_t total = (int64_t)((a.B + walk - 1) / walk) * a.H;
    if (total <= 0 || total > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    (void)hipGetLastError();
    hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(C::NTHREADS), C::LDS_BYTES, stream, a, walk);
    return hipGetLastError();
}

// Eight waves, one block of queries each, where a grid leaves compute units with fewer than four workgroups: twice the waves a
// SIMD, and half as long a walk.  Four waves against eight, rank 16, us: 512 windows of 256 tokens 15.5 / 14.4, of 196 15.5 / 12.7, of 144
// 11.1 / 9.1, with a mask (144, 256) 12.9 / 10.9, 21.0 / 18.7; 1024 windows of 256 29.3 / 26.2, of 196 24.5 / 22.8, with a mask
// 22.9 / 20.0, 35.6 / 31.3; 2048 of 256 47.1 / 45.4, with a mask 37.6 / 35.8, 57.0 / 54.6.  Without a mask and with at most six blocks of
// queries the idle waves count from 512 windows on (1024 of 144 15.5 / 16.7, 2048 28.2 / 30.2), above 2048 windows they do
// everywhere (3072 of 144 with a mask 49.6 / 51.1, 8192 of 256 241 / 245).
template <class T, int NKR, bool FOLD, bool MASK, bool COS = false>
static hipError_t launch_fwd_win_waves(const FwdArgs &a, hipStream_t stream) {
    const int64_t windows = (int64_t)a.B * a.H;
    const bool wide = a.Lq > 128 && (windows <= 2 * (int64_t)num_cus() || ((MASK || a.Lq > 192) && windows <= 8 * (int64_t)num_cus()));
    if (wide) return launch_fwd_win_cfg<T, NKR, FOLD, MASK, 8, true, COS>(a, stream);
    if constexpr (!MASK) {
        if (a.Lk > 128) return launch_fwd_win_cfg<T, NKR, FOLD, MASK, 4, true, COS>(a, stream);
    }
    return launch_fwd_win_cfg<T, NKR, FOLD, MASK, 4, false, COS>(a, stream);
}

template <class T, int NKR>
static hipError_t launch_fwd_win_r(const FwdArgs &a, hipStream_t stream) {
    if (a.cosine.ptr)
        return a.mask.type == kMatrixMask ? launch_fwd_win_waves<T, NKR, true, true, true>(a, stream) : launch_fwd_win_waves<T, NKR, true, false, true>(a, stream);
    if (a.mask.type == kMatrixMask) // (the mask is not divided by the scale)
        return a.scale == 1.f ? launch_fwd_win_waves<T, NKR, true, true>(a, stream) : launch_fwd_win_waves<T, NKR, false, true>(a, stream);
    return a.r == 0 || a.scale == 1.f ? launch_fwd_win_waves<T, NKR, true, false>(a, stream) : launch_fwd_win_waves<T, NKR, false, false>(a, stream);
}

// Compiled once per element type for head dim 32 (see Makefile).  When fb_fwd takes this path is decided by
// window_forward() in fb_kernels.h.
#define FB_CAT2(a, b) a##b
#define FB_CAT(a, b) FB_CAT2(a, b)
hipError_t FB_CAT(launch_fwd_win_, FB_SUFFIX)(const FwdArgs &a, hipStream_t stream) {
    return a.r == 0 ? launch_fwd_win_r<FB_T, 0>(a, stream) : launch_fwd_win_r<FB_T, 1>(a, stream);
}

} // namespace fb
