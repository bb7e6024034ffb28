// Backward FlashBias attention for gfx950, window regime without factor gradients: dq, dk and dv of one
// (batch, head) in one workgroup when the whole sequence fits it (Lq, Lk <= 256: the window attention of
// 2_Vision_Transformer/swin_transformer_v2.py:178-203, whose factors are constants).  Replaces the key-block loop
// of _bwd_kernel_one_col_block (flash_bias/flash_bias_triton.py:575-869) without its factor gradients, as
// fb_bwd_win.hip does with them.
//
// fb_bwd_win.hip gives a window a whole compute unit: eight waves that pass the same barriers, so that copies, the
// dk/dv products and the dq products (which need the dS of all keys) follow each other and nothing overlaps.  Here a
// window is a workgroup of four waves in 80 KB, two of them share a compute unit, and whatever one waits for the
// other fills.  What makes it small is that dS never leaves its wave: wave w owns keys [64 w, 64 w + 64) (K, K_b, V
// and the K^T operand of dq in registers), transposes its own 32 x 32 block of dS through 2 KB of LDS that no other
// wave touches, and adds its keys' share to the block's dq accumulator, which travels from wave to wave:
//
//   queries in halves of 128, a half in four steps; at step s wave w takes query block (s + w) % 4, reads the
//   block's dq accumulator (4 KB of LDS; at step 0 it starts at zero), adds its 64 keys and hands it on; at
//   step 3 it is complete and goes to memory.  One barrier a step, no two waves at one accumulator.
//
// Every query-side fragment (Q, Q_b, dO by rows and by columns) is read once per 64 keys, half of what 32 keys a
// wave take.  All sums have a fixed order: the results are bit-reproducible.
//
// 4096 x 16 windows of 256 tokens, rank 16, bf16: 3.97 ms in the window kernel, 2.85 here; 1024 x 16 with shifted-window
// masks 1.36 and 0.95.  Loads and stores alone take 1.9 ms (8.6 GB; the loads 1.08), the matrix pipe is busy for a
// fifth of the time, the vector units for two: two waves per SIMD (240 registers) do not cover each other entirely, and
// what would pipeline the blocks of one wave does not fit beside its operands.
#include "fb_kernels.h"
#include "fb_lean_tiles.h"

namespace fb {

// NKR_: 16-wide steps of the rank (0, 1).  FOLD_: the scores are scale * (q k^T + q_b k_b^T), no multiply per score
// for the scale (no factors and a positive scale, or a scale of exactly 1).  MASK_: an additive mask of the 16-bit type, a vector mask as
// one value per lane (key) or a matrix mask as a 32 x 32 tile per block, copied to LDS by the wave that uses it.
// HIDE_: some wave's 64 keys are not all there, their scores are set to -inf (a branch on it inside the step cost 200
// bytes of scratch).
// COS_: q and k are rows of a cosine block's projection, normalised here as in the forward (fb_unit.h), and dq and dk become the
// projection's gradients where they are stored.  The rows of a dq block come from memory a second time, copied to where the block's
// accumulator was while its last step runs, the rows of K are this wave's operand, and a row's norm and reciprocal are kept in LDS
// (16 x 64 x 16 windows of 256 tokens with masks: both formed again from rows loaded at the end 1074 us, norms and K kept 1037, rows copied ahead
// and bf16 quotients without a correction 1000).
template <class T, int NKR_, bool FOLD_, int MASK_, bool HIDE_, bool COS_ = false>
struct RingCfg {
    static constexpr bool HIDE = HIDE_, COS = COS_;
    static_assert(FOLD_ || !COS_, "a cosine block's scale is 1");
    static constexpr bool FOLD = FOLD_, MASK = MASK_ == kMatrixMask, VMASK = MASK_ == kVectorMask;
    static constexpr int NKD = 2, NKR = NKR_, NK = NKD + NKR_;
    static constexpr int NWAVES = 4, NTHREADS = 64 * NWAVES, KBW = 2, LQ = 256, HALF = 128;
    // LDS, bytes: dense regions of 64-byte rows (Q, dO) and 32-byte rows (Q_b), the four accumulators of a half, a
    // dS block per wave, statistics, a mask tile per wave
    static constexpr int Q = 0, DO = Q + LQ * 64, QB = DO + LQ * 64, ACC = QB + (NKR ? LQ * 32 : 0), DS = ACC + 4 * 4096,
                         STAT = DS + NWAVES * 2048, MT = STAT + 2 * LQ * 4,
                         NORM = MT + (MASK ? NWAVES * 2048 : 0), LDS_BYTES = NORM + (COS ? 4 * LQ * 4 + NTHREADS * 4 : 0); // (NORM: of Q's rows, of K's, then a thread's sum(dq * unit q))
    static_assert(LDS_BYTES <= 80 * 1024, "two workgroups per compute unit");
};

// A 32 x 32 accumulator block (lane = row, as store_acc_rows takes it) to rows [row0, row0 + 32) of a tensor through 2 KB
// of LDS that only this wave touches: packed, written by rows, read back in the order of a copy (lean_copy_place), so
// that four neighbouring lanes store a row of 64 bytes.
template <class T>
__device__ __forceinline__ void store_block_rows(const Tensor &t, int b, int h, int row0, int nrows, const f32x16_t &acc, float mul,
                                                 uint8_t *buf, int lane) {
    const int c = lane & 31, g = lane >> 5;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        *reinterpret_cast<u32x2_t *>(buf + lean_chunk_off<4>(c, j) + 8 * g) =
            u32x2_t{T::pack2(acc[4 * j] * mul, acc[4 * j + 1] * mul), T::pack2(acc[4 * j + 2] * mul, acc[4 * j + 3] * mul)};
    uint16_t *base = const_cast<uint16_t *>(t.ptr) + b * t.sb + h * t.sh;
    int row, chunk;
    lean_copy_place<4>(lane, row, chunk);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const u32x4_t x = *reinterpret_cast<const u32x4_t *>(buf + j * 1024 + lane * 16);
        const int r = row0 + 16 * j + row;
        if (r < nrows) *reinterpret_cast<u32x4_t *>(base + (int64_t)r * t.ss + 8 * chunk) = x;
    }
}

// The same for the gradient g of unit rows n = x / |x|, which becomes that of x: s (g - n (n . g)) / |x|, as cosine_bwd_kernel forms it
// from the rounded g.  The rows' n: this wave's operand `unit` (UNIT: K), or from the block's rows of x in LDS at `raw`, in the order of a copy
// (Q, whose tile holds the products with the scale); `norms`: |x| of the block's rows and, 256 floats on, what they are multiplied
// by.  Returns this lane's share of sum(g n).
template <class T, bool UNIT>
__device__ __forceinline__ float store_block_rows_unit(const Tensor &t, const u32x4_t (&unit)[2], const uint8_t *raw, const float *norms, int b, int h, int row0,
                                                       int nrows, const f32x16_t &acc, float s, uint8_t *buf, int lane) {
    asm volatile("" : "+v"(lane)); // (what derives from it is formed here, not kept in registers across the steps)
    const int c = lane & 31, g = lane >> 5;
    uint16_t *base = const_cast<uint16_t *>(t.ptr) + b * t.sb + h * t.sh;
    int row, chunk;
    lean_copy_place<4>(lane, row, chunk);
    u32x4_t x[2];
    if constexpr (UNIT) {
#pragma unroll
        for (int k = 0; k < 2; ++k) *reinterpret_cast<u32x4_t *>(buf + lean_chunk_off<4>(c, 2 * k + g)) = unit[k];
#pragma unroll
        for (int j = 0; j < 2; ++j) x[j] = *reinterpret_cast<const u32x4_t *>(buf + j * 1024 + lane * 16);
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) x[j] = *reinterpret_cast<const u32x4_t *>(raw + j * 1024 + lane * 16);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        *reinterpret_cast<u32x2_t *>(buf + lean_chunk_off<4>(c, j) + 8 * g) =
            u32x2_t{T::pack2(acc[4 * j], acc[4 * j + 1]), T::pack2(acc[4 * j + 2], acc[4 * j + 3])};
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float gr[8], n[8];
        chunk_floats<T>(*reinterpret_cast<const u32x4_t *>(buf + j * 1024 + lane * 16), gr);
        const int at = row0 + 16 * j + row;
        const bool ok = at < nrows;
        RowNorm r;
        r.norm = norms[16 * j + row];
        r.inv = norms[256 + 16 * j + row];
        r.template finish<T>();
        if constexpr (!UNIT) x[j] = chunk_unit<T>(x[j], r);
        chunk_floats<T>(x[j], n);
        float dot = 0.f;
        if constexpr (!UNIT) { // (the scale's own gradient; k has none)
            float mine = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                mine = __builtin_fmaf(gr[e], n[e], mine);
                gr[e] *= s;
            }
            sum += ok ? mine : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(gr[e], n[e], dot);
        dot = quad_sum(dot);
        if (r.norm < round16<T>(kNormEps)) dot = 0.f; // (a row of zeros: the clamped denominator is a constant)
#pragma unroll
        for (int e = 0; e < 8; ++e) gr[e] = (gr[e] - n[e] * dot) * r.inv;
        if (ok)
            *reinterpret_cast<u32x4_t *>(base + (int64_t)at * t.ss + 8 * chunk) =
                u32x4_t{T::pack2(gr[0], gr[1]), T::pack2(gr[2], gr[3]), T::pack2(gr[4], gr[5]), T::pack2(gr[6], gr[7])};
    }
    return sum;
}

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void bwd_ring_kernel(const BwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = lds_addr_of(smem);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    // a workgroup walks `walk` consecutive batch entries of its head
    const int walk = a.walk > 1 ? a.walk : 1;
    const int nbg = (a.B + walk - 1) / walk;
    const int work = xcd_remap(blockIdx.x, nbg * a.H);
    const int bg = work / a.H, h = work % a.H;
    const int wk0 = 64 * wave; // first key of this wave
    const bool visible = wk0 < a.Lk;

    if constexpr (C::NKR > 0) { // (the channel padding of a rank below 16 is never written)
        for (int i = threadIdx.x; i < C::LQ * 2; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem + C::QB)[i] = u32x4_t{0u, 0u, 0u, 0u};
        __syncthreads();
    }
    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e;
    u32x4_t kbr[C::KBW][C::NKR > 0 ? C::NKR : 1]; // (kept across entries when the batch shares the factor)
    float cos_scale = 1.f;
    float *sNorm = reinterpret_cast<float *>(smem + C::NORM);
    if constexpr (C::COS) {
        cos_scale = scale_of_head(a.cosine, h);
        sNorm[4 * C::LQ + threadIdx.x] = 0.f;
    }

    for (int bi = 0; bi < walk; ++bi) {
        const int b = __builtin_amdgcn_readfirstlane(bg * walk + bi);
        if (b >= a.B) break;
        int tid_again = threadIdx.x; // (opaque: what derives from the lane id is recomputed per entry, not kept in registers)
        asm volatile("" : "+v"(tid_again));
        const int tid = tid_again, lane = tid & 63, c = lane & 31, g = lane >> 5;

        // ---- copies of the query side (every wave has left the previous entry's tiles: the barrier that ends a step);
        // wave w copies rows [64 w, 64 w + 64) of Q and dO, rows past the end re-read the last one
        {
            LeanCopy4<C::LQ> cq, cd;
            cq.init(wave, lane, a.q.ss);
            cd.init(wave, lane, a.dout.ss);
            cq.issue(reinterpret_cast<const uint8_t *>(a.q.ptr + b * a.q.sb + h * a.q.sh), lds0 + C::Q, wave, lane, a.Lq);
            cd.issue(reinterpret_cast<const uint8_t *>(a.dout.ptr + b * a.dout.sb + h * a.dout.sh), lds0 + C::DO, wave, lane, a.Lq);
            if constexpr (C::NKR > 0) {
                if (bi == 0 || a.qb.sb != 0) {
                    DenseCopy<C::LQ / 2, 2> cb;
                    cb.init(a.qb.ptr + b * a.qb.sb + h * a.qb.sh, a.qb.ss, a.r, false, wave, lane, 0);
                    cb.issue(lds0 + C::QB, 0, a.Lq);
                    // (only where it has rows: the copy's offsets count down from the half's first row, unsigned)
                    if (a.Lq > C::LQ / 2) cb.issue(lds0 + C::QB + C::LQ * 16, C::LQ / 2, a.Lq);
                }
            }
        }
        // ---- key-side operands, resident in registers (keys past the end: the last one, whose scores are hidden)
        u32x4_t kr[C::KBW][C::NKD], vr[C::KBW][C::NKD], kt[C::KBW][2];
#pragma unroll
        for (int kb = 0; kb < C::KBW; ++kb) {
            const int key = min(wk0 + 32 * kb + c, a.Lk - 1);
            const uint16_t *krow = a.k.ptr + b * a.k.sb + h * a.k.sh + (int64_t)key * a.k.ss + 8 * g;
            const uint16_t *vrow = a.v.ptr + b * a.v.sb + h * a.v.sh + (int64_t)key * a.v.ss + 8 * g;
#pragma unroll
            for (int t = 0; t < C::NKD; ++t) {
                kr[kb][t] = *reinterpret_cast<const u32x4_t *>(krow + 16 * t);
                vr[kb][t] = *reinterpret_cast<const u32x4_t *>(vrow + 16 * t);
            }
            if constexpr (C::NKR > 0) {
                if (bi == 0 || a.kb.sb != 0)
                    kbr[kb][0] = load_chunk<true>(a.kb.ptr + b * a.kb.sb + h * a.kb.sh, a.kb.ss, key, a.Lk, 8 * g, a.r);
            }
        }
        float mkey[C::KBW]; // vector mask: the values of this lane's keys
        const uint8_t *mbase = nullptr;
        if constexpr (C::VMASK) {
#pragma unroll
            for (int kb = 0; kb < C::KBW; ++kb)
                mkey[kb] = T::to_float(reinterpret_cast<const uint16_t *>(a.mask.ptr)[mask_offset(a.mask, b, h) + min(wk0 + 32 * kb + c, a.Lk - 1)]);
        }
        // Matrix mask: the tile (queries r0 .., keys k0 ..) as 32 rows of 64 bytes, two copy instructions of the wave that
        // reads it; rows and 16-byte chunks past the end re-read the last ones.
        const uint32_t lds_m = lds0 + C::MT + wave * 2048;
        if constexpr (C::MASK) mbase = reinterpret_cast<const uint8_t *>(a.mask.ptr) + mask_offset(a.mask, b, h) * 2;
        auto copy_mask = [&](int r0, int k0) {
            int row, chunk;
            lean_copy_place<4>(lane, row, chunk);
            const int col = min(k0 + 8 * chunk, a.Lk - 8);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                lds_dma16_all((uint32_t)(min(r0 + 16 * j + row, a.Lq - 1) * (int)(a.mask.sm * 2) + col * 2), mbase, lds_m + j * 1024);
        };
        if constexpr (C::MASK) {
            if (visible) copy_mask(32 * wave, wk0);
        }

        // ---- statistics of query `tid` (_bwd_preprocess_do_o_dot, flash_bias_triton.py:358-400): -delta = -rowsum(o * dO)
        // and lse * log2(e); queries past the end get P = 0
        {
            const int row = min(tid, a.Lq - 1);
            const uint16_t *orow = a.o.ptr + b * a.o.sb + h * a.o.sh + (int64_t)row * a.o.ss;
            u32x4_t so[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) so[j] = *reinterpret_cast<const u32x4_t *>(orow + 8 * j);
            const float slse = a.lse[((int64_t)b * a.H + h) * a.Lq + row];
            if constexpr (C::COS) {
#pragma unroll
                for (int kb = 0; kb < C::KBW; ++kb) {
                    const RowNorm r = unit_operand<T>(kr[kb]);
                    sNorm[2 * C::LQ + wk0 + 32 * kb + c] = r.norm;
                    sNorm[3 * C::LQ + wk0 + 32 * kb + c] = r.inv;
                }
            }
            // K^T: this wave's rows of K through the first 16 KB of the accumulators (free until step 0, and the block
            // that this wave writes first)
            const uint32_t kst = lds0 + C::ACC + wave * 4096;
#pragma unroll
            for (int kb = 0; kb < C::KBW; ++kb)
#pragma unroll
                for (int t = 0; t < C::NKD; ++t)
                    *reinterpret_cast<u32x4_t *>(smem + C::ACC + wave * 4096 + kb * 2048 + lean_chunk_off<4>(c, 2 * t + g)) = kr[kb][t];
#pragma unroll
            for (int kb = 0; kb < C::KBW; ++kb)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    kt[kb][t] = lds_load_tr(kst + lean_tr_addr4(c, g, 0) + (2 * kb + t) * 1024, kst + lean_tr_addr4(c, g, 1) + (2 * kb + t) * 1024);
            wait_vmcnt<0>(); // this wave's copies have landed, among them row `tid` of Q and dO
            if constexpr (C::COS) {
                u32x4_t x[4];
                float sq[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    x[j] = lds_load16(lds0 + C::Q + lean_chunk_off<4>(tid, j));
                    sq[j] = chunk_squares<T>(x[j]);
                }
                const RowNorm r = RowNorm::of<T>((sq[0] + sq[1]) + (sq[2] + sq[3]));
                sNorm[tid] = r.norm;
                sNorm[C::LQ + tid] = r.inv;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *(__attribute__((address_space(3))) u32x4_t *)(lds0 + C::Q + lean_chunk_off<4>(tid, j)) = chunk_times<T>(chunk_unit<T>(x[j], r), cos_scale);
            }
            float sum[2];
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                sum[half] = 0.f;
#pragma unroll
                for (int j = 2 * half; j < 2 * half + 2; ++j) {
                    const u32x4_t sd = lds_load16(lds0 + C::DO + lean_chunk_off<4>(tid, j));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sum[half] = __builtin_fmaf(T::to_float((uint16_t)(so[j][e] & 0xffffu)), T::to_float((uint16_t)(sd[e] & 0xffffu)), sum[half]);
                        sum[half] = __builtin_fmaf(T::to_float((uint16_t)(so[j][e] >> 16)), T::to_float((uint16_t)(sd[e] >> 16)), sum[half]);
                    }
                }
            }
            float *sStat = reinterpret_cast<float *>(smem + C::STAT);
            const bool ok = tid < a.Lq;
            sStat[tid] = ok ? slse * kLog2e : INFINITY;
            sStat[C::LQ + tid] = ok ? -(sum[0] + sum[1]) : 0.f;
        }
        f32x16_t acc_dv[C::KBW], acc_dk[C::KBW];
#pragma unroll
        for (int kb = 0; kb < C::KBW; ++kb)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc_dv[kb][v] = acc_dk[kb][v] = 0.f;
        barrier_lds();

        const uint32_t row_off[2] = {lean_row_addr<4>(c, g), lean_row_addr<4>(c, 2 + g)};
        const uint32_t col_off[2] = {lean_tr_addr4(c, g, 0), lean_tr_addr4(c, g, 1)};
        const uint32_t qb_row = lds0 + C::QB + lean_row_addr<2>(c, g);

        const int nsteps = a.Lq > C::HALF ? 8 : 4;
#pragma unroll 1
        for (int step = 0; step < nsteps; ++step) {
            const int blk = (step + wave) & 3, r0 = (step >> 2) * C::HALF + 32 * blk; // this wave's query block
            const int next_r0 = ((step + 1) >> 2) * C::HALF + 32 * ((step + 1 + wave) & 3);
            f32x16_t dq;
            float *acc = reinterpret_cast<float *>(smem + C::ACC + blk * 4096 + lane * 16);
            if ((step & 3) == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) dq[v] = 0.f;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4_t x = *reinterpret_cast<const f32x4_t *>(acc + 256 * j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dq[4 * j + e] = x[e];
                }
            }
            // The raw rows of the block that this step completes, for store_block_rows_unit, to where its accumulator was.
            if constexpr (C::COS) {
                if ((step & 3) == 3 && r0 < a.Lq) {
                    int row, chunk, l = lane;
                    asm volatile("" : "+v"(l));
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (the accumulator has left LDS)
                    lean_copy_place<4>(l, row, chunk);
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        lds_dma16_all((uint32_t)(min(r0 + 16 * j + row, a.Lq - 1) * (int)(a.q.ss * 2) + chunk * 16),
                                      reinterpret_cast<const uint8_t *>(a.q.ptr + b * a.q.sb + h * a.q.sh), lds0 + C::ACC + blk * 4096 + j * 1024);
                }
            }
            if (visible && r0 < a.Lq) {
                const uint32_t rows = lds0 + (r0 >> 5) * 2048;
                u32x4_t qa[C::NK], da[C::NKD];
#pragma unroll
                for (int t = 0; t < C::NKD; ++t) {
                    qa[t] = lds_load16(rows + C::Q + row_off[t]);
                    da[t] = lds_load16(rows + C::DO + row_off[t]);
                }
                if constexpr (C::NKR > 0) qa[C::NKD] = lds_load16(qb_row + (r0 >> 5) * 1024);
                f32x16_t lse2;
                auto lses = [&]() { // register v <-> query r0 + 8 (v / 4) + 4 g + v % 4
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(smem + C::STAT + 4 * (r0 + 8 * j + 4 * g));
#pragma unroll
                        for (int e = 0; e < 4; ++e) lse2[4 * j + e] = x[e];
                    }
                };
                u32x4_t mt[2]; // mask values of the block, packed in the same order
                auto mask_tile = [&](int kb) {
                    if constexpr (C::MASK) {
                        wait_vmcnt<0>();
#pragma unroll
                        for (int t = 0; t < 2; ++t) mt[t] = lds_load_tr(lds_m + col_off[0] + t * 1024, lds_m + col_off[1] + t * 1024);
                        // the tile after this one, once these values have left LDS: the other key block, then the next step's
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        if (kb + 1 < C::KBW)
                            copy_mask(r0, wk0 + 32 * kb + 32);
                        else if (step + 1 < nsteps)
                            copy_mask(next_r0, wk0);
                    }
                };
                auto mask_at = [&](int v) { return T::to_float((uint16_t)(v & 1 ? mt[v >> 3][(v & 7) >> 1] >> 16 : mt[v >> 3][(v & 7) >> 1] & 0xffffu)); };
                auto scores = [&](int kb, f32x16_t &s) { // q k^T
                    mask_tile(kb);
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[v] = C::FOLD && C::MASK ? mask_at(v) : 0.f;
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) s = T::mfma(qa[t], kr[kb][t], s);
                };
                auto bias = [&](int kb, f32x16_t &s) { // the softmax scale multiplies q k^T only (flash_bias_triton.py:248)
                    if constexpr (!C::FOLD) {
#pragma unroll
                        for (int v = 0; v < 16; ++v)
                            s[v] = C::MASK ? __builtin_fmaf(s[v], a.scale, mask_at(v)) : C::VMASK ? __builtin_fmaf(s[v], a.scale, mkey[kb]) : s[v] * a.scale;
                    }
                    if constexpr (C::NKR > 0) s = T::mfma(qa[C::NKD], kbr[kb][0], s);
                    if constexpr (C::HIDE) {
                        const int key = wk0 + 32 * kb + c;
#pragma unroll
                        for (int v = 0; v < 16; ++v) s[v] = key < a.Lk ? s[v] : -INFINITY;
                    }
                };
                auto deltas = [&](f32x16_t &dp) { // dO V^T - delta: -delta is the initial value
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(smem + C::STAT + 4 * (C::LQ + r0 + 8 * j + 4 * g));
#pragma unroll
                        for (int e = 0; e < 4; ++e) dp[4 * j + e] = x[e];
                    }
                };
                auto grads = [&](int kb, f32x16_t &dp) {
#pragma unroll
                    for (int t = 0; t < C::NKD; ++t) dp = T::mfma(da[t], vr[kb][t], dp);
                };
                // P and dS, packed per 16-query step; dS of (this key, queries 16 t + 8 half + 4 g + 0..3) also to row c of the
                // wave's dS block, which comes back column-wise (lane = query)
                const uint32_t ds = lds0 + C::DS + wave * 2048;
                u32x4_t pp[2], pds[2], dsb[2];
                auto probs = [&](const f32x16_t &s, const f32x16_t &dp) {
#pragma unroll
                    for (int v = 0; v < 16; v += 2) {
                        const float p0 = fast_exp2(__builtin_fmaf(s[v], to_log2, -lse2[v]));
                        const float p1 = fast_exp2(__builtin_fmaf(s[v + 1], to_log2, -lse2[v + 1]));
                        pp[v >> 3][(v & 7) >> 1] = T::pack2(p0, p1);
                        pds[v >> 3][(v & 7) >> 1] = T::pack2(p0 * dp[v], p1 * dp[v + 1]);
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int half = 0; half < 2; ++half)
                            *reinterpret_cast<u32x2_t *>(smem + C::DS + wave * 2048 + lean_chunk_off<4>(c, 2 * t + half) + 8 * g) =
                                u32x2_t{pds[t][2 * half], pds[t][2 * half + 1]};
                };
                auto block_back = [&]() {
#pragma unroll
                    for (int t = 0; t < 2; ++t) dsb[t] = lds_load_tr(ds + col_off[0] + t * 1024, ds + col_off[1] + t * 1024);
                };
                u32x4_t dot[2], qt[2]; // dO^T and Q^T of the block, for both key blocks
                auto sums = [&](int kb) { // dV^T += dO^T P ; dK^T += Q^T dS  (contraction over the block's queries)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        acc_dv[kb] = T::mfma(dot[t], pp[t], acc_dv[kb]);
                        acc_dk[kb] = T::mfma(qt[t], pds[t], acc_dk[kb]);
                    }
                };
                auto query_sums = [&](int kb) { // dQ^T += K^T dS^T over the 32 keys
#pragma unroll
                    for (int t = 0; t < 2; ++t) dq = T::mfma(kt[kb][t], dsb[t], dq);
                };
                auto columns = [&]() {
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        dot[t] = lds_load_tr(rows + C::DO + col_off[0] + t * 1024, rows + C::DO + col_off[1] + t * 1024);
                        qt[t] = lds_load_tr(rows + C::Q + col_off[0] + t * 1024, rows + C::Q + col_off[1] + t * 1024);
                    }
                };
                // The second block's first products stand between the first one's dS and its way back from LDS, and the
                // wave that feeds the matrix pipe goes first.  4096 x 16 windows of 256 tokens, rank 16: block after block
                // 3.10 ms, this order 2.95, with the priorities 2.89.  A matrix mask's values do not fit beside two blocks.
                if constexpr (!C::MASK) {
                    f32x16_t s0, dp0, s1, dp1;
                    __builtin_amdgcn_s_setprio(1);
                    lses();
                    deltas(dp0);
                    scores(0, s0);
                    grads(0, dp0);
                    bias(0, s0);
                    columns();
                    __builtin_amdgcn_s_setprio(0);
                    probs(s0, dp0);
                    __builtin_amdgcn_s_setprio(1);
                    block_back();
                    deltas(dp1);
                    scores(1, s1);
                    sums(0);
                    grads(1, dp1);
                    bias(1, s1);
                    lses();
                    query_sums(0);
                    __builtin_amdgcn_s_setprio(0);
                    probs(s1, dp1);
                    __builtin_amdgcn_s_setprio(1);
                    block_back();
                    sums(1);
                    query_sums(1);
                } else {
#pragma unroll
                    for (int kb = 0; kb < C::KBW; ++kb) {
                        f32x16_t s, dp;
                        __builtin_amdgcn_s_setprio(1);
                        scores(kb, s);
                        deltas(dp);
                        grads(kb, dp);
                        bias(kb, s);
                        lses();
                        __builtin_amdgcn_s_setprio(0);
                        probs(s, dp);
                        __builtin_amdgcn_s_setprio(1);
                        columns();
                        block_back();
                        sums(kb);
                        query_sums(kb);
                    }
                }
                __builtin_amdgcn_s_setprio(0);
            } else if (C::MASK && visible && step + 1 < nsteps) { // (a block past the end: its tile is replaced by the next step's)
                wait_vmcnt<0>();
                copy_mask(next_r0, wk0);
            }
            asm volatile("s_nop 11" : "+v"(dq)); // (as above: the branch around the products)
            if ((step & 3) < 3) {
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4_t *>(acc + 256 * j) = f32x4_t{dq[4 * j], dq[4 * j + 1], dq[4 * j + 2], dq[4 * j + 3]};
            } else if constexpr (C::COS) {
                if (r0 < a.Lq) {
                    wait_vmcnt<0>();
                    sNorm[4 * C::LQ + threadIdx.x] += store_block_rows_unit<T, false>(a.dq, kr[0], smem + C::ACC + blk * 4096, sNorm + r0, b, h, r0, a.Lq, dq, cos_scale, smem + C::DS + wave * 2048, lane);
                }
            } else {
                store_block_rows<T>(a.dq, b, h, r0, a.Lq, dq, a.scale, smem + C::DS + wave * 2048, lane);
            }
            barrier_lds(); // the accumulators are handed on
        }

#pragma unroll
        for (int kb = 0; kb < C::KBW; ++kb) {
            asm volatile("s_nop 11" : "+v"(acc_dv[kb]), "+v"(acc_dk[kb]));
            store_block_rows<T>(a.dv, b, h, wk0 + 32 * kb, a.Lk, acc_dv[kb], 1.f, smem + C::DS + wave * 2048, lane);
            if constexpr (C::COS) {
                if (wk0 + 32 * kb < a.Lk)
                    store_block_rows_unit<T, true>(a.dk, kr[kb], nullptr, sNorm + 2 * C::LQ + wk0 + 32 * kb, b, h, wk0 + 32 * kb, a.Lk, acc_dk[kb], 1.f, smem + C::DS + wave * 2048, lane);
            } else {
                store_block_rows<T>(a.dk, b, h, wk0 + 32 * kb, a.Lk, acc_dk[kb], a.scale, smem + C::DS + wave * 2048, lane);
            }
        }
    }
    if constexpr (C::COS) { // this wave's share of the head's sum(dq * unit q), in a fixed order
        float cos_sum = quad_sum(sNorm[4 * C::LQ + threadIdx.x]);
#pragma unroll
        for (int m = 4; m < 64; m <<= 1) cos_sum += __shfl_xor(cos_sum, m, 64);
        if ((threadIdx.x & 63) == 0) a.cosine_partial[((int64_t)h * nbg + bg) * C::NWAVES + wave] = cos_sum;
    }
}

template <class T, int NKR, bool FOLD, int MASK, bool HIDE, bool COS = false>
static hipError_t launch_ring_cfg(const BwdArgs &a, hipStream_t stream) {
    typedef RingCfg<T, NKR, FOLD, MASK, HIDE, COS> C;
    auto kern = bwd_ring_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    BwdArgs b = a;
    b.walk = ring_walk(a.B, a.H);
    return launch_flat(kern, (int64_t)((a.B + b.walk - 1) / b.walk) * a.H, C::NTHREADS, C::LDS_BYTES, stream, b);
}

template <class T, int NKR, int MASK>
static hipError_t launch_ring_m(const BwdArgs &a, bool fold, hipStream_t stream) {
    const bool hide = a.Lk % 64 != 0;
    if constexpr (MASK != kVectorMask) // (there the mask rides on the scale's FMA)
        if (fold) return hide ? launch_ring_cfg<T, NKR, true, MASK, true>(a, stream) : launch_ring_cfg<T, NKR, true, MASK, false>(a, stream);
    return hide ? launch_ring_cfg<T, NKR, false, MASK, true>(a, stream) : launch_ring_cfg<T, NKR, false, MASK, false>(a, stream);
}

template <class T, int NKR>
static hipError_t launch_ring_r(const BwdArgs &a, hipStream_t stream) {
    if (a.cosine.ptr) {
        const bool hide = a.Lk % 64 != 0;
        if (a.mask.type == kMatrixMask)
            return hide ? launch_ring_cfg<T, NKR, true, kMatrixMask, true, true>(a, stream) : launch_ring_cfg<T, NKR, true, kMatrixMask, false, true>(a, stream);
        return hide ? launch_ring_cfg<T, NKR, true, kNoMask, true, true>(a, stream) : launch_ring_cfg<T, NKR, true, kNoMask, false, true>(a, stream);
    }
    switch (a.mask.type) {
    // (a negative scale is not folded: it would turn the -inf of the keys past the end round)
    case kNoMask: return launch_ring_m<T, NKR, kNoMask>(a, (a.r == 0 && a.scale > 0.f) || a.scale == 1.f, stream);
    case kVectorMask: return launch_ring_m<T, NKR, kVectorMask>(a, false, stream);
    default: return launch_ring_m<T, NKR, kMatrixMask>(a, a.scale == 1.f, stream);
    }
}

// Compiled once per element type for head dim 32 (see Makefile).  When fb_bwd takes this path is decided by
// ring_backward() in fb_kernels.h.
#define FB_CAT2(a, b) a##b
#define FB_CAT(a, b) FB_CAT2(a, b)
hipError_t FB_CAT(launch_bwd_ring_, FB_SUFFIX)(const BwdArgs &a, hipStream_t stream) {
    return a.r == 0 ? launch_ring_r<FB_T, 0>(a, stream) : launch_ring_r<FB_T, 1>(a, stream);
}

} // namespace fb
