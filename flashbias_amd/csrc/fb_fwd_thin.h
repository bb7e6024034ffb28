// Forward for head dim 32 with one query block a wave and four waves a SIMD: aligned tensors, ranks up to 32, no mask or a
// vector mask.  Included by fb_fwd.hip after the general kernel, whose arithmetic it shares (one query per lane, S^T =
// [K | K_b] [Q | Q_b]^T, online softmax over groups of 64 keys against a lagging reference point, O^T += V^T P^T, P from
// registers).
//
// What bounds it is the vector unit: 95 instructions a 32 x 32 block and wave, 16 of them exponentials, about 510 issue cycles
// with what the products take of the port, against 160 to 256 cycles of matrix work.  The general kernel needs 182 to 252
// registers (its loader holds the next tile of K, K_b and V in about 40, two query blocks a wave share their fragments)
// and leaves two or three waves a SIMD, which wait for LDS, for their own chains and, where a workgroup walks a few key
// tiles, for its first tile at the same time: 1200 cycles a block at 384 keys and rank 32.  Here global_load_lds copies tiles
// of 64 keys row-major into two stages, one tile ahead, V^T fragments come from transposing LDS reads, and no register
// holds a tile or a fragment that is not in use: 97 to 127 of them, four workgroups a compute unit.
//
// General kernel against this one, us, bf16: rank 32, 384 x 4 rows of 384 with a padding mask 101 -> 78, 301 x 4 of 301 80 -> 53,
// 512 x 4 of 512 163 -> 159, 768 x 4 of 768 528 -> 508 (masked 570 -> 551); rank 16, causal B1 H50 L=4096 137 -> 121, L=8192
// 460 -> 424, B4 H16 L=1500 46 -> 42, B8 H32 L=4096 1008 -> 985, B2 H4 L=16384 equal; rank 8 with a padding mask, B2 H4 L=8192
// 167 -> 155; 128 x 4 rows of 128 and B2 H4 L=777 equal.  Not kept: five waves a SIMD (512 x 16 windows of 128 at rank 32 88
// -> 95), three waves and all fragments of a tile ahead (rank 32 padded 80, masked 768 586), turns by tile (rank 8 masked 156 ->
// 168), priority for the products (no gain), scores and bias in one chain (2 % at rank 32, but the bias product then starts from
// q k^T instead of zero: closed-form factors in the thousands lose its low bits, dq_bias of the ALiBi workload 0.067 for 0.01).
//
// SPLIT: on small grids a second group of four waves takes the second half of the keys for the same queries, in stages of its own, and hands
// its sums over in LDS.  One group alone has one wave a SIMD there, which waits for itself: 1150 cycles a block where four waves take 500
// (B1 H16 L=1500, causal: 192 workgroups 24.3 -> 19.5 us; dispatch and figures at thin_split).
#pragma once
#include "fb_lean_tiles.h"

namespace fb {

template <class T, int NKR_, int MASK_, bool FOLD_, int SPLIT_>
struct FwdThinCfg {
    static constexpr int NKD = 2, NKR = NKR_, NK = NKD + NKR_;
    static constexpr bool VMASK = MASK_ == kVectorMask, FOLD = FOLD_;
    static_assert(MASK_ != kMatrixMask && NKR_ <= 2 && !(FOLD_ && VMASK), "");
    static constexpr int SPLIT = SPLIT_, NWAVES = 4, NTHREADS = 64 * NWAVES * SPLIT, BM = 32 * NWAVES; // (NWAVES: of a group)
    static constexpr int KBLK = 2, BN = 32 * KBLK;
    static constexpr int CPR = NKR == 2 ? 4 : 2; // 16-byte chunks per row of K_b
    static constexpr int K = 0, V = K + BN * 64, KB = V + BN * 64, MK = KB + (NKR ? BN * CPR * 16 : 0), STAGE = MK + (VMASK ? BN * 4 : 0);
    static constexpr int LDS_BYTES = 2 * STAGE * SPLIT;
    static constexpr int WAVES_EU = 4;
    static_assert(WAVES_EU * LDS_BYTES / SPLIT <= 160 * 1024 && (SPLIT == 1 || LDS_BYTES >= 4 * 4608), "");
    static __device__ __forceinline__ bool low_parts(const FwdArgs &a) { return FOLD_ && NKR_ == 1 && a.r <= 8 && a.scale != 1.f; }
};

template <class T, class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void fwd_thin_kernel(const FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int grp = C::SPLIT == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8); // takes its share of the tiles of keys, in stages of its own
    uint8_t *const stages = smem + grp * 2 * C::STAGE;
    const uint32_t lds0 = lds_addr_of(stages);
    const int tid = threadIdx.x & (64 * C::NWAVES - 1), lane = tid & 63, c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    const int total = a.ntiles_m * a.B * a.H;
    int bh, tile_m;
    work_order(blockIdx.x, a.ntiles_m, total, a.causal, bh, tile_m);
    if (a.causal) tile_m = a.ntiles_m - 1 - tile_m; // the last query tile sees the most keys
    const int b = bh / a.H, h = bh % a.H;
    const int m0 = tile_m * C::BM, wq0 = m0 + wave * 32;
    const int query = wq0 + c;

    int k_end = a.Lk; // causal: keys past the last query of this workgroup are never visible
    if (a.causal && m0 + C::BM < k_end) k_end = m0 + C::BM;
    const int ntiles = (k_end + C::BN - 1) / C::BN;
    const int walk = (ntiles + C::SPLIT - 1) / C::SPLIT, tile0 = grp * walk; // this group's tiles: from tile0 on, `walk` of them if there are so many
    const uint8_t *kptr = reinterpret_cast<const uint8_t *>(a.k.ptr + b * a.k.sb + h * a.k.sh);
    const uint8_t *vptr = reinterpret_cast<const uint8_t *>(a.v.ptr + b * a.v.sb + h * a.v.sh);
    LeanCopy4<C::BN> kd, vd;
    kd.init(wave, lane, a.k.ss);
    vd.init(wave, lane, a.v.ss);
    DenseCopy<C::BN, C::CPR> kbd;
    if constexpr (C::NKR > 0) {
        kbd.init(a.kb.ptr + b * a.kb.sb + h * a.kb.sh, a.kb.ss, a.r, C::low_parts(a), wave, lane, tile0 * C::BN);
        if (a.r < 16 * C::NKR && !C::low_parts(a)) { // (the channel padding of the rank is never written)
            for (int i = threadIdx.x; i < C::LDS_BYTES / 16; i += C::NTHREADS) reinterpret_cast<u32x4_t *>(smem)[i] = u32x4_t{0u, 0u, 0u, 0u};
            __syncthreads();
        }
    }
    auto issue = [&](int buf, int n0) {
        const uint32_t base = lds0 + buf * C::STAGE;
        kd.issue(kptr + (int64_t)n0 * kd.pitch, base + C::K, wave, lane, a.Lk - n0);
        if constexpr (C::NKR > 0) kbd.issue(base + C::KB, n0, a.Lk);
        vd.template issue<true>(vptr + (int64_t)n0 * vd.pitch, base + C::V, wave, lane, a.Lk - n0);
    };
    // Vector mask: thread `tid` carries the value of key n0 + tid of the tile that follows.
    float mkey = 0.f;
    auto load_vmask = [&](int n0) {
        const int key = min(n0 + (tid & (C::BN - 1)), a.Lk - 1); // (past the end: the score is set to -inf below)
        const uint8_t *mbase = reinterpret_cast<const uint8_t *>(a.mask.ptr) + mask_offset(a.mask, b, h) * (a.mask.is_f32 ? 4 : 2);
        mkey = a.mask.is_f32 ? reinterpret_cast<const float *>(mbase)[key] : T::to_float(reinterpret_cast<const uint16_t *>(mbase)[key]);
    };
    auto store_vmask = [&](int buf) {
        if (tid < C::BN) *reinterpret_cast<float *>(stages + buf * C::STAGE + C::MK + 4 * tid) = mkey;
    };
    if (C::SPLIT == 1 || tile0 < ntiles) {
        issue(0, tile0 * C::BN);
        if constexpr (C::VMASK) load_vmask(tile0 * C::BN);
    }

    u32x4_t qr[C::NK];
    const uint16_t *qbase = a.q.ptr + b * a.q.sb + h * a.q.sh;
#pragma unroll
    for (int t = 0; t < C::NKD; ++t) qr[t] = load_chunk<true>(qbase, a.q.ss, query, a.Lq, 16 * t + 8 * g, a.d);
    if constexpr (C::NKR > 0) {
        const uint16_t *qbbase = a.qb.ptr + b * a.qb.sb + h * a.qb.sh;
        const bool low = C::low_parts(a) && g == 1;
#pragma unroll
        for (int t = 0; t < C::NKR; ++t) {
            u32x4_t x = load_chunk<true>(qbbase, a.qb.ss, query, a.Lq, low ? 0 : 16 * t + 8 * g, a.r);
            if (C::FOLD && a.scale != 1.f) x = fold_scale_chunk<T>(x, 1.f / a.scale, C::low_parts(a), low);
            qr[C::NKD + t] = x;
        }
    }
    f32x16_t o;
#pragma unroll
    for (int v = 0; v < 16; ++v) o[v] = 0.f;
    float m_ref = -INFINITY, m2 = 0.f, l_run = 0.f; // (as in fwd_body)
    const float to_log2 = C::FOLD ? a.scale * kLog2e : kLog2e, lag = 8.0f / to_log2;

    // this lane's read addresses inside a stage (stage, key block and step are added)
    const uint32_t row_off[2] = {lds0 + C::K + lean_row_addr<4>(c, g), lds0 + C::K + lean_row_addr<4>(c, 2 + g)};
    const uint32_t col_off[2] = {lds0 + C::V + lean_tr_addr4(c, g, 0), lds0 + C::V + lean_tr_addr4(c, g, 1)};
    uint32_t kb_off[C::NKR > 0 ? C::NKR : 1];
#pragma unroll
    for (int t = 0; t < C::NKR; ++t) kb_off[t] = lds0 + C::KB + lean_row_addr<C::CPR>(c, 2 * t + g);

    if constexpr (C::VMASK) store_vmask(0);
    wait_vmcnt<0>();
    barrier_lds();

#pragma unroll 1
    for (int it = 0; it < walk; ++it) {
        const int cur = it & 1, tile = tile0 + it, n0 = tile * C::BN;
        const bool more = it + 1 < walk && tile + 1 < ntiles;
        if (more) {
            issue(cur ^ 1, n0 + C::BN);
            if constexpr (C::VMASK) load_vmask(n0 + C::BN);
        }
        const uint32_t at = cur * C::STAGE;
        // (a tile hidden from every query of this wave: so are all later ones, but the copies and barriers go on)
        if (!(a.causal && n0 > wq0 + 31) && wq0 < a.Lq && (C::SPLIT == 1 || tile < ntiles)) {
            f32x16_t s[C::KBLK];
            if (!a.causal) __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int kb = 0; kb < C::KBLK; ++kb) {
                // q k^T and q_b k_b^T: two chains joined by the FMA that applies the softmax scale to the first (:246-256),
                // an additive mask the initial value of the second; folded, one chain
                f32x16_t acc, accb;
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[v] = accb[v] = 0.f;
                if constexpr (C::VMASK) {
                    const float *sM = reinterpret_cast<const float *>(stages + at + C::MK) + kb * 32 + 4 * g;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const f32x4_t x = *reinterpret_cast<const f32x4_t *>(sM + 8 * j);
#pragma unroll
                        for (int e = 0; e < 4; ++e) accb[4 * j + e] = x[e];
                    }
                }
#pragma unroll
                for (int t = 0; t < C::NKD; ++t) acc = T::mfma(lds_load16(row_off[t] + at + kb * 2048), qr[t], acc);
#pragma unroll
                for (int t = 0; t < C::NKR; ++t) {
                    const u32x4_t kf = lds_load16(kb_off[t] + at + kb * (32 * C::CPR * 16));
                    if constexpr (C::FOLD)
                        acc = T::mfma(kf, qr[C::NKD + t], acc);
                    else
                        accb = T::mfma(kf, qr[C::NKD + t], accb);
                }
                if constexpr (!C::FOLD) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[v] = (C::NKR > 0 || C::VMASK) ? __builtin_fmaf(acc[v], a.scale, accb[v]) : acc[v] * a.scale;
                }
                s[kb] = acc;
                // (the second block's fragments are not requested ahead of the first block's scores: at rank 32 that spills)
                if constexpr (C::NKR == 2) __builtin_amdgcn_sched_barrier(0);
            }
            // (bitwise on purpose, as in the dq kernel: no scalar block between the last MFMA and the branch)
            const bool edge = (n0 + C::BN > a.Lk) | ((a.causal != 0) & (n0 + C::BN - 1 > wq0));
            if (edge) {
                // (without a mask one comparison a score.  With two, us, rank 16: causal B1 H64 L=256 8.6 for 8.0, L=512 12.2 for 11.6, B1 H8
                // L=1024 17.75 for 17.3; the general kernel 8.1, 12.0, 17.7.  With a mask a last key in a register makes the compiler
                // order the loop so that B1 H12 L=2500 takes 55 for 51.6.)
                int key0 = n0 + 4 * g, last = a.causal ? min(query, a.Lk - 1) : a.Lk - 1;
                if constexpr (C::VMASK)
                    asm volatile("" : "+v"(key0)); // (computed here, not kept in registers across the loop)
                else
                    asm volatile("" : "+v"(key0), "+v"(last));
#pragma unroll
                for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int key = key0 + kb * 32 + 8 * (v >> 2) + (v & 3);
                        if (C::VMASK ? key >= a.Lk || (a.causal && key > query) : key > last) s[kb][v] = -INFINITY;
                    }
            }
            // (exponentials before another workgroup's products, which evens out who gets ahead: B2 H4 L=16384 r16 513 -> 475 us;
            // under a causal mask the long workgroups of the launch's end lose by it, B1 H50 L=4096 120 -> 129)
            if (!a.causal) __builtin_amdgcn_s_setprio(1);
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
                for (int v = 0; v < 16; ++v) o[v] *= alpha;
                m_ref = m_new;
                m2 = reference_log2<T>(m_new, to_log2);
            }
#pragma unroll
            for (int kb = 0; kb < C::KBLK; ++kb)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u32x4_t vt = lds_load_tr(col_off[0] + at + kb * 2048 + t * 1024, col_off[1] + at + kb * 2048 + t * 1024);
                    u32x4_t pb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float p0 = fast_exp2(__builtin_fmaf(s[kb][8 * t + 2 * e], to_log2, -m2));
                        const float p1 = fast_exp2(__builtin_fmaf(s[kb][8 * t + 2 * e + 1], to_log2, -m2));
                        pb[e] = T::pack2(p0, p1);
                        l_run += p0 + p1;
                    }
                    o = T::mfma(vt, pb, o);
                }
        }
        if constexpr (C::VMASK) {
            if (more) store_vmask(cur ^ 1);
        }
        wait_vmcnt<0>(); // the next tile has landed
        barrier_lds();
    }

    if constexpr (C::SPLIT == 2) { // the second group's sums to the first one's (the stages are free: the loop ends with a barrier)
        asm volatile("s_nop 11" : "+v"(o));
        uint8_t *ex = smem + wave * 4608;
        float *em = reinterpret_cast<float *>(smem + wave * 4608 + 4096) + lane;
        if (grp == 1) {
            lds_put_block(ex, o, lane);
            em[0] = m_ref;
            em[64] = l_run;
        }
        barrier_lds();
        if (grp == 1) return;
        float mine, other;
        join_references(m_ref, em[0], to_log2, mine, other);
        l_run = l_run * mine + em[64] * other;
#pragma unroll
        for (int v = 0; v < 16; ++v) o[v] *= mine;
        lds_add_block(ex, o, lane, other);
    }
    int q = query;
    asm volatile("" : "+v"(q)); // (keeps the address arithmetic below the key loop)
    const float l = l_run + __shfl_xor(l_run, 32, 64);
    const bool ok = q < a.Lq;
    if (ok && g == 0) a.lse[(int64_t)bh * a.Lq + q] = m_ref * (C::FOLD ? a.scale : 1.f) + __builtin_amdgcn_logf(l) * kLn2;
    uint16_t *orow = const_cast<uint16_t *>(a.o.ptr) + b * a.o.sb + h * a.o.sh + (int64_t)(ok ? q : 0) * a.o.ss;
    store_acc_rows<T, true>(orow, ok, true, o, 1.f / l, a.d, g);
}

template <class T, int NKR, int MASK, bool FOLD, int SPLIT>
static hipError_t launch_fwd_thin_split(const FwdArgs &a0, hipStream_t stream) {
    typedef FwdThinCfg<T, NKR, MASK, FOLD, SPLIT> C;
    FwdArgs a = a0;
    a.ntiles_m = (a.Lq + C::BM - 1) / C::BM;
    auto kern = fwd_thin_kernel<T, C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    return launch_flat(kern, (int64_t)a.ntiles_m * a.B * a.H, C::NTHREADS, C::LDS_BYTES, stream, a);
}

// Two groups of waves where four leave a compute unit with too few: up to two workgroups on each, under a causal mask, where a launch lasts
// as long as its longest workgroup, up to 2.4 if that one is long, and more than 256 keys.  us, one group / two, rank 16: 64 workgroups (B1 H8 L=1024)
// 16.8 / 13.8, 192 24.5 / 19.9, 256 57.4 / 44.9 (B2 H4 L=4096), 400 22.5 / 22.1, 512 71.4 / 70.3 (B1 H16 L=4096) and 22.3 / 22.5 (B2 H32 L=1024), 600 40.1 /
// 40.3; with a padding mask 64 19.8 / 16.5, 256 68.3 / 51.8, 512 77.9 / 74.7, 600 44.9 / 46.8; causal 64 17.3 / 14.2, 192 24.3 / 19.5, 400 19.1 / 16.9, 512
// 59.0 / 47.9 (B1 H16 L=4096) and 18.9 / 17.9 (B2 H32 L=1024), 576 20.4 / 19.2, 600 26.3 / 25.5 (B1 H50 L=1500) but 16.7 / 17.8 (B2 H50 L=700), 640 21.4 /
// 22.5, 800 39.3 / 38.9; rank 32 (one group: the general kernel up to 256) 64 18.2 / 14.9, 512 45.7 / 43.1, causal 69.7 / 52.2.
// Up to 256 keys (640 at ranks above 16) an entry keeps the bits that it has in a larger call.
inline bool thin_split(const FwdArgs &a) {
    const int64_t wgs = (int64_t)a.B * a.H * ((a.Lq + 127) / 128);
    return a.Lk > (a.r > 16 ? 640 : 256) && 10 * wgs <= (a.causal && a.Lk >= 1024 ? 24 : 20) * (int64_t)num_cus();
}

template <class T, int NKR, int MASK, bool FOLD>
static hipError_t launch_fwd_thin(const FwdArgs &a, hipStream_t stream) {
    return thin_split(a) ? launch_fwd_thin_split<T, NKR, MASK, FOLD, 2>(a, stream) : launch_fwd_thin_split<T, NKR, MASK, FOLD, 1>(a, stream);
}

} // namespace fb
