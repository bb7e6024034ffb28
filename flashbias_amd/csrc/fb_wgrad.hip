// Weight and bias gradient of a projection y = x w^T + b over very many tokens:
//
//   dw (n x k) = dy^T x,   db (n) = column sums of dy,      dy (tokens x n), x (tokens x k), 16-bit, row-major
//
// the products around the attention core of a window block (2_Vision_Transformer/swin_transformer_v2.py:155-207: qkv and
// proj over all tokens of all windows).  The output is small (512 x 1536) and the contraction long (262144 tokens), so
// the tokens are what has to be split: one workgroup takes a 256 x 256 (or smaller) tile of dw and one contiguous share of the
// tokens, `splits` shares fill the compute units, and a second small kernel adds the shares' fp32 tiles in a fixed order
// and rounds once.
//
// Bound: matrix pipe (two bytes in per 256 flops of a 256 x 256 tile).  Both operands are contracted over their rows, so
// both are read column-wise from row-major LDS tiles (ds_read_b64_tr_b16, four tokens of a column per lane; the XOR-swizzled
// chunks of fb_device.h, no bank conflicts), 32 tokens a stage, four stages filled by direct copies.  Four waves, each 128 x 128
// outputs in 256 accumulator registers: 16 KB of LDS reads per 64 products a workgroup, half of what LDS can deliver in
// that time; eight waves of 128 x 64 would need three quarters of it.  One wave per SIMD has nobody to hide behind, so the fragments of the next
// 16 tokens are requested between the products of the current 16, across stages: a stage's barrier sits between its two
// steps.  The workgroups of a share lie on one XCD and meet in its L2.
#include "fb_kernels.h"
#include "fb_lean_tiles.h"

namespace fb {

struct WgradArgs {
    const uint16_t *dy, *x;
    int64_t ldy, ldx; // elements between rows
    void *dw, *db;    // (n, k), (n) contiguous; db null: not wanted
    float *partial;   // (splits, n, k), then (splits, ktiles, n) where db is wanted
    int64_t tokens;
    int n, k;
    int ntiles, ktiles, splits;
};

// TN, TK: 32-channel blocks per wave (2 x 2 waves) along n and k.
template <class T_, int TN_, int TK_>
struct WgradCfg {
    typedef T_ T;
    static constexpr int TN = TN_, TK = TK_;
    static constexpr int BN = 64 * TN, BK = 64 * TK, BT = 32; // output tile, tokens per stage
    static constexpr int NWAVES = 4, NTHREADS = 256, NSTAGE = 4;
    static constexpr int CHN = BN / 8, CHK = BK / 8; // 16-byte chunks of a stage's rows
    static constexpr int SN = BT * BN * 2, STAGE = SN + BT * BK * 2; // bytes
    static constexpr int LDS_BYTES = NSTAGE * STAGE;
    static constexpr int WAVES_EU = TN * TK <= 4 ? 2 : 1;
    static constexpr int NINST = BT * (CHN + CHK) / 64 / NWAVES; // copy instructions per wave and stage
};

// One wave's copies of one operand's stages: 32 rows of CH swizzled chunks, 64 chunks an instruction.  Columns past the end
// re-read the row's last chunk, rows past the end the last row: the first only reach outputs that are not stored, the second
// are overwritten with zeros (clear_past_end).
template <int CH>
struct WgradCopy {
    static constexpr int NI = 32 * CH / 64 / 4;
    uint32_t off[NI];
    const uint8_t *p; // first row of the stage to copy (wave-uniform)
    int64_t step;
    __device__ __forceinline__ void init(const uint16_t *base, int64_t ld, int ncols, int wave, int lane) {
        p = reinterpret_cast<const uint8_t *>(base);
        step = 64 * ld;
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int at = (wave * NI + j) * 64 + lane, r = at / CH, chunk = (at % CH) ^ swz_of<CH>(r);
            off[j] = (uint32_t)r * (uint32_t)(2 * ld) + 2 * min(8 * chunk, ncols - 8);
        }
    }
    __device__ __forceinline__ void issue(int j, uint32_t lds, int wave) { lds_dma16_all(off[j], p, lds + (wave * NI + j) * 1024); }
    __device__ __forceinline__ void last_rows(int rows, int wave, int lane) { // from here on stages have that many rows
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int r = ((wave * NI + j) * 64 + lane) / CH;
            off[j] -= (uint32_t)max(r - (rows - 1), 0) * (uint32_t)(step / 32);
        }
    }
};

// The column-wise fragments of one operand for 16 tokens: block j holds columns [32 j, 32 j + 32) of the wave's part.
// A block's address differs from block 0's in bits that no other term touches (XOR), so two registers serve all.
template <int CH, int NB>
struct WgradFrag {
    uint32_t lo, hi; // byte address of this lane's first four and last four tokens of a step, block 0, stage 0
    uint32_t alo[NB], ahi[NB]; // those of a stage
    __device__ __forceinline__ void init(uint32_t tile, int col0, int c, int g) {
        const int r = 4 * g + ((c & 15) >> 2), chunk = (col0 >> 3) + 2 * (c >> 4) + ((c & 3) >> 1);
        lo = tile + 2 * swz_off<CH>(r, chunk) + 8 * (c & 1);
        hi = tile + 2 * swz_off<CH>(r + 8, chunk) + 8 * (c & 1);
    }
    __device__ __forceinline__ void stage(uint32_t off) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            alo[j] = (lo + off) ^ (uint32_t)(64 * j);
            ahi[j] = (hi + off) ^ (uint32_t)(64 * j);
        }
    }
    template <int STEP>
    __device__ __forceinline__ u32x4_t load(int j) const { return lds_load_tr(alo[j] + STEP * (16 * CH * 16), ahi[j] + STEP * (16 * CH * 16)); }
};

template <class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::WAVES_EU, C::WAVES_EU))) void wgrad_kernel(const WgradArgs a) {
    typedef typename C::T T;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave >> 1, wk = wave & 1;

    const int tiles = a.ntiles * a.ktiles;
    const int work = xcd_remap(blockIdx.x, tiles * a.splits);
    const int split = work / tiles, tile = work % tiles, tn = tile / a.ktiles, tk = tile % a.ktiles;
    const int n0 = tn * C::BN, k0 = tk * C::BK;
    // this share's tokens, in stages of BT (at least one)
    const int64_t steps_all = (a.tokens + C::BT - 1) / C::BT;
    const int64_t s0 = steps_all * split / a.splits, s1 = steps_all * (split + 1) / a.splits;
    const int nst = (int)(s1 - s0);
    const int left = (int)(min(s1 * C::BT, a.tokens) - (s1 - 1) * C::BT); // tokens of the last stage

    WgradCopy<C::CHN> copy_n;
    WgradCopy<C::CHK> copy_k;
    copy_n.init(a.dy + s0 * C::BT * a.ldy + n0, a.ldy, min(C::BN, a.n - n0), wave, lane);
    copy_k.init(a.x + s0 * C::BT * a.ldx + k0, a.ldx, min(C::BK, a.k - k0), wave, lane);
    const uint32_t lds = lds_addr_of(smem);
    // Copies run NSTAGE stages ahead; past the last stage they repeat it, into places that nobody reads any more, so that
    // every stage issues and waits for the same number of them.
    int issued = 0;
    auto to_next = [&]() { // the copies' next stage
        const bool more = issued + 1 < nst;
        copy_n.p += more ? copy_n.step : 0;
        copy_k.p += more ? copy_k.step : 0;
        if (more && issued + 2 == nst && left < C::BT) {
            copy_n.last_rows(left, wave, lane);
            copy_k.last_rows(left, wave, lane);
        }
        ++issued;
    };
    auto issue = [&](int q, uint32_t at) { // copy q of the NINST of a stage
        if (q < C::CHN / 8)
            copy_n.issue(q, at, wave);
        else
            copy_k.issue(q - C::CHN / 8, at + C::SN, wave);
    };
    // After the barrier that publishes the last stage: zeros in its rows past the end.
    auto clear_past_end = [&]() {
        u32x4_t *z = reinterpret_cast<u32x4_t *>(smem + (uint32_t)((nst - 1) & (C::NSTAGE - 1)) * C::STAGE);
        for (int i = left * C::CHN + tid; i < C::BT * C::CHN; i += C::NTHREADS) z[i] = u32x4_t{0u, 0u, 0u, 0u};
        for (int i = left * C::CHK + tid; i < C::BT * C::CHK; i += C::NTHREADS) z[C::SN / 16 + i] = u32x4_t{0u, 0u, 0u, 0u};
        barrier_lds();
    };

    f32x16_t acc[C::TN][C::TK];
#pragma unroll
    for (int i = 0; i < C::TN; ++i)
#pragma unroll
        for (int j = 0; j < C::TK; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    WgradFrag<C::CHN, C::TN> at_n;
    WgradFrag<C::CHK, C::TK> at_k;
    at_n.init(lds, wn * 32 * C::TN, c, g);
    at_k.init(lds + C::SN, wk * 32 * C::TK, c, g);

    // The products of one step; between them, pinned there, the requests for the next step's fragments (in the first half,
    // so that the last ones are back when that step begins) and copies [q0, q0 + NINST / 2) of a stage (all at once they
    // would hold up the wave's products until the memory pipeline has taken them).
    auto step = [&](const u32x4_t (&fn)[C::TN], const u32x4_t (&fk)[C::TK], auto &&request, int q0, uint32_t at) {
        constexpr int NP = C::TN * C::TK, NR = C::TN + C::TK, NQ = C::NINST / 2;
#pragma unroll
        for (int m = 0; m < NP; ++m) {
            acc[m / C::TK][m % C::TK] = T::mfma(fn[m / C::TK], fk[m % C::TK], acc[m / C::TK][m % C::TK]);
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (r * (NP / 2) / NR == m) request(r);
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                if (q * NP / NQ == m) issue(q0 + q, at);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Column sums of dy: every k tile takes the stages whose number is its own modulo their count, its two wave columns half
    // of the fragments each, two tokens an instruction (tokens 262144, 512 x 512: 163 us with all
    // fragments converted and added by one wave at a time, 153 now; products with a column of ones cost the accumulators
    // their place in the register file: 169).
    constexpr int HB = C::TN / 2;
    float bsum[HB];
#pragma unroll
    for (int m = 0; m < HB; ++m) bsum[m] = 0.f;
    auto column_sums = [&](const u32x4_t (&fn)[C::TN]) {
#pragma unroll
        for (int m = 0; m < HB; ++m) {
            const u32x4_t f = wk ? fn[HB + m] : fn[m];
#pragma unroll
            for (int e = 0; e < 4; ++e) bsum[m] = T::add2(f[e], bsum[m]);
        }
    };
    int turn = a.db ? a.ktiles - 1 - tk : -1; // its next stage is when this is ktiles - 1

    u32x4_t fn0[C::TN], fk0[C::TK], fn1[C::TN], fk1[C::TK];
    if (nst == 1 && left < C::BT) {
        copy_n.last_rows(left, wave, lane);
        copy_k.last_rows(left, wave, lane);
    }
#pragma unroll
    for (int s = 0; s < C::NSTAGE; ++s) {
        const int n = s < C::NSTAGE - 1 ? C::NINST : C::NINST / 2; // (the last one's second half: in the loop)
#pragma unroll
        for (int q = 0; q < n; ++q) issue(q, lds + s * C::STAGE);
        if (s < C::NSTAGE - 1) to_next();
    }
    wait_vmcnt<2 * C::NINST + C::NINST / 2>();
    barrier_lds();
    if (nst == 1 && left < C::BT) clear_past_end();
    at_n.stage(0);
    at_k.stage(0);
#pragma unroll
    for (int r = 0; r < C::TN + C::TK; ++r) {
        if (r < C::TN) fn0[r] = at_n.template load<0>(r);
        else fk0[r - C::TN] = at_k.template load<0>(r - C::TN);
    }
    for (int st = 0; st < nst; ++st) {
        const uint32_t cur = lds + (uint32_t)(st & (C::NSTAGE - 1)) * C::STAGE, nxt = (uint32_t)((st + 1) & (C::NSTAGE - 1)) * C::STAGE;
        const uint32_t prev = lds + (uint32_t)((st + 3) & (C::NSTAGE - 1)) * C::STAGE;
        step(fn0, fk0, [&](int r) {
            if (r < C::TN) fn1[r] = at_n.template load<1>(r);
            else fk1[r - C::TN] = at_k.template load<1>(r - C::TN);
        }, C::NINST / 2, prev);
        to_next();
        const bool sum = turn == a.ktiles - 1;
        if (a.db) turn = sum ? 0 : turn + 1;
        if (sum) column_sums(fn0);
        // the next stage has landed for every wave (the copies of two later ones may be in flight), and every wave has this
        // stage's last fragments in registers: its place is free
        wait_vmcnt<2 * C::NINST>();
        barrier_lds();
        if (st + 2 == nst && left < C::BT) clear_past_end();
        at_n.stage(nxt); // (after the last stage: fragments that nobody uses)
        at_k.stage(nxt);
        step(fn1, fk1, [&](int r) {
            if (r < C::TN) fn0[r] = at_n.template load<0>(r);
            else fk0[r - C::TN] = at_k.template load<0>(r - C::TN);
        }, 0, cur);
        if (sum) column_sums(fn1);
    }
    wait_vmcnt<0>(); // (no copy may land after the workgroup has ended)

    // lane = column k, register = row n
    float *out = a.partial + (int64_t)split * a.n * a.k;
#pragma unroll
    for (int i = 0; i < C::TN; ++i)
#pragma unroll
        for (int j = 0; j < C::TK; ++j) {
            const int kk = k0 + (wk * C::TK + j) * 32 + c;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int nn = n0 + (wn * C::TN + i) * 32 + 8 * (v >> 2) + 4 * g + (v & 3);
                if (nn < a.n && kk < a.k) out[(int64_t)nn * a.k + kk] = acc[i][j][v];
            }
        }
    if (a.db) {
        float *sums = a.partial + (int64_t)a.splits * a.n * a.k + ((int64_t)split * a.ktiles + tk) * a.n;
#pragma unroll
        for (int m = 0; m < HB; ++m) {
            const float s = bsum[m] + __shfl_xor(bsum[m], 32, 64);
            const int nn = n0 + (wn * C::TN + wk * HB + m) * 32 + c;
            if (g == 0 && nn < a.n) sums[nn] = s;
        }
    }
}

// dw and db from the shares' partial sums, added in order.  One thread per four elements of dw (k is a multiple of 8), then
// one per element of db.
template <class T>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const WgradArgs a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, nk = (int64_t)a.n * a.k, quads = nk / 4;
    if (i < quads) {
        f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int p = 0; p < a.splits; ++p) {
            const f32x4_t x = *reinterpret_cast<const f32x4_t *>(a.partial + p * nk + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += x[e];
        }
        *reinterpret_cast<u32x2_t *>(static_cast<uint16_t *>(a.dw) + 4 * i) = u32x2_t{T::pack2(s[0], s[1]), T::pack2(s[2], s[3])};
    } else if (a.db && i - quads < a.n) {
        const float *x = a.partial + a.splits * nk + (i - quads);
        float s = 0.f;
        const int rows = a.splits * a.ktiles;
#pragma unroll 8
        for (int p = 0; p < rows; ++p) s += x[(int64_t)p * a.n];
        static_cast<uint16_t *>(a.db)[i - quads] = T::from_float(s);
    }
}

// Tile: 256 wide where that wastes less than an eighth of the products, else 128.
static int wgrad_tile(int n) { return n > 128 && ((n + 255) / 256 * 256 - n) * 8 <= n ? 256 : 128; }

static void wgrad_plan(WgradArgs &a) {
    const int bn = wgrad_tile(a.n), bk = wgrad_tile(a.k);
    a.ntiles = (a.n + bn - 1) / bn;
    a.ktiles = (a.k + bk - 1) / bk;
    const int per_cu = bn == 128 && bk == 128 ? 2 : 1; // workgroups of a compute unit
    const int64_t stages = (a.tokens + 31) / 32, tiles = (int64_t)a.ntiles * a.ktiles;
    int64_t s = per_cu * (int64_t)num_cus() / tiles;
    if (s > stages / 8) s = stages / 8; // (a share of eight stages at least: the pipeline is four deep)
    a.splits = s < 1 ? 1 : (int)s;
}

size_t wgrad_workspace(int64_t tokens, int n, int k, bool bias) {
    WgradArgs a;
    a.tokens = tokens;
    a.n = n;
    a.k = k;
    wgrad_plan(a);
    return ((size_t)a.splits * n * k + (bias ? (size_t)a.splits * a.ktiles * n : 0)) * sizeof(float);
}

// Where this is ahead of the vendor library's product of the same shape (bf16, no bias, this / library, us):
//   tokens      384 x 128    768 x 256     512 x 512   1536 x 512   1024 x 1024  1600 x 1600  2048 x 2048  3200 x 3200
//     4096      10.5 / 35    23 / 30       25 / 29     29 / 31      35 / 33      44 / 48      52 / 49      110 / 103
//     6000      12.7 / 51    26 / 45       27 / 44     34 / 46      38 / 47      51 / 73      63 / 75      144 / 142
//     8192      13.2 / 59    25 / 50       26 / 54     35 / 54      40 / 55      60 / 81      75 / 83      186 / 172
//    16384      19 / 114     27 / 90       32 / 100    44 / 101     52 / 103     98 / 146     124 / 158    362 / 478
//    32768      21 / 128     36 / 166      38 / 152    64 / 196     77 / 198     183 / 328    233 / 303    710 / 877
//   262144      63 / 529     143 / 717     153 / 839   393 / 1102
// (flashbias_amd/modules.py asks for the 6000 tokens before anything else.)
// A bias gradient costs it 1-10 %; as a sum of its own it is another pass over dy (18 us at 4096 tokens, 75 at 262144 x 512).
bool wgrad_recommended(int64_t tokens, int n, int k) {
    const int64_t nk = (int64_t)n * k;
    return (tokens >= 6000 && nk <= 1 << 22) || (tokens >= 16384 && nk <= 3200 * 3200);
}

template <class T, int TN, int TK>
static hipError_t launch_wgrad_t(const WgradArgs &a, hipStream_t stream) {
    typedef WgradCfg<T, TN, TK> C;
    auto kern = wgrad_kernel<C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    return launch_flat(kern, (int64_t)a.ntiles * a.ktiles * a.splits, C::NTHREADS, C::LDS_BYTES, stream, a);
}

template <class T>
static hipError_t launch_wgrad_any(const WgradArgs &a, hipStream_t stream) {
    const bool wide_n = wgrad_tile(a.n) == 256, wide_k = wgrad_tile(a.k) == 256;
    const hipError_t e = wide_n ? (wide_k ? launch_wgrad_t<T, 4, 4>(a, stream) : launch_wgrad_t<T, 4, 2>(a, stream))
                                : (wide_k ? launch_wgrad_t<T, 2, 4>(a, stream) : launch_wgrad_t<T, 2, 2>(a, stream));
    if (e != hipSuccess) return e;
    const int64_t threads = (int64_t)a.n * a.k / 4 + (a.db ? a.n : 0);
    return launch_flat(wgrad_reduce_kernel<T>, (threads + 255) / 256, 256, 0, stream, a);
}

hipError_t launch_wgrad(const void *dy, int64_t ldy, const void *x, int64_t ldx, void *dw, void *db, float *partial, int64_t tokens,
                        int n, int k, bool bf16, hipStream_t stream) {
    WgradArgs a;
    a.dy = static_cast<const uint16_t *>(dy);
    a.x = static_cast<const uint16_t *>(x);
    a.ldy = ldy;
    a.ldx = ldx;
    a.dw = dw;
    a.db = db;
    a.partial = partial;
    a.tokens = tokens;
    a.n = n;
    a.k = k;
    wgrad_plan(a);
    return bf16 ? launch_wgrad_any<BF16>(a, stream) : launch_wgrad_any<F16>(a, stream);
}

} // namespace fb
