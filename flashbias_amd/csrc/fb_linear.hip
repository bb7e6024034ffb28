// A projection of many tokens by a small weight (the layers of a Swin-V2 window block, 2_Vision_Transformer/swin_transformer_v2.py:
// 155-207): y (tokens, n) = x (tokens, k) w^T + b, fp32 sums, the bias added to them, rounded once.
//
// What bounds such products is the matrix pipe (at the clock that power leaves: 1.6 PFLOP/s without copies and stores at k = 512), then
// the results (3 n bytes of y where x has k) and the way of x from memory, which the two stages of a tile cover in part.  Split: a
// workgroup is four waves, one a SIMD, and forms tiles of 64 PN channels x 64 PM tokens, a wave 32 PN x 32 PM of one (D = W X^T: a
// lane holds a token, its registers channels).  At 4 x 4 blocks a wave the LDS has 256 cycles of reads and 128 of copies for 512 of
// products; eight waves of 2 x 4 would need every cycle it has.
//   * Stages hold 64 columns, rows of 128 bytes: a copy of 64 bytes a row fetches its whole line and the other half again a
//     step later (32 columns in four stages: 262144 tokens of 512 to 1536 channels 491 us for 445).
//   * A step is four slices of 16 columns.  The reads of a slice stand between the products of the slice before, also across
//     the step's one barrier, which comes after the third slice: everyone has then read the stage, and the copies of NSTAGE steps
//     later go out beside the products of the fourth slice and of the next step's first.
//   * Workgroups stay for as many tiles as they get, and the copies run on into the next tile.  What a tile's end still has to copy
//     goes out ahead of its stores, so that the next waits, which count in order, can leave the stores in flight.
//   * Results that no cache will hold until they are read go past them (kPastCaches: 805 MB 426 -> 390 us).
// Vendor library / this, us: 262144 tokens, 512 to 1536 channels 482 / 393, 512 to 512 with bias 162 / 143, 256 to 768 161 / 111;
// 147456 tokens, 512 to 1536 366 / 215, 256 to 768 103 / 67; 36864 tokens, 256 to 768 35 / 24; 16384, 256 to 768 19.9 / 13.8.
// Not kept: a line of x touched two steps ahead of its copy (431 -> 443, the touches wait in the same queue), workgroups that
// start one after the other (no gain).
#include "fb_kernels.h"
#include "fb_lean_tiles.h"

namespace fb {

struct LinearArgs {
    const uint16_t *x, *w, *b; // b: null for none
    uint16_t *y;
    int64_t ldx;
    int n, tokens, k;
    int ntiles, ttiles; // tiles of channels, of tokens
    bool stream;        // results past the caches
};

template <class T_, int PN_, int PM_, int NSTAGE_, bool BIAS_>
struct LinearCfg {
    typedef T_ T;
    static constexpr int PN = PN_, PM = PM_, TN = 64 * PN, TM = 64 * PM, NSTAGE = NSTAGE_;
    static constexpr bool BIAS = BIAS_;
    static constexpr int NTHREADS = 256;
    static constexpr int CW = TN / 32, CX = TM / 32, NC = CW + CX; // copies of a wave and step, eight rows each
    static constexpr int SW = TN * 128, STAGE = (TN + TM) * 128;
    // after the stages 4 or 8 KB of each wave for its results
    static constexpr int OUT = NSTAGE * STAGE, NB = OUT + 4 * 8192 <= 160 * 1024 ? 2 : 1, OUTB = NB * 4096, LDS_BYTES = OUT + 4 * OUTB;
    static constexpr int NSTORE = PM * PN / 2 * 4;
    static_assert(LDS_BYTES <= 160 * 1024 && (NSTAGE - 1) * NC < 64 && (NSTAGE - 2) * NC + NSTORE < 64, "");
};

template <class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void linear_kernel(const LinearArgs a) {
    typedef typename C::T T;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = lds_addr_of(smem);
    const int lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wn = wave & 1, wm = wave >> 1;

    // An XCD's workgroups walk a contiguous share of the tiles side by side, channel tiles of the same tokens next to each other.
    const int total = a.ntiles * a.ttiles, share = (total + 7) / 8, xcd = blockIdx.x & 7;
    const int stride = gridDim.x >> 3, end = min((xcd + 1) * share, total);
    int item = xcd * share + (int)(blockIdx.x >> 3);
    if (item >= end) return;

    // ---- copies: eight rows of 128 bytes an instruction, chunks swizzled by the row; rows past the end are the last one again
    const int nsteps = a.k / 64;
    uint32_t off[C::NC];
    const uint8_t *wp, *xp;
    auto place = [&](int it) {
        const int n0 = it % a.ntiles * C::TN, m0 = it / a.ntiles * C::TM;
#pragma unroll
        for (int j = 0; j < C::NC; ++j) {
            const int row = 8 * (j < C::CW ? C::CW * wave + j : C::CX * wave + j - C::CW) + (lane >> 3), chunk = (lane & 7) ^ swz_of<8>(row);
            off[j] = j < C::CW ? (uint32_t)min(row, a.n - 1 - n0) * (uint32_t)(a.k * 2) + chunk * 16
                               : (uint32_t)min(row, a.tokens - 1 - m0) * (uint32_t)(a.ldx * 2) + chunk * 16;
        }
        wp = reinterpret_cast<const uint8_t *>(a.w) + (int64_t)n0 * a.k * 2;
        xp = reinterpret_cast<const uint8_t *>(a.x) + (int64_t)m0 * a.ldx * 2;
    };
    int citem = item, cstep = 0; // of the next copies
    place(citem);
    auto copy = [&](int j, int stage) {
        if (j < C::CW)
            lds_dma16_all(off[j], wp, lds0 + stage * C::STAGE + (C::CW * wave + j) * 1024);
        else
            lds_dma16_all(off[j], xp, lds0 + stage * C::STAGE + C::SW + (C::CX * wave + j - C::CW) * 1024);
    };
    auto advance = [&]() { // (past the last tile: its last columns again, so that every wait is for a constant number)
        if (cstep + 1 < nsteps) {
            ++cstep;
            wp += 128;
            xp += 128;
        } else if (citem + stride < end) {
            citem += stride;
            cstep = 0;
            place(citem);
        }
    };
#pragma unroll 1
    for (int s = 0; s < C::NSTAGE; ++s) {
#pragma unroll
        for (int j = 0; j < C::NC; ++j) copy(j, s);
        advance();
    }

    f32x16_t acc[C::PN][C::PM];
    u32x4_t f[2][C::PN + C::PM]; // a slice's fragments and the next one's
    uint32_t row_off[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) row_off[t] = 2 * swz_off<8>(c, 2 * t + g);
    const uint32_t wrow = lds0 + wn * (C::PN * 4096), xrow = lds0 + C::SW + wm * (C::PM * 4096);
    auto read = [&](int i, int t, int stage) {
        f[t & 1][i] = i < C::PN ? lds_load16(wrow + row_off[t] + stage * C::STAGE + i * 4096) : lds_load16(xrow + row_off[t] + stage * C::STAGE + (i - C::PN) * 4096);
    };
    wait_vmcnt<(C::NSTAGE - 1) * C::NC>();
    barrier_lds();
#pragma unroll
    for (int i = 0; i < C::PN + C::PM; ++i) read(i, 0, 0);

    // A slice: its products, beside the first ones the next slice's reads, and half of a step's copies (from `copies` on, none if negative).
    auto slice = [&](auto first, auto slice_of_step, auto copies, int read_stage, int copy_stage) {
        constexpr int t = decltype(slice_of_step)::value, NR = C::PN + C::PM, NM = C::PN * C::PM, PER = (NR + NM - 1) / NM;
        constexpr int C0 = decltype(copies)::value, NCOPY = C0 < 0 ? 0 : C::NC / 2;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int p = m / C::PM, q = m % C::PM;
            if constexpr (decltype(first)::value) {
                f32x16_t zero;
#pragma unroll
                for (int v = 0; v < 16; ++v) zero[v] = 0.f;
                acc[p][q] = T::mfma(f[t & 1][p], f[t & 1][C::PN + q], zero);
            } else {
                acc[p][q] = T::mfma(f[t & 1][p], f[t & 1][C::PN + q], acc[p][q]);
            }
#pragma unroll
            for (int i = m * PER; i < (m + 1) * PER && i < NR; ++i) read(i, (t + 1) & 3, read_stage);
#pragma unroll
            for (int j = m * NCOPY / NM; j < (m + 1) * NCOPY / NM; ++j) copy(C0 + j, copy_stage);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const std::true_type yes{};
    const std::false_type no{};
    const std::integral_constant<int, 0> s0{}, early{};
    const std::integral_constant<int, 1> s1{};
    const std::integral_constant<int, 2> s2{};
    const std::integral_constant<int, 3> s3{};
    const std::integral_constant<int, C::NC / 2> late{};
    const std::integral_constant<int, -1> none{};
    int stage = 0;
    bool stores_left = false; // the last tile's stores may be in flight, all NSTORE of them
    while (true) {
#pragma unroll 1
        for (int step = 0; step < nsteps; ++step) {
            const int prev = stage == 0 ? C::NSTAGE - 1 : stage - 1, next = stage + 1 == C::NSTAGE ? 0 : stage + 1;
            if (step == 0) {
                slice(yes, s0, none, stage, 0);
            } else { // (with the second half of the copies that the step before began)
                slice(no, s0, late, stage, prev);
                advance();
            }
            if constexpr (C::BIAS) { // this wave's channels of the bias, to where its results go next
                if (step + 1 == nsteps) {
                    int l = lane;
                    asm volatile("" : "+v"(l));
                    lds_dma4(a.b + min(item % a.ntiles * C::TN + 32 * C::PN * wn + 2 * l, a.n - 2), lds0 + C::OUT + wave * C::OUTB);
                }
            }
            slice(no, s1, none, stage, 0);
            slice(no, s2, none, stage, 0);
            // the next stage has landed: of what was asked for after it NSTAGE - 2 steps' copies may still be on their way
            constexpr int LATER = (C::NSTAGE - 2) * C::NC;
            if (C::BIAS && step + 1 == nsteps)
                wait_vmcnt<0>();
            else if (step == 0 && stores_left)
                wait_vmcnt<LATER + C::NSTORE>();
            else
                wait_vmcnt<LATER>();
            barrier_lds();
            slice(no, s3, early, next, stage);
            stage = next;
        }
#pragma unroll
        for (int j = C::NC / 2; j < C::NC; ++j) copy(j, stage == 0 ? C::NSTAGE - 1 : stage - 1);
        advance();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 11" ::: "memory"); // (wait states between the last products and their readers, which stand behind a branch)
        __builtin_amdgcn_sched_barrier(0);

        // ---- results: 64 channels x 32 tokens at a time through 4 KB of this wave's own, lines of 128 bytes, chunks XORed with the line
        const int n0 = item % a.ntiles * C::TN, m0 = item / a.ntiles * C::TM;
        const bool whole = n0 + C::TN <= a.n && m0 + C::TM <= a.tokens;
        int l = lane;
        asm volatile("" : "+v"(l)); // (formed here, not kept across the steps)
        const int lc = l & 31, lg = l >> 5;
        const int ch = n0 + 32 * C::PN * wn + 8 * (l & 7), tok = m0 + 32 * C::PM * wm + (l >> 3);
        uint16_t *out = a.y + (int64_t)tok * a.n + ch;
        uint8_t *buf = smem + C::OUT + wave * C::OUTB;
        u32x2_t bias[C::BIAS ? 4 * C::PN : 1];
        if constexpr (C::BIAS) {
#pragma unroll
            for (int i = 0; i < 4 * C::PN; ++i) bias[i] = *reinterpret_cast<const u32x2_t *>(buf + 16 * i + 8 * lg);
        }
        auto pack = [&](int r) { // channels 64 (r / PM) .. and tokens 32 (r % PM) ..
            const int p2 = r / C::PM * 2, q = r % C::PM;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                f32x16_t x = acc[p2 + p][q];
                asm volatile("" : "+v"(x)); // (read here: ahead of the branches below, all of them would be in registers twice)
                if constexpr (C::BIAS) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const uint32_t w = bias[4 * (p2 + p) + v / 4][(v % 4) / 2];
                        x[v] += T::to_float((uint16_t)(v & 1 ? w >> 16 : w & 0xffffu));
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<u32x2_t *>(buf + (r % C::NB) * 4096 + lc * 128 + (((4 * p + j) ^ (lc & 7)) << 4) + 8 * lg) =
                        u32x2_t{T::pack2(x[4 * j], x[4 * j + 1]), T::pack2(x[4 * j + 2], x[4 * j + 3])};
            }
        };
        auto store = [&](int r, auto all, auto stream) {
            const int p2 = r / C::PM * 2, q = r % C::PM;
            u32x4_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int line = 8 * i + (l >> 3);
                v[i] = *reinterpret_cast<const u32x4_t *>(buf + (r % C::NB) * 4096 + line * 128 + (((l & 7) ^ (line & 7)) << 4));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                u32x4_t *to = reinterpret_cast<u32x4_t *>(out + (int64_t)(32 * q + 8 * i) * a.n + 32 * p2);
                if constexpr (decltype(stream)::value)
                    __builtin_nontemporal_store(v[i], to);
                else if (decltype(all)::value || (tok + 32 * q + 8 * i < a.tokens && ch + 32 * p2 < a.n))
                    *to = v[i];
            }
        };
        auto results = [&](auto all, auto stream) {
            constexpr int R = C::PM * C::PN / 2;
            pack(0);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (C::NB == 2 && r + 1 < R) pack(r + 1);
                store(r, all, stream);
                if (C::NB == 1 && r + 1 < R) pack(r + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (!whole)
            results(no, no);
        else if (a.stream)
            results(yes, yes);
        else
            results(yes, no);
        stores_left = whole;
        item += stride;
        if (item >= end) break;
    }
    wait_vmcnt<0>(); // (the copies past the end)
}

template <class T, int PN, int PM, int NSTAGE, bool BIAS>
static hipError_t launch_linear_t(LinearArgs a, hipStream_t stream) {
    typedef LinearCfg<T, PN, PM, NSTAGE, BIAS> C;
    a.ntiles = (a.n + C::TN - 1) / C::TN;
    a.ttiles = (a.tokens + C::TM - 1) / C::TM;
    auto kern = linear_kernel<C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    const int64_t total = (int64_t)a.ntiles * a.ttiles, most = num_cus() / 8 * 8; // one workgroup a compute unit, the same number for every XCD
    return launch_flat(kern, total < most ? (total + 7) / 8 * 8 : most, C::NTHREADS, C::LDS_BYTES, stream, a);
}

// Microseconds of the rounds of a tile of tn channels x 256 tokens: a step of 64 columns and what a tile takes beside its steps, fitted to
// 2 and 8 steps of 262144 tokens (a tile of 256: 6.6 and 16.4; of 128: 4.0 and 9.6).
static float linear_rounds(int64_t tokens, int n, int k, int tn) {
    const int64_t tiles = ((n + tn - 1) / tn) * ((tokens + 255) / 256), rounds = (tiles + num_cus() - 1) / num_cus();
    return (float)rounds * (tn == 256 ? 1.63f * (k / 64) + 3.3f : 0.93f * (k / 64) + 2.1f);
}

// Vendor library / this, us, in a graph.  Two tiles of 128 channels a compute unit: 65536 x 64 to 192 12.7 / 10.9, 147456 x 64 to 64
// 23.5 / 14.7, 36864 x 512 to 512 35.6 / 32.2, 65536 x 256 to 256 18.1 / 17.9; one and many channels: 16384 x 192 to 576 20.5 / 12.7, 36864 x 128
// to 384 21.0 / 13.2, 9216 x 512 to 1536 21.5 / 21.1.  Fewer: 36864 x 256 to 256 13.6 / 15.1, 36864 x 192 to 192 12.0 / 12.8, 6016 x 128 to 384 6.8 / 7.2,
// 9216 x 512 to 512 12.1 / 13.1.  Long rows, where the library's way of x from memory is ahead: 65536 x 768 to 768 70 / 76, 36864 x 1024 to
// 1024 75 / 88, 262144 x 1536 to 512 338 / 382.
bool linear_recommended(int64_t tokens, int n, int k) {
    const int64_t tiles = (int64_t)((n + 127) / 128) * ((tokens + 255) / 256);
    return k <= 512 && tiles >= (n >= 2 * k ? 1 : 2) * (int64_t)num_cus();
}

template <class T>
static hipError_t launch_linear_w(const LinearArgs &a, hipStream_t stream) {
    if (linear_rounds(a.tokens, a.n, a.k, 128) < linear_rounds(a.tokens, a.n, a.k, 256))
        return a.b ? launch_linear_t<T, 2, 4, 3, true>(a, stream) : launch_linear_t<T, 2, 4, 3, false>(a, stream);
    return a.b ? launch_linear_t<T, 4, 4, 2, true>(a, stream) : launch_linear_t<T, 4, 4, 2, false>(a, stream);
}

// Bytes of results from which they are stored past the caches.  The kernel alone is ahead from 40 MB on, but the next one reads them, and up to
// about 200 MB from the memory side's 256 MB.  This and its reader, through the caches / past them, us: the window forward (256 tokens) on 70 MB of
// 256 to 768 channels 67.1 / 70.6, 100 MB 84.5 / 91.7, 130 MB 113.1 / 115.9, 180 MB 151.4 / 156.4, 250 MB 215.0 / 208.2, 400 MB 332.7 / 325.6, 800 MB of 512
// to 1536 805 / 786; windows of 64, 128 to 384, 180 MB 128.4 / 133.6, 250 MB 181.4 / 176.4; an addition on 100 MB of 512 to 512 102.3 / 105.5, 180 MB
// 195.2 / 194.0, 250 MB 267.3 / 261.7.
constexpr int64_t kPastCaches = (int64_t)200 << 20;

hipError_t launch_linear(const void *x, int64_t ldx, const void *w, const void *b, void *y, int64_t tokens, int n, int k, bool bf16, hipStream_t stream) {
    LinearArgs a = {};
    a.x = static_cast<const uint16_t *>(x);
    a.w = static_cast<const uint16_t *>(w);
    a.b = static_cast<const uint16_t *>(b);
    a.y = static_cast<uint16_t *>(y);
    a.ldx = ldx;
    a.n = n;
    a.tokens = (int)tokens;
    a.k = k;
    a.stream = tokens * n * 2 >= kPastCaches;
    return bf16 ? launch_linear_w<BF16>(a, stream) : launch_linear_w<F16>(a, stream);
}

// out (cols, rows) = in (rows, cols)^T of 16-bit elements, both multiples of 64: a tile of 64 x 64 a workgroup through LDS, 16 bytes a lane on both
// sides.  A weight before the product that contracts its rows (an input's gradient); 512 x 512 takes 3 us, launch included.
__global__ __launch_bounds__(256) void transpose_kernel(const uint16_t *in, uint16_t *out, int rows, int cols) {
    __shared__ uint16_t tile[64][66];
    const int r0 = blockIdx.x / (cols / 64) * 64, c0 = blockIdx.x % (cols / 64) * 64;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = 32 * i + (threadIdx.x >> 3), c = 8 * (threadIdx.x & 7);
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(in + (int64_t)(r0 + r) * cols + c0 + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t *>(&tile[r][c + 2 * e]) = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = 32 * i + (threadIdx.x >> 3), r = 8 * (threadIdx.x & 7);
        u32x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tile[r + 2 * e][c] | (uint32_t)tile[r + 2 * e + 1][c] << 16;
        *reinterpret_cast<u32x4_t *>(out + (int64_t)(c0 + c) * rows + r0 + r) = v;
    }
}

hipError_t launch_transpose(const void *in, void *out, int rows, int cols, hipStream_t stream) {
    (void)hipGetLastError();
    hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)(rows / 64) * (unsigned)(cols / 64)), dim3(256), 0, stream, static_cast<const uint16_t *>(in), static_cast<uint16_t *>(out), rows, cols);
    return hipGetLastError();
}

} // namespace fb
