// Projections of one input by up to three weights in one launch (the q, k and v projections of an attention block,
// 1_Language_Model/attention_with_alibi_bias.py:26-28): y_i (tokens, n_i) = x (tokens, k) w_i^T, fp32 sums, rounded once.
//
// For a few thousand tokens one product of this kind does not fill the chip: 1500 x 1600 x 1600 is 84 tiles of 256 x 128.  The
// three weights' tiles together are one round of workgroups (252).  Measured, three weights, against three products of
// the vendor library (us): 1500 x 1600 x 1600 27.8 / 50.3, 600 x 1024 x 1024 9.8 / 22.6, 256 x 512 x 512 6.3 / 15.8,
// 4096 x 512 x 512 12.1 / 23.4, 2048 x 1024 x 1024 18.5 / 31, 4096 x 1600 x 1600 83 / 96.  What bounds it: a wave's own
// order of copies, LDS reads and products, about 1000 cycles a step where the products take 512 (more stages change nothing); the
// library is ahead (238 / 278 at 4096 x 3200 x 3200) where many rounds of larger tiles hide it.
//
// A workgroup forms a tile of 64 WN channels x 64 WM tokens, a wave 64 x 64 of it (D = W X^T, so a lane holds a token and its
// registers channels).  Both operands stream through three LDS stages of 64 columns (rows of 128 bytes, the dense regions of
// fb_lean_tiles.h): one in use and two on their way.  The copies of a step are issued between its products (all of them ahead
// of the fragment reads: 1600 channels 28.7, 600 x 1024 x 1024 11.0, one token 13.6 against 11.9).  Every wave issues the same
// number of them in every step (past the end: the last columns again), so the waits are constants.  Four and five stages of the
// 128 x 64 tile measured as three do; 32 columns a step in five stages took 37.1 for 1500 x 1600 x 1600.
#include "fb_kernels.h"
#include "fb_lean_tiles.h"

namespace fb {

struct ProjectArgs {
    const uint16_t *x, *w[3];
    uint16_t *y[3];
    int64_t ldx;
    int n[3];       // channels of each weight, 0: none
    int tiles[3];   // ... in tiles
    int tokens, k;
    int ttiles;     // token tiles
};

// WN: waves along the channels (64 each), WM along the tokens (64 each).
template <class T_, int WN_, int WM_>
struct ProjectCfg {
    typedef T_ T;
    static constexpr int WN = WN_, WM = WM_, TN = 64 * WN, TM = 64 * WM;
    static constexpr int NWAVES = WN * WM, NTHREADS = 64 * NWAVES, NSTAGE = 3;
    static constexpr int SW = TN * 128, STAGE = (TN + TM) * 128, LDS_BYTES = NSTAGE * STAGE;
    static constexpr int CW = TN / 8 / NWAVES, CX = TM / 8 / NWAVES; // copies of a wave and step, eight rows each
    static constexpr int EU_WAVES = 160 * 1024 / LDS_BYTES * NWAVES / 4;
};

template <class C>
__global__ __launch_bounds__(C::NTHREADS) __attribute__((amdgpu_waves_per_eu(C::EU_WAVES))) void project_kernel(const ProjectArgs a) {
    typedef typename C::T T;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t lds0 = lds_addr_of(smem);
    const int lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wn = wave % C::WN, wm = wave / C::WN; // this wave's 64 channels and 64 tokens

    // token tiles of a channel tile next to each other: an XCD's share reads few rows of the weights and all of x
    const int work = xcd_remap(blockIdx.x, (a.tiles[0] + a.tiles[1] + a.tiles[2]) * a.ttiles);
    int nt = work / a.ttiles;
    const int m0 = (work % a.ttiles) * C::TM;
    int i = 0;
    if (nt >= a.tiles[0]) {
        nt -= a.tiles[0];
        i = 1;
        if (nt >= a.tiles[1]) {
            nt -= a.tiles[1];
            i = 2;
        }
    }
    const int n0 = nt * C::TN, n = a.n[i];

    // Copies of eight 128-byte rows, chunks swizzled by the row (swz_of<8>); rows past the end: the last one again.
    uint32_t off[C::CW + C::CX];
#pragma unroll
    for (int j = 0; j < C::CW + C::CX; ++j) {
        const bool is_w = j < C::CW;
        const int row = 8 * (is_w ? C::CW * wave + j : C::CX * wave + j - C::CW) + (lane >> 3), chunk = (lane & 7) ^ swz_of<8>(row);
        off[j] = is_w ? (uint32_t)min(row, n - 1 - n0) * (uint32_t)(a.k * 2) + chunk * 16
                      : (uint32_t)min(row, a.tokens - 1 - m0) * (uint32_t)(a.ldx * 2) + chunk * 16;
    }
    const uint8_t *wp = reinterpret_cast<const uint8_t *>(a.w[i]) + (int64_t)n0 * a.k * 2, *xp = reinterpret_cast<const uint8_t *>(a.x) + (int64_t)m0 * a.ldx * 2;
    const int nsteps = a.k / 64;
    auto issue = [&](int step, int stage, int part, int parts) { // (this part of the copies)
        const int at = min(step, nsteps - 1) * 128;
        const uint32_t dst = lds0 + stage * C::STAGE;
#pragma unroll
        for (int j = 0; j < C::CW + C::CX; ++j)
            if (j * parts / (C::CW + C::CX) == part) {
                if (j < C::CW)
                    lds_dma16_all(off[j], wp + at, dst + (C::CW * wave + j) * 1024);
                else
                    lds_dma16_all(off[j], xp + at, dst + C::SW + (C::CX * wave + j - C::CW) * 1024);
            }
    };
    issue(0, 0, 0, 1);
    issue(1, 1, 0, 1);

    f32x16_t acc[2][2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[p][q][v] = 0.f;
    uint32_t row_off[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) row_off[t] = 2 * swz_off<8>(c, 2 * t + g);
    wait_vmcnt<C::CW + C::CX>();
    barrier_lds();
    int stage = 0;
#pragma unroll 1
    for (int step = 0; step < nsteps; ++step) {
        const int into = stage == 0 ? 2 : stage - 1; // (the stage of the step before: everyone has left it)
        const uint32_t aw = lds0 + stage * C::STAGE + 8192 * wn, ax = lds0 + stage * C::STAGE + C::SW + 8192 * wm;
        u32x4_t wf[2][4], xf[2][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                wf[p][t] = lds_load16(aw + 4096 * p + row_off[t]);
                xf[p][t] = lds_load16(ax + 4096 * p + row_off[t]);
            }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q) acc[p][q] = T::mfma(wf[p][t], xf[q][t], acc[p][q]);
            issue(step + 2, into, t, 4);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        wait_vmcnt<C::CW + C::CX>(); // the next step's columns
        barrier_lds();
        stage = stage == 2 ? 0 : stage + 1;
    }
    wait_vmcnt<0>();
    barrier_lds(); // (the stages become the waves' output buffers)

    // 32 tokens x 64 channels at a time through 4 KB of this wave's own: lines of 128 bytes, chunks XORed with the line
    uint8_t *buf = smem + wave * 4096;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            asm volatile("s_nop 11" : "+v"(acc[p][q]));
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<u32x2_t *>(buf + c * 128 + (((4 * p + j) ^ (c & 7)) << 4) + 8 * g) =
                    u32x2_t{T::pack2(acc[p][q][4 * j], acc[p][q][4 * j + 1]), T::pack2(acc[p][q][4 * j + 2], acc[p][q][4 * j + 3])};
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int line = 8 * r + (lane >> 3), token = m0 + 64 * wm + 32 * q + line, ch = n0 + 64 * wn + 8 * (lane & 7);
            const u32x4_t v = *reinterpret_cast<const u32x4_t *>(buf + line * 128 + (((lane & 7) ^ (line & 7)) << 4));
            if (token < a.tokens && ch < n) *reinterpret_cast<u32x4_t *>(a.y[i] + (int64_t)token * n + ch) = v;
        }
    }
}

template <int TN, int TM>
static int64_t project_tiles(int64_t tokens, const int *n, int count) {
    int64_t channels = 0;
    for (int i = 0; i < count; ++i) channels += (n[i] + TN - 1) / TN;
    return channels * ((tokens + TM - 1) / TM);
}

// Up to three rounds of the large tile: at exactly three 37.0 us against the library's 47.1 (16384 x 512 x 512); four and more
// 116 / 107 (6144 x 1600 x 1600), 278 / 238 (4096 x 3200 x 3200), 47 / 50 (65536 x 256 x 256).  A single weight gains nothing from
// the shared launch (1500 x 1600 x 1600: 29.5 against 17.4).
// Up to 4096 columns of x: a workgroup walks all of them, 6.5 us per 1024 however few tiles there are, where the library splits
// long sums.  Few tokens, weights from memory, this / library, us: 1 x 1024 x 1024 9.1 / 17.0, 1 x 2048 x 64 14.6 / 15.4,
// 16 x 1600 x 1600 12.5 / 25.9, 1 x 4096 x 256 25.6 / 32.5 (32 tokens 26.0 / 25.4), 1 x 4096 x 4096 37.4 / 46.5 (32: 37.4 / 39.4);
// 16 x 5120 x 512 36.7 / 23.8, 1 x 5120 x 5120 50.8 / 43.8, 1 x 8192 x 1024 59.4 / 35.1, 64 x 16384 x 256 123 / 55.
bool project_recommended(int64_t tokens, int k, const int *n, int count) {
    return count == 3 && k <= 4096 && project_tiles<256, 128>(tokens, n, count) <= 3 * (int64_t)num_cus();
}

template <class T, int WN, int WM>
static hipError_t launch_project_t(ProjectArgs a, hipStream_t stream) {
    typedef ProjectCfg<T, WN, WM> C;
    a.ttiles = (a.tokens + C::TM - 1) / C::TM;
    for (int i = 0; i < 3; ++i) a.tiles[i] = (a.n[i] + C::TN - 1) / C::TN;
    auto kern = project_kernel<C>;
    static KernelOnce once;
    const hipError_t e = allow_lds(kern, C::LDS_BYTES, once);
    if (e != hipSuccess) return e;
    return launch_flat(kern, (int64_t)(a.tiles[0] + a.tiles[1] + a.tiles[2]) * a.ttiles, C::NTHREADS, C::LDS_BYTES, stream, a);
}

hipError_t launch_project(const void *x, int64_t ldx, const void *const *w, void *const *y, const int *n, int count, int64_t tokens, int k, bool bf16,
                          hipStream_t stream) {
    ProjectArgs a = {};
    a.x = static_cast<const uint16_t *>(x);
    a.ldx = ldx;
    a.tokens = (int)tokens;
    a.k = k;
    for (int i = 0; i < count; ++i) {
        a.w[i] = static_cast<const uint16_t *>(w[i]);
        a.y[i] = static_cast<uint16_t *>(y[i]);
        a.n[i] = n[i];
    }
    // The tile that fills the chip in one round, us (256 x 128 with eight waves, 144 KB and one workgroup a compute unit / 128 x 128
    // with four, 96 KB, one / 128 x 64 with two, 72 KB, two): 600 x 1024 x 1024 14.7 / 10.1 / 9.8 (240 of the small ones),
    // 1024 x 1024 x 1024 15.5 / 10.7 / 14.7 (384 of them, 192 of 128 x 128), 2048 x 512 x 512 11.4 / 8.7 / 10.1 (the same),
    // 777 x 1600 x 1600 22.9 / 27.0 / 20.2 (507, 273), 2048 x 768 x 768 14.5 / 16.7 / 16.9 (576, 288), 4096 x 512 x 512 12.1 /
    // 13.3 / 15.0.  Tiles of 64 x 64 with one wave are ahead nowhere.
    const int64_t cus = num_cus(), small = project_tiles<128, 64>(tokens, n, count);
    if (small > cus && project_tiles<128, 128>(tokens, n, count) <= cus)
        return bf16 ? launch_project_t<BF16, 2, 2>(a, stream) : launch_project_t<F16, 2, 2>(a, stream);
    if (small <= 2 * cus) return bf16 ? launch_project_t<BF16, 2, 1>(a, stream) : launch_project_t<F16, 2, 1>(a, stream);
    return bf16 ? launch_project_t<BF16, 4, 2>(a, stream) : launch_project_t<F16, 4, 2>(a, stream);
}

} // namespace fb
