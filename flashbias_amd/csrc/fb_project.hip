// Projections of one input by up to three weights in one launch (the q, k and v projections of an attention block,
// 1_Language_Model/attention_with_alibi_bias.py:26-28): y_i (tokens, n_i) = x (tokens, k) w_i^T, fp32 sums, rounded once.
//
// For a few thousand tokens one product of this kind does not fill the chip: 1500 x 1600 x 1600 is 84 tiles of 256 x 128.  The
// three weights' tiles together are one round of workgroups (252).  Measured, three weights, against three products of
// the vendor library (us): 1500 x 1600 x 1600 28.7 / 50.3, 600 x 1024 x 1024 11.3 / 22.6, 256 x 512 x 512 7.2 / 15.8,
// 4096 x 512 x 512 12.7 / 23.4, 2048 x 2048 x 2048 64 / 69, 4096 x 1600 x 1600 88 / 96.  What bounds it: at one round, the
// fill and drain of the pipeline around k / 64 steps of about 2000 cycles of matrix work a SIMD (750 TFLOP/s); the library is ahead
// (238 / 278 at 4096 x 3200 x 3200) where many rounds of larger tiles hide both.
//
// A workgroup forms a tile of 64 WN channels x 64 WM tokens, a wave 64 x 64 of it (D = W X^T, so a lane holds a token and its
// registers channels).  Both operands stream through three LDS stages of 64 columns (rows of 128 bytes, the dense regions of
// fb_lean_tiles.h): one in use and two on their way.  Every wave issues the same number of copies in every step (past the
// end: the last columns again), so the waits are constants.  Tiles of 256 x 128 with eight waves (144 KB, one workgroup a compute
// unit) move the fewest bytes per product; where tiles of 128 x 64 with two waves (72 KB, two a unit) are no more than one
// round, they are ahead by filling more of the chip (600 x 1024 x 1024: 11.3 against 16.1; 1024 x 1024 x 1024: 15.6 / 16.5;
// just past a round, 1500 x 1024 x 1024, 23.4 against 17.9).  Tiles of 128 x 128 and 64 x 64 were ahead nowhere by more than
// a few per cent; 32 columns a step in five stages took 37.1 for 1500 x 1600 x 1600.
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
    auto issue = [&](int step, int stage) {
        const int at = min(step, nsteps - 1) * 128;
        const uint32_t dst = lds0 + stage * C::STAGE;
#pragma unroll
        for (int j = 0; j < C::CW; ++j) lds_dma16_all(off[j], wp + at, dst + (C::CW * wave + j) * 1024);
#pragma unroll
        for (int j = 0; j < C::CX; ++j) lds_dma16_all(off[C::CW + j], xp + at, dst + C::SW + (C::CX * wave + j) * 1024);
    };
    issue(0, 0);
    issue(1, 1);

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
        issue(step + 2, stage == 0 ? 2 : stage - 1); // (the stage of the step before: everyone has left it)
        const uint32_t aw = lds0 + stage * C::STAGE + 8192 * wn, ax = lds0 + stage * C::STAGE + C::SW + 8192 * wm;
        u32x4_t wf[2][4], xf[2][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                wf[p][t] = lds_load16(aw + 4096 * p + row_off[t]);
                xf[p][t] = lds_load16(ax + 4096 * p + row_off[t]);
            }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q) acc[p][q] = T::mfma(wf[p][t], xf[q][t], acc[p][q]);
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

// Up to three rounds of the large tile: at exactly three 38.7 us against the library's 47.1 (16384 x 512 x 512) and 62 / 64
// (8192 x 1024 x 1024); four and more 123 / 107 (6144 x 1600 x 1600), 278 / 238 (4096 x 3200 x 3200), 50 / 50 (65536 x 256
// x 256).  A single weight gains nothing from the shared launch (1500 x 1600 x 1600: 29.5 against 17.4).
bool project_recommended(int64_t tokens, const int *n, int count) {
    return count == 3 && project_tiles<256, 128>(tokens, n, count) <= 3 * (int64_t)num_cus();
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
    if (project_tiles<128, 64>(tokens, n, count) <= 2 * (int64_t)num_cus())
        return bf16 ? launch_project_t<BF16, 2, 1>(a, stream) : launch_project_t<F16, 2, 1>(a, stream);
    return bf16 ? launch_project_t<BF16, 4, 2>(a, stream) : launch_project_t<F16, 4, 2>(a, stream);
}

} // namespace fb
