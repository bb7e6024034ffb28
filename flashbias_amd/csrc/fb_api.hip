// C ABI of the library (declared in include/flashbias.h): translation of fb_params into kernel
// argument blocks and dispatch to the instantiation that covers (dtype, head dim, rank).  The
// argument checks themselves (fb_check) are plain C++ in fb_checks.cpp.
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "flashbias.h"
#include "fb_checks.h"
#include "fb_kernels.h"

namespace fb {
#define FB_DECL(sfx)                                                          \
    hipError_t launch_fwd_##sfx(const FwdArgs &a, hipStream_t stream);        \
    hipError_t launch_bwd_dkv_##sfx(const BwdArgs &a, hipStream_t stream);    \
    hipError_t launch_bwd_dq_##sfx(const BwdArgs &a, hipStream_t stream);
FB_DECL(bf16_1) FB_DECL(bf16_2) FB_DECL(bf16_4) FB_DECL(bf16_8)
FB_DECL(f16_1) FB_DECL(f16_2) FB_DECL(f16_4) FB_DECL(f16_8)
#undef FB_DECL
hipError_t launch_bwd_both_bf16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_both_f16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_both_general_bf16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_both_general_f16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_win_bf16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_win_f16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_fwd_win_bf16_2(const FwdArgs &a, hipStream_t stream);
hipError_t launch_fwd_win_f16_2(const FwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_ring_bf16_2(const BwdArgs &a, hipStream_t stream);
hipError_t launch_bwd_ring_f16_2(const BwdArgs &a, hipStream_t stream);

// elementwise part of a cosine-attention window block (fb_cosine.hip)
hipError_t launch_cosine(const fb_cosine *p, bool fp32, bool backward, hipStream_t stream);
hipError_t launch_cosine_scale_grad(const fb_cosine *p, int shares, hipStream_t stream);
int64_t cosine_sweep(int64_t tokens, int H, int d);

// weight and bias gradient of a projection (fb_wgrad.hip)
size_t wgrad_workspace(int64_t tokens, int n, int k, bool bias);
bool wgrad_recommended(int64_t tokens, int n, int k);
hipError_t launch_wgrad(const void *dy, int64_t ldy, const void *x, int64_t ldx, void *dw, void *db, float *partial, int64_t tokens,
                        int n, int k, bool bf16, hipStream_t stream);
// projections of one input by up to three weights (fb_project.hip)
bool project_recommended(int64_t tokens, int k, const int *n, int count);
hipError_t launch_project(const void *x, int64_t ldx, const void *const *w, void *const *y, const int *n, int count, int64_t tokens, int k, bool bf16,
                          hipStream_t stream);
// a projection of many tokens (fb_linear.hip)
bool linear_recommended(int64_t tokens, int n, int k);
hipError_t launch_linear(const void *x, int64_t ldx, const void *w, const void *b, void *y, int64_t tokens, int n, int k, bool bf16, hipStream_t stream);
hipError_t launch_transpose(const void *in, void *out, int rows, int cols, hipStream_t stream);

hipError_t launch_fwd(const FwdArgs &a, bool bf16, hipStream_t stream) {
    if (window_forward(a)) return bf16 ? launch_fwd_win_bf16_2(a, stream) : launch_fwd_win_f16_2(a, stream);
    switch (nkd_of(a.d)) {
    case 1: return bf16 ? launch_fwd_bf16_1(a, stream) : launch_fwd_f16_1(a, stream);
    case 2: return bf16 ? launch_fwd_bf16_2(a, stream) : launch_fwd_f16_2(a, stream);
    case 4: return bf16 ? launch_fwd_bf16_4(a, stream) : launch_fwd_f16_4(a, stream);
    default: return bf16 ? launch_fwd_bf16_8(a, stream) : launch_fwd_f16_8(a, stream);
    }
}

hipError_t launch_bwd_dkv(const BwdArgs &a, bool bf16, hipStream_t stream) {
    switch (nkd_of(a.d)) {
    case 1: return bf16 ? launch_bwd_dkv_bf16_1(a, stream) : launch_bwd_dkv_f16_1(a, stream);
    case 2: return bf16 ? launch_bwd_dkv_bf16_2(a, stream) : launch_bwd_dkv_f16_2(a, stream);
    case 4: return bf16 ? launch_bwd_dkv_bf16_4(a, stream) : launch_bwd_dkv_f16_4(a, stream);
    default: return bf16 ? launch_bwd_dkv_bf16_8(a, stream) : launch_bwd_dkv_f16_8(a, stream);
    }
}

hipError_t launch_bwd_dq(const BwdArgs &a, bool bf16, hipStream_t stream) {
    switch (nkd_of(a.d)) {
    case 1: return bf16 ? launch_bwd_dq_bf16_1(a, stream) : launch_bwd_dq_f16_1(a, stream);
    case 2: return bf16 ? launch_bwd_dq_bf16_2(a, stream) : launch_bwd_dq_f16_2(a, stream);
    case 4: return bf16 ? launch_bwd_dq_bf16_4(a, stream) : launch_bwd_dq_f16_4(a, stream);
    default: return bf16 ? launch_bwd_dq_bf16_8(a, stream) : launch_bwd_dq_f16_8(a, stream);
    }
}
// dq and dk/dv workgroups of the streamlined kernels in one launch (fb_bwd_both.hip; head dim 32)
hipError_t launch_bwd_both(const BwdArgs &a, bool bf16, hipStream_t stream) {
    return bf16 ? launch_bwd_both_bf16_2(a, stream) : launch_bwd_both_f16_2(a, stream);
}
// the same for the calls with factors of rank 8 ... 32 that the streamlined kernels do not cover
hipError_t launch_bwd_both_general(const BwdArgs &a, bool bf16, hipStream_t stream) {
    return bf16 ? launch_bwd_both_general_bf16_2(a, stream) : launch_bwd_both_general_f16_2(a, stream);
}
// all five gradients of a short sequence in one workgroup (fb_bwd_win.hip; head dim 32)
hipError_t launch_bwd_win(const BwdArgs &a, bool bf16, hipStream_t stream) {
    return bf16 ? launch_bwd_win_bf16_2(a, stream) : launch_bwd_win_f16_2(a, stream);
}
// the same without factor gradients, two workgroups per compute unit (fb_bwd_ring.hip; head dim 32)
hipError_t launch_bwd_ring(const BwdArgs &a, bool bf16, hipStream_t stream) {
    return bf16 ? launch_bwd_ring_bf16_2(a, stream) : launch_bwd_ring_f16_2(a, stream);
}
} // namespace fb

// Scratch of fb_bwd_static: device memory that belongs to the library image, so that the entry
// point never calls an allocator.  One copy per GPU that loads the library; it keeps the last
// call's contents (the backward overwrites every element it later reads, nothing has to start
// at zero).  In host code the array's name is only a handle for hipGetSymbolAddress: the kernels
// get the address that call returns.
static __device__ __align__(256) unsigned char scratch[FB_STATIC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {nullptr}; // address of `scratch` on each device, looked up once

// Address of this device's copy of the scratch array (looked up on first use with the device
// current), or nullptr with *err set.
void *static_scratch(hipError_t *err) {
    int dev = 0;
    *err = hipGetDevice(&dev);
    if (*err != hipSuccess) return nullptr;
    if (dev < 0 || dev >= kMaxDevices) {
        *err = hipErrorInvalidDevice;
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        *err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (*err != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

bool vec_ok(const fb_tensor &t) {
    return (reinterpret_cast<uintptr_t>(t.ptr) % 16 == 0) && t.stride_b % 8 == 0 && t.stride_h % 8 == 0 &&
           t.stride_s % 8 == 0;
}

fb::Tensor dev(const fb_tensor &t) {
    fb::Tensor o;
    o.ptr = static_cast<const uint16_t *>(t.ptr);
    o.sb = t.stride_b;
    o.sh = t.stride_h;
    o.ss = t.stride_s;
    o.vec_ok = vec_ok(t) ? 1 : 0;
    return o;
}

fb::MaskDesc dev_mask(const fb_params *p) {
    fb::MaskDesc m;
    m.ptr = p->mask_type ? p->mask.ptr : nullptr;
    m.sb = p->mask.stride_b;
    m.sh = p->mask.stride_h;
    m.batches = fb::mask_batches(p);
    m.sm = p->mask_type == FB_MASK_MATRIX ? p->mask.stride_s : 0;
    m.type = p->mask_type;
    m.is_f32 = p->mask_dtype == FB_F32;
    const uintptr_t align = m.is_f32 ? 16 : 8; // four consecutive keys
    m.vec_ok = p->mask_type && reinterpret_cast<uintptr_t>(m.ptr) % align == 0 && m.sb % 4 == 0 && m.sh % 4 == 0 &&
               m.sm % 4 == 0;
    return m;
}

fb::FwdArgs fwd_args(const fb_params *p) {
    fb::FwdArgs a;
    std::memset(&a, 0, sizeof(a));
    a.q = dev(p->q);
    a.k = dev(p->k);
    a.v = dev(p->v);
    a.o = dev(p->o);
    if (p->r > 0) {
        a.qb = dev(p->q_bias);
        a.kb = dev(p->k_bias);
    }
    a.mask = dev_mask(p);
    a.lse = p->lse;
    a.B = p->B; a.H = p->H; a.Lq = p->Lq; a.Lk = p->Lk; a.d = p->d; a.r = p->r;
    a.causal = p->causal ? 1 : 0;
    a.scale = p->scale;
    return a;
}

fb::BwdArgs bwd_args(const fb_params *p) {
    fb::BwdArgs a;
    std::memset(&a, 0, sizeof(a));
    a.q = dev(p->q);
    a.k = dev(p->k);
    a.v = dev(p->v);
    a.o = dev(p->o);
    a.dout = dev(p->dout);
    a.dq = dev(p->dq);
    a.dk = dev(p->dk);
    a.dv = dev(p->dv);
    if (p->r > 0) {
        a.qb = dev(p->q_bias);
        a.kb = dev(p->k_bias);
        a.dqb = dev(p->dq_bias);
        a.dkb = dev(p->dk_bias);
    }
    a.mask = dev_mask(p);
    a.lse = p->lse;
    a.delta = p->delta;
    a.B = p->B; a.H = p->H; a.Lq = p->Lq; a.Lk = p->Lk; a.d = p->d; a.r = p->r;
    a.causal = p->causal ? 1 : 0;
    a.scale = p->scale;
    a.group = p->r > 0 && p->bias_grad_group > 1 ? p->bias_grad_group : 1;
    a.stat_chunks = fb::dkv_streamlined(a) ? 1 : 0;
    return a;
}

int launched(hipError_t e, const char *what) {
    if (e == hipSuccess) return FB_OK;
    return fb::api_fail(FB_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
}

} // namespace

extern "C" {

int fb_init(void) {
    fb::api_clear_error();
    hipError_t e = hipSuccess;
    if (!static_scratch(&e)) return launched(e, "fb_init (hipGetSymbolAddress)");
    return FB_OK;
}

int fb_fwd(const fb_params *p, void *stream) {
    const int rc = fb_check(p, 0);
    if (rc) return rc;
    return launched(fb::launch_fwd(fwd_args(p), p->dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_fwd");
}

int fb_bwd_preprocess(const fb_params *p, void *stream) {
    const int rc = fb_check(p, 1);
    if (rc) return rc;
    return launched(fb::launch_bwd_preprocess(bwd_args(p), p->dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                    "fb_bwd_preprocess");
}

int fb_bwd_dkv(const fb_params *p, void *stream) {
    const int rc = fb_check(p, 1);
    if (rc) return rc;
    return launched(fb::launch_bwd_dkv(bwd_args(p), p->dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                    "fb_bwd_dkv");
}

int fb_bwd_dq(const fb_params *p, void *stream) {
    const int rc = fb_check(p, 1);
    if (rc) return rc;
    return launched(fb::launch_bwd_dq(bwd_args(p), p->dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                    "fb_bwd_dq");
}

int fb_sum_over_batch(const void *full, void *out, int dtype, int out_dtype, int64_t B, int64_t n, int64_t batch_stride,
                      void *stream) {
    fb::api_clear_error();
    if (!full || !out) return fb::api_fail(FB_ERR_NULL, "fb_sum_over_batch: null pointer");
    if (dtype != FB_F16 && dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (out_dtype != dtype && out_dtype != FB_F32) return fb::api_fail(FB_ERR_DTYPE, "output must have the input dtype or fp32");
    if (B <= 0 || n <= 0 || (n + 63) / 64 > 0x7fffffff) return fb::api_fail(FB_ERR_SHAPE, "B and n must be positive (n below 2^37)");
    if (n % 8 != 0 || batch_stride % 8 != 0 || batch_stride < n || reinterpret_cast<uintptr_t>(full) % 16 != 0)
        return fb::api_fail(FB_ERR_STRIDE, "fb_sum_over_batch: rows must be 16-byte aligned multiples of 8 elements that do not overlap");
    return launched(fb::launch_sum_over_batch(full, out, dtype == FB_BF16, out_dtype == FB_F32, B, n, batch_stride,
                                              static_cast<hipStream_t>(stream)),
                    "fb_sum_over_batch");
}

int fb_resize_rank(const void *in, void *out, int64_t rows, int r_in, int r_out, void *stream) {
    fb::api_clear_error();
    if (!in || !out) return fb::api_fail(FB_ERR_NULL, "fb_resize_rank: null pointer");
    if (rows <= 0 || r_in <= 0 || r_out <= 0 || r_in > 4096 || r_out > 4096 || (rows + 255) / 256 > 0x7fffffff)
        return fb::api_fail(FB_ERR_SHAPE, "fb_resize_rank: rows and both ranks must be positive (ranks up to 4096, rows below 2^39)");
    return launched(fb::launch_resize_rank(in, out, rows, nullptr, nullptr, 0, r_in, r_out, static_cast<hipStream_t>(stream)), "fb_resize_rank");
}

int fb_resize_ranks(const void *q_in, void *q_out, int64_t q_rows, const void *k_in, void *k_out, int64_t k_rows, int r_in, int r_out,
                    void *stream) {
    fb::api_clear_error();
    if (!q_in || !q_out || !k_in || !k_out) return fb::api_fail(FB_ERR_NULL, "fb_resize_ranks: null pointer");
    if (q_rows <= 0 || k_rows <= 0 || r_in <= 0 || r_out <= 0 || r_in > 4096 || r_out > 4096 || (q_rows + 255) / 256 > 0x3fffffff ||
        (k_rows + 255) / 256 > 0x3fffffff)
        return fb::api_fail(FB_ERR_SHAPE, "fb_resize_ranks: rows and both ranks must be positive (ranks up to 4096, rows below 2^38)");
    return launched(fb::launch_resize_rank(q_in, q_out, q_rows, k_in, k_out, k_rows, r_in, r_out, static_cast<hipStream_t>(stream)), "fb_resize_ranks");
}

int fb_alibi_factors(void *q_bias, void *k_bias, int dtype, int Lq, int Lk, int H, int r, int reference_sign, void *stream) {
    fb::api_clear_error();
    if (!q_bias || !k_bias) return fb::api_fail(FB_ERR_NULL, "fb_alibi_factors: null pointer");
    if (dtype != FB_F16 && dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (Lq <= 0 || Lk <= 0 || Lq > 65536 || Lk > 65536 || H <= 0 || H > (1 << 20) || r < 8 || r > FB_MAX_RANK || r % 8 != 0)
        return fb::api_fail(FB_ERR_SHAPE, "fb_alibi_factors: up to 65536 positions, a rank of 8, 16, ... 128");
    if (reinterpret_cast<uintptr_t>(q_bias) % 16 != 0 || reinterpret_cast<uintptr_t>(k_bias) % 16 != 0)
        return fb::api_fail(FB_ERR_STRIDE, "fb_alibi_factors: factors must be 16-byte aligned");
    return launched(fb::launch_alibi_factors(q_bias, k_bias, dtype == FB_BF16, Lq, Lk, H, r, reference_sign != 0, static_cast<hipStream_t>(stream)),
                    "fb_alibi_factors");
}

// Sizes a caller's block may have (the shorter one: before there was `fp32`).
static bool known_size(const fb_cosine *p) { return p->size == sizeof(fb_cosine) || p->size == offsetof(fb_cosine, fp32); }

static int check_cosine(const fb_cosine *p, bool backward) {
    fb::api_clear_error();
    if (!p) return fb::api_fail(FB_ERR_NULL, "fb_cosine: null pointer");
    if (!known_size(p))
        return fb::api_fail(FB_ERR_ABI, "fb_cosine.size does not match this library");
    if (p->dtype != FB_F16 && p->dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (p->in_dtype < FB_F16 || p->in_dtype > FB_F32 || p->scale_dtype < FB_F16 || p->scale_dtype > FB_F32)
        return fb::api_fail(FB_ERR_DTYPE, "qkv and logit_scale must be fp16, bf16 or fp32");
    if (p->tokens <= 0 || p->H <= 0 || p->H > (1 << 20) || p->d < 8 || p->d > FB_MAX_HEADDIM || (p->d & (p->d - 1)))
        return fb::api_fail(FB_ERR_SHAPE, "fb_cosine: tokens and H must be positive, d one of 8, 16, 32, 64, 128");
    const void *need[] = {p->qkv, p->logit_scale, backward ? p->dq : p->q, backward ? p->dk : p->k, backward ? p->dqkv : p->q};
    for (const void *x : need)
        if (!x) return fb::api_fail(FB_ERR_NULL, "fb_cosine: null pointer");
    const void *rows[] = {p->qkv, p->q, p->k, p->v, p->dq, p->dk, p->dv, p->dqkv};
    for (const void *x : rows)
        if (reinterpret_cast<uintptr_t>(x) % 16 != 0) return fb::api_fail(FB_ERR_STRIDE, "fb_cosine: tensors must be 16-byte aligned");
    if (backward) {
        if (!p->dlogit_scale || !p->partial) return fb::api_fail(FB_ERR_NULL, "fb_cosine: null pointer");
        if (p->grad_stride < (int64_t)p->H * p->d || p->grad_stride % 8 != 0)
            return fb::api_fail(FB_ERR_STRIDE, "fb_cosine: grad_stride must be a multiple of 8 and at least H d");
    }
    return FB_OK;
}

// (a block that ends before the field was there: 0)
static bool cosine_fp32(const fb_cosine *p) { return p->size > offsetof(fb_cosine, fp32) && p->fp32 != 0; }

size_t fb_cosine_workspace_bytes(const fb_cosine *p) {
    if (!p || p->tokens <= 0 || p->H <= 0 || p->d < 8) return 0;
    return (size_t)fb::cosine_sweep(p->tokens, p->H, p->d) * p->H * sizeof(float);
}

int fb_cosine_fwd(const fb_cosine *p, void *stream) {
    const int rc = check_cosine(p, false);
    if (rc) return rc;
    return launched(fb::launch_cosine(p, cosine_fp32(p), false, static_cast<hipStream_t>(stream)), "fb_cosine_fwd");
}

int fb_cosine_bwd(const fb_cosine *p, void *stream) {
    const int rc = check_cosine(p, true);
    if (rc) return rc;
    return launched(fb::launch_cosine(p, cosine_fp32(p), true, static_cast<hipStream_t>(stream)), "fb_cosine_bwd");
}

// A cosine block's attention with the normalisation inside: q, k, v (and dq, dk, dv) of p are the parts of the projection c.qkv.
static bool window_block(const fb_params *p, const fb_cosine *c, bool backward) {
    return p->scale == 1.f && c->dtype == p->dtype && c->in_dtype == p->dtype && !cosine_fp32(c) &&
           c->scale_dtype >= FB_F16 && c->scale_dtype <= FB_F32 && c->logit_scale && c->H == p->H && c->d == p->d &&
           (backward ? fb::ring_shape(bwd_args(p)) && p->mask_type != FB_MASK_VECTOR : fb::window_shape(fwd_args(p)));
}

static int check_window(const fb_params *p, const fb_cosine *c, bool backward) {
    if (!backward || !p || !fb::known_size(p)) {
        const int rc = fb_check(p, backward);
        if (rc) return rc;
    } else { // (the scratch buffer is not used: any address will do for the check)
        fb_params q;
        std::memset(&q, 0, sizeof(q));
        std::memcpy(&q, p, p->size);
        q.delta = p->lse;
        const int rc = fb_check(&q, 1);
        if (rc) return rc;
    }
    if (!c) return fb::api_fail(FB_ERR_NULL, "fb_window: null pointer");
    if (!known_size(c)) return fb::api_fail(FB_ERR_ABI, "fb_cosine.size does not match this library");
    if (!window_block(p, c, backward)) return fb::api_fail(FB_ERR_SHAPE, "fb_window: not a block that fb_window_ready takes");
    return FB_OK;
}

int fb_window_ready(const fb_params *p, const fb_cosine *c, int pass) {
    const fb::KeptError kept; // (a "no" is an answer, nothing has failed)
    return check_window(p, c, pass == 1) == FB_OK ? 1 : 0;
}

size_t fb_window_workspace_bytes(const fb_params *p) {
    if (!p || p->B <= 0 || p->H <= 0) return 0;
    return (size_t)p->B * p->H * 4 * sizeof(float); // (a share of each wave; workgroups that walk several entries leave fewer)
}

int fb_window_fwd(const fb_params *p, const fb_cosine *c, void *stream) {
    const int rc = check_window(p, c, false);
    if (rc) return rc;
    fb::FwdArgs a = fwd_args(p);
    a.cosine = {c->logit_scale, c->scale_dtype};
    return launched((p->dtype == FB_BF16 ? fb::launch_fwd_win_bf16_2 : fb::launch_fwd_win_f16_2)(a, static_cast<hipStream_t>(stream)), "fb_window_fwd");
}

int fb_window_bwd(const fb_params *p, const fb_cosine *c, void *stream) {
    const int rc = check_window(p, c, true);
    if (rc) return rc;
    if (!c->dlogit_scale || !c->partial) return fb::api_fail(FB_ERR_NULL, "fb_window_bwd: null pointer");
    fb::BwdArgs a = bwd_args(p);
    a.cosine = {c->logit_scale, c->scale_dtype};
    a.cosine_partial = c->partial;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int rc2 = launched(fb::launch_bwd_ring(a, p->dtype == FB_BF16, s), "fb_window_bwd");
    if (rc2) return rc2;
    const int walk = fb::ring_walk(a.B, a.H);
    return launched(fb::launch_cosine_scale_grad(c, 4 * ((a.B + walk - 1) / walk), s), "fb_window_bwd (logit scale)");
}

static bool weight_grad_sizes(int64_t tokens, int n, int k) {
    return tokens > 0 && tokens <= ((int64_t)1 << 40) && n > 0 && k > 0 && n <= (1 << 16) && k <= (1 << 16) && n % 8 == 0 && k % 8 == 0;
}

size_t fb_weight_grad_workspace_bytes(int64_t tokens, int n, int k, int with_bias) {
    return weight_grad_sizes(tokens, n, k) ? fb::wgrad_workspace(tokens, n, k, with_bias != 0) : 0;
}

int fb_weight_grad_recommended(int64_t tokens, int n, int k) {
    return weight_grad_sizes(tokens, n, k) && fb::wgrad_recommended(tokens, n, k) ? 1 : 0;
}

int fb_weight_grad(const void *dy, int64_t ldy, const void *x, int64_t ldx, void *dw, void *db, float *scratch, int dtype, int64_t tokens,
                   int n, int k, void *stream) {
    fb::api_clear_error();
    if (!dy || !x || !dw || !scratch) return fb::api_fail(FB_ERR_NULL, "fb_weight_grad: null pointer");
    if (dtype != FB_F16 && dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (!weight_grad_sizes(tokens, n, k))
        return fb::api_fail(FB_ERR_SHAPE, "fb_weight_grad: tokens must be positive, n and k multiples of 8 up to 65536");
    if (ldy < n || ldx < k || ldy % 8 != 0 || ldx % 8 != 0 || ldy >= (1 << 24) || ldx >= (1 << 24))
        return fb::api_fail(FB_ERR_STRIDE, "fb_weight_grad: row strides must be multiples of 8 below 2^24 and hold a row");
    for (const void *p : {dy, x, static_cast<const void *>(dw), static_cast<const void *>(scratch)})
        if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return fb::api_fail(FB_ERR_STRIDE, "fb_weight_grad: tensors must be 16-byte aligned");
    return launched(fb::launch_wgrad(dy, ldy, x, ldx, dw, db, scratch, tokens, n, k, dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                    "fb_weight_grad");
}

static bool project_sizes(int64_t tokens, int k, const int *n, int count) {
    if (!n || count < 1 || count > 3 || tokens <= 0 || tokens > (1 << 24) || k <= 0 || k > (1 << 16) || k % 64 != 0) return false;
    for (int i = 0; i < count; ++i)
        if (n[i] <= 0 || n[i] > (1 << 16) || n[i] % 8 != 0) return false;
    return true;
}

int fb_project_recommended(int64_t tokens, int k, const int *n, int count) {
    return project_sizes(tokens, k, n, count) && fb::project_recommended(tokens, k, n, count) ? 1 : 0;
}

int fb_project(const void *x, int64_t ldx, const void *const *w, void *const *y, const int *n, int count, int dtype, int64_t tokens, int k,
               void *stream) {
    fb::api_clear_error();
    if (!x || !w || !y || !n) return fb::api_fail(FB_ERR_NULL, "fb_project: null pointer");
    if (dtype != FB_F16 && dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (!project_sizes(tokens, k, n, count))
        return fb::api_fail(FB_ERR_SHAPE, "fb_project: one to three weights, tokens up to 2^24, k a multiple of 64 and n of 8, both up to 65536");
    if (ldx < k || ldx % 8 != 0 || ldx >= (1 << 22))
        return fb::api_fail(FB_ERR_STRIDE, "fb_project: the row stride must be a multiple of 8 below 2^22 and hold a row");
    bool aligned = reinterpret_cast<uintptr_t>(x) % 16 == 0;
    for (int i = 0; i < count; ++i) {
        if (!w[i] || !y[i]) return fb::api_fail(FB_ERR_NULL, "fb_project: null pointer");
        aligned = aligned && reinterpret_cast<uintptr_t>(w[i]) % 16 == 0 && reinterpret_cast<uintptr_t>(y[i]) % 16 == 0;
    }
    if (!aligned) return fb::api_fail(FB_ERR_STRIDE, "fb_project: tensors must be 16-byte aligned");
    return launched(fb::launch_project(x, ldx, w, y, n, count, tokens, k, dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_project");
}

int fb_linear_recommended(int64_t tokens, int n, int k) { return project_sizes(tokens, k, &n, 1) && fb::linear_recommended(tokens, n, k) ? 1 : 0; }

int fb_linear(const void *x, int64_t ldx, const void *w, const void *b, void *y, int dtype, int64_t tokens, int n, int k, void *stream) {
    fb::api_clear_error();
    if (!x || !w || !y) return fb::api_fail(FB_ERR_NULL, "fb_linear: null pointer");
    if (dtype != FB_F16 && dtype != FB_BF16) return fb::api_fail(FB_ERR_DTYPE, "only fp16 and bf16 are supported");
    if (!project_sizes(tokens, k, &n, 1))
        return fb::api_fail(FB_ERR_SHAPE, "fb_linear: tokens up to 2^24, k a multiple of 64 and n of 8, both up to 65536");
    if (ldx < k || ldx % 8 != 0 || ldx >= (1 << 22))
        return fb::api_fail(FB_ERR_STRIDE, "fb_linear: the row stride must be a multiple of 8 below 2^22 and hold a row");
    for (const void *p : {x, w, static_cast<const void *>(y)})
        if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return fb::api_fail(FB_ERR_STRIDE, "fb_linear: tensors must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(b) % 4 != 0) return fb::api_fail(FB_ERR_STRIDE, "fb_linear: the bias must be 4-byte aligned");
    return launched(fb::launch_linear(x, ldx, w, b, y, tokens, n, k, dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_linear");
}

int fb_transpose(const void *in, void *out, int rows, int cols, void *stream) {
    fb::api_clear_error();
    if (!in || !out) return fb::api_fail(FB_ERR_NULL, "fb_transpose: null pointer");
    if (rows <= 0 || cols <= 0 || rows > (1 << 16) || cols > (1 << 16) || rows % 64 != 0 || cols % 64 != 0)
        return fb::api_fail(FB_ERR_SHAPE, "fb_transpose: rows and columns must be multiples of 64 up to 65536");
    for (const void *p : {in, static_cast<const void *>(out)})
        if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return fb::api_fail(FB_ERR_STRIDE, "fb_transpose: matrices must be 16-byte aligned");
    return launched(fb::launch_transpose(in, out, rows, cols, static_cast<hipStream_t>(stream)), "fb_transpose");
}

int fb_bwd_static(const fb_params *p, void *stream) {
    // fb_bwd with the scratch buffer taken from the library's own static device array instead of
    // fb_params.delta (which is ignored): no allocation, here or in anything it calls.
    fb::api_clear_error();
    if (!p) return fb::api_fail(FB_ERR_NULL, "params: null pointer");
    if (!fb::known_size(p)) return fb::api_fail(FB_ERR_ABI, "fb_params.size does not match this library");
    const size_t need = fb_bwd_workspace_bytes(p);
    if (need == 0) return fb::api_fail(FB_ERR_SHAPE, "B, H, Lq, Lk must be positive");
    if (need > (size_t)FB_STATIC_SCRATCH_BYTES)
        return fb::api_fail(FB_ERR_SHAPE, "fb_bwd_static: B * H * Lq exceeds the static scratch buffer (FB_STATIC_SCRATCH_BYTES); use fb_bwd");
    hipError_t e = hipSuccess;
    void *ptr = static_scratch(&e);
    if (!ptr) return launched(e, "fb_bwd_static (hipGetSymbolAddress)");
    fb_params q;
    std::memset(&q, 0, sizeof(q));
    std::memcpy(&q, p, p->size); // (which may be smaller)
    q.delta = static_cast<float *>(ptr);
    return fb_bwd(&q, stream);
}

int fb_bwd(const fb_params *p, void *stream) {
    // Two launches: the dq kernel computes delta for its own queries on the way (each query belongs
    // to exactly one of its workgroups) and leaves the statistics in the scratch buffer for the
    // dk/dv kernel.  The three phases above stay callable one by one.
    const int rc = fb_check(p, 1);
    if (rc) return rc;
    fb::BwdArgs a = bwd_args(p);
    if (fb::ring_backward(a)) // ... without factor gradients
        return launched(fb::launch_bwd_ring(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_bwd (ring)");
    if (fb::window_backward(a)) // whole sequences of at most 256 positions: one workgroup per (batch, head), one launch
        return launched(fb::launch_bwd_win(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_bwd (window)");
    const bool general_mix = p->dtype == FB_BF16 ? fb::mixed_general_backward<fb::BF16>(a) : fb::mixed_general_backward<fb::F16>(a);
    if (fb::mixed_backward(a) || general_mix) {
        // small grids of the streamlined kernels: the preprocess step, then one launch that holds the dq and
        // the dk/dv workgroups side by side (same bits as the two launches)
        const int rc1 = launched(fb::launch_bwd_preprocess(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                                 "fb_bwd_preprocess");
        if (rc1) return rc1;
        return launched((general_mix ? fb::launch_bwd_both_general : fb::launch_bwd_both)(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)),
                        "fb_bwd (dq + dk/dv)");
    }
    a.stats_here = 1;
    const int rc2 = launched(fb::launch_bwd_dq(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_bwd_dq");
    if (rc2) return rc2;
    a.stats_here = 0;
    return launched(fb::launch_bwd_dkv(a, p->dtype == FB_BF16, static_cast<hipStream_t>(stream)), "fb_bwd_dkv");
}

} // extern "C"
