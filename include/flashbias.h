/*
 * flashbias.h -- C ABI of the MI355X (gfx950) FlashBias attention library.
 *
 * The library is the device side of the reference's operator
 *     flash_bias_func(q, k, v, q_bias, k_bias, mask, causal, softmax_scale)
 * (flash_bias/flash_bias_triton.py:1345-1405).  Each entry point below names the reference
 * function it replaces.  Conventions shared by all of them:
 *
 *   - Nothing here allocates or frees device memory: every buffer, including scratch
 *     (lse, delta), is owned by the caller, as in the reference where
 *     torch allocates o/lse/tmp/delta/dq_accum (flash_bias_triton.py:1145-1148, :1212-1219).
 *   - Launches are asynchronous on the given hipStream_t (passed as void*); no autotuning side
 *     effects.  The only process-wide state are write-once caches (compute units per device,
 *     per-kernel occupancy and LDS limit; atomics, safe under concurrent first calls) and the
 *     scratch array of fb_bwd_static.
 *   - Return value: FB_OK (0) or a negative fb_status; fb_last_error() gives the text of the
 *     last failure on the calling thread.  No C++ exception crosses the boundary.
 *   - Tensors use the reference layout (batch, seq, heads, channels) with the channel
 *     dimension contiguous (stride 1: the ABI has no channel stride, a caller with another one
 *     must make the tensor contiguous first, as the reference does, :1357-1360); batch / head /
 *     seq are addressed through element strides, the way the Triton launchers pass them
 *     (flash_bias_triton.py:1163-1177).  Sequence strides of 2^24 elements or more are correct
 *     but take slower instantiations (the fast loaders keep a tile row's offset in 32 bits).
 */
#ifndef FLASHBIAS_H
#define FLASHBIAS_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* 4: mask_batches at the end of fb_params (blocks of version 3 are accepted), fb_alibi_factors and fb_cosine_* */
#define FB_VERSION 4
#define FB_MAX_HEADDIM 128 /* flash_bias_triton.py:1106 */
#define FB_MAX_RANK 128
/* Size of the library-owned scratch buffer used by fb_bwd_static (one copy per GPU, held until the
 * process ends): enough for B * H * Lq <= 1398101 query rows (24 bytes each). */
#define FB_STATIC_SCRATCH_BYTES (32u << 20)

typedef enum fb_status {
    FB_OK = 0,
    FB_ERR_NULL = -1,       /* required pointer missing */
    FB_ERR_SHAPE = -2,      /* non-positive size, d > 128, r > 128, B * H * ceil(L / 32) >= 2^31 */
    FB_ERR_DTYPE = -3,      /* only fp16 / bf16 inputs (flash_bias_triton.py:1108) */
    FB_ERR_STRIDE = -4,     /* stride would alias gradient rows / negative stride */
    FB_ERR_MASK = -5,       /* bad mask type / dtype */
    FB_ERR_RESERVED = -6,
    FB_ERR_ABI = -7,        /* fb_params.size is none that this library knows */
    FB_ERR_LAUNCH = -8,     /* HIP reported a launch error */
    FB_ERR_SCALE = -9       /* softmax scale not finite or zero (negative scales are accepted) */
} fb_status;

typedef enum fb_dtype { FB_F16 = 0, FB_BF16 = 1, FB_F32 = 2 /* mask only */ } fb_dtype;

/* flash_bias_triton.py:1112-1123 */
typedef enum fb_mask_type { FB_MASK_NONE = 0, FB_MASK_VECTOR = 1, FB_MASK_MATRIX = 2 } fb_mask_type;

/* A (batch, seq, heads, channels) tensor with contiguous channels.  Strides are in elements.
 * For the mask, which is (batch, heads, Lq|1, Lk), stride_s is the stride of the query row
 * (0 for the vector type) and stride_b / stride_h may be 0 (broadcast). */
typedef struct fb_tensor {
    void *ptr;
    int64_t stride_b, stride_h, stride_s;
} fb_tensor;

typedef struct fb_params {
    uint32_t size; /* sizeof(fb_params) as seen by the caller; FB_PARAMS_SIZE_3, the block of version 3, is taken too */
    int32_t dtype; /* fb_dtype of q, k, v, factors, o and all gradients */
    int32_t B, H, Lq, Lk;
    int32_t d;     /* head dim, 1..128 */
    int32_t r;     /* bias rank, 0 = no factors (plain attention, flash_bias_triton.py:1359) */
    int32_t causal;     /* top-left aligned: key j visible from query i iff j <= i (:262) */
    int32_t mask_type;  /* fb_mask_type */
    int32_t mask_dtype; /* dtype or FB_F32 (:1115) */
    float scale;        /* softmax scale, applied to q k^T only, never to the bias (:248) */

    fb_tensor q, k, v;        /* in */
    fb_tensor q_bias, k_bias; /* in; stride_b / stride_h = 0 broadcasts (:1135-1136) */
    fb_tensor mask;           /* in, additive, no gradient (:1371) */
    fb_tensor o;              /* fwd: out; bwd: in */
    float *lse;               /* (B, H, Lq) fp32, natural log; fwd: out; bwd: in (:323) */

    fb_tensor dout;             /* bwd in: upstream gradient of o */
    fb_tensor dq, dk, dv;       /* bwd out */
    fb_tensor dq_bias, dk_bias; /* bwd out, full (B, L, H, r) shape: the caller reduces over
                                   broadcast dims (but see bias_grad_group).  Both pointers NULL: the
                                   factor gradients are not wanted (constant factors) and are neither
                                   stored nor, in the streamlined kernels, computed; the reference
                                   always computes them (flash_bias_triton.py:718-719, :725-817) */
    float *delta;               /* backward scratch of fb_bwd_workspace_bytes() bytes, 16-byte aligned, written by the
                                   backward: -delta and lse * log2(e) per query row, as fp32 and as 16-bit parts */
    int32_t bias_grad_group;    /* 0 or 1: as above.  g > 1, for factors that the batch shares (stride_b = 0, the
                                   window attention of swin_transformer_v2.py:178-203): dq_bias and dk_bias have
                                   ceil(B / g) batch rows and row i receives the sum of the gradients of batch
                                   entries [i g, (i + 1) g), accumulated in fp32 inside the kernels and rounded
                                   once; the caller reduces the remaining rows.  (The reference accumulates the factor
                                   gradients with atomic adds into fp32 buffers laid out like the factors
                                   themselves, flash_bias_triton.py:1219-1231, :1342.) */
    int32_t reserved0;          /* not read (padding at the end of version 3's block) */
    int32_t mask_batches;       /* 0: the mask has B batch entries, or one (stride_b = 0).  n > 0: it has n, and batch
                                   entry b takes b % n: the masks of a shifted-window block, one per window of an image,
                                   which the reference repeats over the images (swin_transformer_v2.py:190-203) */
    int32_t reserved1[3];       /* not read */
} fb_params;

/* The block of version 3 ends before mask_batches, which is then 0. */
#define FB_PARAMS_SIZE_3 offsetof(fb_params, mask_batches)

/* Library / ABI version. */
int fb_version(void);

/* Optional set-up for the current device: looks up the address of the static scratch array that
 * fb_bwd_static uses (one hipGetSymbolAddress per device, cached), so that no later call has to.
 * fb_bwd_static does the same on its first call on a device; a caller that wants that first call
 * inside a HIP graph capture calls fb_init() (or fb_bwd_static once, eagerly) on the device
 * beforehand, because a symbol lookup is not a stream operation and must not happen while a
 * stream is capturing.  Launches nothing, allocates nothing.  No counterpart in the reference. */
int fb_init(void);

/* Text of the last error on this thread ("" if none). */
const char *fb_last_error(void);

/* Argument checks of _flash_attn_forward / _flash_attn_backward
 * (flash_bias_triton.py:1102-1129, :1201-1225) without touching the GPU.
 * pass: 0 = forward, 1 = backward. */
int fb_check(const fb_params *p, int pass);

/* The bias_grad_group this library recommends for a backward call: 1 unless both factors are shared by
 * the batch (stride_b = 0) and the call is a large batch of short sequences (the window attention of
 * swin_transformer_v2.py:178-203), where writing the full-shape factor gradients and summing them
 * afterwards costs more than the attention itself saves; then the largest of 8, 4, 2 (32, 16, ... for whole
 * sequences of at most 256 positions at head dim 32, which one workgroup per batch entry and head serves) that still
 * leaves every compute unit several workgroups.  Reads the sizes, the causal flag, the element types, the mask type and the factors' strides only.
 * No counterpart in the reference. */
int fb_suggest_bias_grad_group(const fb_params *p);

/* Bytes of the backward's scratch buffer fb_params.delta for these sizes (24 per query row: two
 * floats and one 16-byte chunk of 16-bit parts, the second array starting on a 16-byte boundary;
 * the reference allocates delta, dq_accum and dq_bias_accum itself, flash_bias_triton.py:1212-1219).
 * Only B, H and Lq are read; returns 0 for a null pointer or non-positive sizes. */
size_t fb_bwd_workspace_bytes(const fb_params *p);

/* Replaces _flash_attn_forward + _fwd_kernel (flash_bias_triton.py:1100-1194, :62-355):
 * o = softmax(scale q k^T + q_bias k_bias^T + mask) v and lse. */
int fb_fwd(const fb_params *p, void *stream);

/* Replaces _flash_attn_backward (flash_bias_triton.py:1197-1342).  Two launches on the stream: the
 * query-stationary kernel (dq, dq_bias), which also forms delta = rowsum(o * dout) for its own
 * queries and leaves -delta and lse * log2(e) in the scratch buffer, then the key-stationary kernel
 * (dk, dv, dk_bias) that reads them.  (On grids that would give each of these kernels at most one
 * workgroup per compute unit: the preprocess phase, then a single launch that holds the workgroups of
 * both kernels side by side.)  The results of these are bit-identical to the three phases below
 * called one by one.  Whole sequences of at most 256 positions (head dim 32, rank a multiple of 8 up to
 * 32, aligned tensors, no causal or fp32 mask, at least one (batch, head) pair per compute unit: the
 * window attention of swin_transformer_v2.py:178-203) take a single launch instead in which one
 * workgroup forms delta and the gradients of a (batch, head) pair, dq summed inside the workgroup:
 * without factor gradients at ranks up to 16 from four pairs per compute unit on (gradients and the
 * rows of a matrix mask in aligned 16-byte chunks), else with more than 128 positions on one side (64
 * under a vector mask).  Such a launch leaves the scratch buffer untouched and its results equal the
 * phases' up to the rounding of other summation orders.  Unlike the reference there is no
 * fp32 dq_accum buffer, no atomics and no final cast on any of these paths (:1212-1219, :1340-1342):
 * dq and dq_bias are accumulated in registers (or, for windows, in a fixed order through LDS) and
 * written once, so every gradient is bit-reproducible. */
int fb_bwd(const fb_params *p, void *stream);

/* fb_bwd for callers that cannot allocate device memory (code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  No counterpart in the reference, whose
 * backward allocates its scratch through torch (flash_bias_triton.py:1212-1219).  Same inputs,
 * outputs and results as fb_bwd, except that fb_params.delta is ignored: the scratch lives in a
 * static device array of FB_STATIC_SCRATCH_BYTES inside the library.  Neither this call nor
 * anything it calls allocates or frees memory.  Returns FB_ERR_SHAPE when
 * fb_bwd_workspace_bytes(p) exceeds FB_STATIC_SCRATCH_BYTES.  All calls on one GPU share that
 * GPU's array: calls that overlap in time on one GPU (two streams, two threads) race; calls
 * ordered on one stream are safe.  Nothing in the array has to be cleared between calls.  The
 * first call on a device looks the array's address up (see fb_init): make it, or fb_init(), outside
 * graph capture. */
int fb_bwd_static(const fb_params *p, void *stream);

/* The last step of the backward for factors that every batch entry shares: the kernels write such
 * a factor's gradient in full (B, L, H, r) shape, and this sums it over the batch:
 * out[j] = sum_b full[b * batch_stride + j] for j < n = L * H * r, accumulated in fp32 in a fixed
 * order (bit-reproducible), written in the input dtype or (out_dtype = FB_F32) in fp32.  The
 * reference has no such step: it hands the kernels the un-expanded tensors with expanded strides
 * (flash_bias_triton.py:1227-1231), so every batch entry overwrites the same gradient rows.
 * n and batch_stride must be multiples of 8 elements, full 16-byte aligned (FB_ERR_STRIDE else). */
int fb_sum_over_batch(const void *full, void *out, int dtype, int out_dtype, int64_t B, int64_t n,
                      int64_t batch_stride, void *stream);

/* Factors of a rank that is no multiple of 8 (ALiBi: 2, a distance bias in three dimensions: 5) have rows the
 * kernels' 16-byte loads cannot take; their owner, or the operator on every call, pads them with zero columns,
 * which change nothing in q_bias k_bias^T.  out[row][c] = c < min(r_in, r_out) ? in[row][c] : 0 for `rows`
 * contiguous rows of 16-bit elements (either dtype): r_out > r_in pads, r_out < r_in takes the original columns of
 * a gradient back out.  One launch.  The reference pads inside its kernels instead (BLOCK_RANKDIM, the next power
 * of two of at least 16, with masked loads: flash_bias_triton.py:1137, :195-200). */
int fb_resize_rank(const void *in, void *out, int64_t rows, int r_in, int r_out, void *stream);

/* The same of two tensors of one rank, the two factors of a call, in one launch. */
int fb_resize_ranks(const void *q_in, void *q_out, int64_t q_rows, const void *k_in, void *k_out, int64_t k_rows,
                    int r_in, int r_out, void *stream);

/* The exact ALiBi bias -m_h (i - j) as factors of rank 4, zero-padded to `r` columns (positions below 65536 in two
 * 8-bit digits, i = 256 a + b, so that every column is a whole number or a slope in 16 bits):
 *     q_bias[i] = [a_i, b_i, 256 m, m, 0 ...],   k_bias[j] = [-256 m, -m, a_j, b_j, 0 ...],
 * both (L, H, r) contiguous and 16-byte aligned, r a multiple of 8, m_h = 2^(-8 (h + 1) / H) rounded to the dtype;
 * reference_sign: +m_h (i - j), what the reference's module builds (attention_with_alibi_bias.py:44-52).  One launch. */
int fb_alibi_factors(void *q_bias, void *k_bias, int dtype, int Lq, int Lk, int H, int r, int reference_sign, void *stream);

/* The backward in three phases, exported so that a harness can time them separately (call them in
 * this order: the two main kernels read what the preprocess wrote).
 *   fb_bwd_preprocess: delta = rowsum(o * dout)       (_bwd_preprocess_do_o_dot, :358-400); fills the
 *                      scratch with -delta (first B*H*Lq floats), lse * log2(e) (next B*H*Lq) and, from the
 *                      next 16-byte boundary on, both once more per query row as three 16-bit parts each
 *                      (what the streamlined dk/dv kernel feeds to its MFMAs; written only for the calls
 *                      that kernel takes: aligned, unmasked, head dim 32, rank 8 or 0)
 *   fb_bwd_dkv:        recompute P from lse; dk, dv, dk_bias, one workgroup per key tile
 *                      (_bwd_kernel / _bwd_kernel_one_col_block, :450-1097, minus dq)
 *   fb_bwd_dq:         recompute P from lse; dq, dq_bias, one workgroup per query tile
 *                      (the dq / dq_bias updates of :725-817) */
int fb_bwd_preprocess(const fb_params *p, void *stream);
int fb_bwd_dkv(const fb_params *p, void *stream);
int fb_bwd_dq(const fb_params *p, void *stream);

/* The elementwise part of a cosine-attention window block around the operator
 * (swin_transformer_v2.py:155-207: normalize(q) * exp(min(logit_scale, 4.6052)), normalize(k)), one pass over the
 * packed projection in each direction.  qkv and dqkv are (tokens, 3, H, d), contiguous and 16-byte aligned;
 * d is 8, 16, 32, 64 or 128. */
typedef struct fb_cosine {
    uint32_t size;        /* sizeof(fb_cosine) as seen by the caller */
    int32_t dtype;        /* FB_F16 or FB_BF16: q, k, v and their gradients */
    int32_t in_dtype;     /* fb_dtype of qkv and dqkv */
    int32_t scale_dtype;  /* fb_dtype of logit_scale and its gradient */
    int32_t H, d;
    int64_t tokens;
    const void *qkv;         /* in */
    const void *logit_scale; /* in, (H) */
    void *q, *k, *v;         /* fwd out, (tokens, H, d) contiguous; v NULL: not wanted (it can be read from qkv in place) */
    const void *dq, *dk, *dv; /* bwd in, rows of H d elements; dv NULL: already in dqkv */
    int64_t grad_stride;     /* elements from one token's dq (dk, dv) to the next's.  dq and dk may lie where the
                                gradient of their part of dqkv goes (then in_dtype = dtype, grad_stride = 3 H d) */
    void *dqkv;              /* bwd out */
    void *dlogit_scale;      /* bwd out, (H) */
    float *partial;          /* bwd scratch of fb_cosine_workspace_bytes() bytes */
    int32_t fp32;            /* 0: norm, quotient, exponential and product are rounded to the type of their tensors one after
                                the other, as tensor operations do; else they stay in fp32 and only the results are
                                rounded, as under autocast.  (A block whose size ends before this field is accepted: 0.) */
    int32_t reserved;        /* 0 */
} fb_cosine;

size_t fb_cosine_workspace_bytes(const fb_cosine *p);
int fb_cosine_fwd(const fb_cosine *p, void *stream);
int fb_cosine_bwd(const fb_cosine *p, void *stream);

/* The attention of such a block with the normalisation inside the attention kernels: q, k, v (and dq, dk, dv) of `p` are the
 * parts of the packed projection c->qkv (c->dqkv) itself, o and lse those of the attention on the normalised rows, scale 1, no
 * factor gradients.  The backward reads the projection again, writes the projection's gradient and dlogit_scale, and takes
 * c->partial of fb_window_workspace_bytes() bytes; p->delta is not used, and neither are the other pointers of `c`.  The bits are those of
 * fb_cosine_fwd, the forward and the backward for windows (which fb_fwd and fb_bwd use on grids that fill the chip) and fb_cosine_bwd one after the other, but for
 * dlogit_scale (another order of the same sum) and, in fp16, for some of the gradients of q and k: fb_cosine_bwd adds up products in pairs there, whose
 * fp32 roundings differ (about 2^-20 of a row's largest value before the result is rounded, one element in 2^12).
 * fb_window_ready (pass: 0 = forward, 1 = backward): 1 for the calls these take: head dim 32, at most 256 positions, rank up to
 * 16, one 16-bit type, fp32 = 0, aligned tensors, no mask or a matrix mask of 16-byte chunks; the others return FB_ERR_SHAPE.
 * It leaves fb_last_error as it was. */
int fb_window_ready(const fb_params *p, const fb_cosine *c, int pass);
size_t fb_window_workspace_bytes(const fb_params *p);
int fb_window_fwd(const fb_params *p, const fb_cosine *c, void *stream);
int fb_window_bwd(const fb_params *p, const fb_cosine *c, void *stream);

/* Weight and bias gradient of a projection y = x w^T + b, the products around the attention of a block
 * (swin_transformer_v2.py:155-207), for many tokens and a small weight: dw (n, k) = dy^T x and db (n) = the column sums
 * of dy, both contiguous in the input dtype, accumulated in fp32 in a fixed order and rounded once; db NULL: not wanted.
 * dy (tokens, n) and x (tokens, k) have contiguous rows at strides ldy, ldx (elements).  n, k, ldy and ldx are multiples
 * of 8, dy, x, dw and scratch 16-byte aligned; scratch: fb_weight_grad_workspace_bytes() bytes.  Two launches.
 * fb_weight_grad_recommended: 1 where this was measured ahead of the vendor library's product of the same shape. */
size_t fb_weight_grad_workspace_bytes(int64_t tokens, int n, int k, int with_bias);
int fb_weight_grad_recommended(int64_t tokens, int n, int k);
int fb_weight_grad(const void *dy, int64_t ldy, const void *x, int64_t ldx, void *dw, void *db, float *scratch, int dtype, int64_t tokens,
                   int n, int k, void *stream);

/* Up to three projections of one input in one launch (the q, k and v projections of an attention block,
 * 1_Language_Model/attention_with_alibi_bias.py:26-28): y[i] (tokens, n[i]) = x (tokens, k) w[i]^T in the input dtype,
 * accumulated in fp32 and rounded once.  w[i] (n[i], k) and y[i] are contiguous, x has contiguous rows at a stride of ldx elements.
 * k is a multiple of 64, n[i] and ldx of 8, ldx below 2^22, n[i] and k at most 65536, tokens at most 2^24; all 16-byte aligned.
 * fb_project_recommended: 1 where this was measured ahead of the vendor library's products of the same shape. */
int fb_project_recommended(int64_t tokens, int k, const int *n, int count);
int fb_project(const void *x, int64_t ldx, const void *const *w, void *const *y, const int *n, int count, int dtype, int64_t tokens,
               int k, void *stream);

/* A projection of many tokens (the layers of a window block, swin_transformer_v2.py:155-207): y (tokens, n) = x (tokens, k) w^T + b
 * in the input dtype, accumulated in fp32 and rounded once; b (n) NULL: none.  w (n, k) and y are contiguous, x has contiguous rows at
 * a stride of ldx elements.  k is a multiple of 64, n and ldx of 8, ldx below 2^22, n and k at most 65536, tokens at most 2^24; x, w
 * and y 16-byte aligned, b 4-byte aligned.
 * fb_linear_recommended: 1 where this was measured ahead of the vendor library's product of the same shape. */
int fb_linear_recommended(int64_t tokens, int n, int k);
int fb_linear(const void *x, int64_t ldx, const void *w, const void *b, void *y, int dtype, int64_t tokens, int n, int k, void *stream);
/* out (cols, rows) = in (rows, cols)^T of 16-bit elements, both contiguous and 16-byte aligned, rows and cols multiples of 64 up to 65536: the
 * weight of the product above where it contracts the other way (an input's gradient dy w). */
int fb_transpose(const void *in, void *out, int rows, int cols, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* FLASHBIAS_H */
