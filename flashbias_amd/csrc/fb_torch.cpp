// The operator's autograd function in C++: what flashbias_amd/interface.py does per call (argument
// checks of _flash_attn_forward / _flash_attn_backward, flash_bias/flash_bias_triton.py:1100-1143 and
// :1197-1231, the parameter block, the output allocations, the launch on torch's current stream, the
// reduction of broadcast factors' gradients) without the interpreter in the way: at sequence lengths
// of a few thousand the kernels of a forward + backward take 50-150 us, which is what the Python
// path costs on the host.  Everything that touches the GPU still goes through the C ABI of
// include/flashbias.h; torch provides memory, the stream and the autograd graph.
//
// Expects kernel-ready inputs (flash_bias_func in interface.py prepares the rare cases with ordinary
// differentiable tensor operations before calling in): q, k, v (B, L, H, d); factors (B|1, L, H|1, r)
// or none; additive mask (B|1, H|1, 1|Lq, Lk) or none.
#include <torch/extension.h>

#include <ATen/FuncTorchTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cmath>
#include <cstring>

#include "flashbias.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::tensor_list;

fb_tensor t4(const Tensor &x) { return fb_tensor{x.data_ptr(), x.stride(0), x.stride(2), x.stride(1)}; }

Tensor channel_contiguous(const Tensor &x) { return x.stride(-1) == 1 ? x : x.contiguous(); }

int dtype_code(c10::ScalarType t) {
    if (t == torch::kFloat16) return FB_F16;
    if (t == torch::kBFloat16) return FB_BF16;
    if (t == torch::kFloat32) return FB_F32;
    TORCH_CHECK(false, "unsupported dtype ", t);
}

void check(int status) { TORCH_CHECK(status == FB_OK, "flashbias status ", status, ": ", fb_last_error()); }

// A contiguous tensor straight from the caching allocator: a backward makes six of them, and the dispatcher's way
// to the same call takes a microsecond longer each.
Tensor fresh(at::IntArrayRef sizes, c10::ScalarType type, c10::Device device) {
    return Tensor(at::detail::empty_cuda(sizes, type, device, c10::nullopt));
}
Tensor fresh_like(const Tensor &x) { return x.is_contiguous() ? fresh(x.sizes(), x.scalar_type(), x.device()) : torch::empty_like(x); }

// The stride of a dimension that may be 1 where `n` is wanted (broadcast: stride 0).
int64_t broadcast_stride(const Tensor &x, int dim, int64_t n, const char *what) {
    if (x.size(dim) == n) return x.stride(dim);
    TORCH_CHECK(x.size(dim) == 1, what, ": dimension ", dim, " must be 1 or ", n, ", got ", x.size(dim));
    return 0;
}
fb_tensor factor(const Tensor &x, int64_t B, int64_t L, int64_t H, const char *what) {
    return fb_tensor{x.data_ptr(), broadcast_stride(x, 0, B, what), broadcast_stride(x, 2, H, what), broadcast_stride(x, 1, L, what)};
}

// What one call of the operator is given.  `mask_batches`: the mask's batch entries where they repeat (else 0).
struct Call {
    Tensor q, k, v, qb, kb, mask;
    bool causal;
    double scale;
    int mask_batches;
};

// The parameter block shared by forward and backward.
fb_params block(const Call &c) {
    const Tensor &q = c.q, &k = c.k, &v = c.v, &qb = c.qb, &kb = c.kb, &mask = c.mask;
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k, v must be (batch, seqlen, nheads, headdim)");
    const int64_t B = q.size(0), Lq = q.size(1), H = q.size(2), d = q.size(3), Lk = k.size(1);
    TORCH_CHECK(k.size(0) == B && k.size(2) == H && k.size(3) == d && v.sizes() == k.sizes(), "k, v must be (batch, seqlen_k, nheads, headdim)");
    TORCH_CHECK(d <= FB_MAX_HEADDIM, "FlashBias only supports head dimensions up to 128");
    TORCH_CHECK(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(), "All tensors must have the same type");
    TORCH_CHECK(q.scalar_type() == torch::kFloat16 || q.scalar_type() == torch::kBFloat16, "Only support fp16 and bf16");
    TORCH_CHECK(q.is_cuda() && k.is_cuda() && v.is_cuda(), "q, k, v must be on the GPU");
    fb_params p;
    std::memset(&p, 0, sizeof(p));
    p.size = sizeof(p);
    p.dtype = dtype_code(q.scalar_type());
    p.B = (int32_t)B; p.H = (int32_t)H; p.Lq = (int32_t)Lq; p.Lk = (int32_t)Lk; p.d = (int32_t)d;
    p.causal = c.causal ? 1 : 0;
    p.scale = (float)c.scale;
    p.q = t4(q); p.k = t4(k); p.v = t4(v);
    if (qb.defined()) {
        TORCH_CHECK(kb.defined() && qb.scalar_type() == q.scalar_type() && kb.scalar_type() == q.scalar_type() && qb.is_cuda() &&
                        kb.is_cuda() && qb.dim() == 4 && kb.dim() == 4 && qb.size(3) == kb.size(3),
                    "q_bias, k_bias must be GPU tensors of the input dtype and one rank");
        p.r = (int32_t)qb.size(3);
        // stride-0 broadcast over batch / heads (flash_bias_triton.py:1135-1136)
        p.q_bias = factor(qb, B, Lq, H, "q_bias");
        p.k_bias = factor(kb, B, Lk, H, "k_bias");
    }
    if (mask.defined()) {
        TORCH_CHECK(mask.dim() == 4 && mask.is_cuda() && (mask.scalar_type() == q.scalar_type() || mask.scalar_type() == torch::kFloat32),
                    "mask must be a 4-d GPU tensor of the input dtype or fp32");
        if (mask.size(2) == 1 && mask.size(3) == Lk)
            p.mask_type = FB_MASK_VECTOR;
        else if (mask.size(2) == Lq && mask.size(3) == Lk)
            p.mask_type = FB_MASK_MATRIX;
        else
            TORCH_CHECK(false, "Last 2 dimensions of mask must be (1, seqlen_k) or (seqlen_q, seqlen_k)");
        p.mask = fb_tensor{mask.data_ptr(), c.mask_batches ? mask.stride(0) : broadcast_stride(mask, 0, B, "mask"),
                           broadcast_stride(mask, 1, H, "mask"), mask.size(2) == Lq ? mask.stride(2) : 0};
        p.mask_dtype = dtype_code(mask.scalar_type());
        p.mask_batches = c.mask_batches;
    }
    return p;
}

hipStream_t stream_of(const Tensor &x) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream(); }

// The gradient of `ref` from the full (B, L, H, r) gradient the kernels wrote: summed over the dims in
// which `ref` was broadcast, in fp32 (over the batch by the library's streaming kernel).
Tensor reduce_like(Tensor full, const Tensor &ref, hipStream_t stream) {
    bool over_batch = ref.size(0) == 1 && full.size(0) != 1;
    const bool over_heads = ref.size(2) == 1 && full.size(2) != 1;
    const int64_t n = full.size(1) * full.size(2) * full.size(3);
    if (over_batch && full.is_contiguous() && n % 8 == 0) {
        Tensor out = torch::empty({1, full.size(1), full.size(2), full.size(3)},
                                  full.options().dtype(over_heads ? torch::kFloat32 : full.scalar_type()));
        check(fb_sum_over_batch(full.data_ptr(), out.data_ptr(), dtype_code(full.scalar_type()), dtype_code(out.scalar_type()),
                                full.size(0), n, n, stream));
        full = out;
        over_batch = false;
    }
    if (over_batch || over_heads) {
        std::vector<int64_t> dims;
        if (over_batch) dims.push_back(0);
        if (over_heads) dims.push_back(2);
        full = full.sum(dims, /*keepdim=*/true, torch::kFloat32);
    }
    if (full.scalar_type() != ref.scalar_type()) full = full.to(ref.scalar_type());
    return full.is_contiguous() ? full : full.contiguous();
}

// o and lse of a call.
std::pair<Tensor, Tensor> attend(const Call &c) {
    fb_params p = block(c);
    Tensor o = fresh_like(c.q);
    Tensor lse = fresh({p.B, p.H, p.Lq}, torch::kFloat32, c.q.device());
    p.o = t4(o);
    p.lse = lse.data_ptr<float>();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(c.q.device()); // (torch on ROCm presents its devices as "cuda")
    check(fb_fwd(&p, stream_of(c.q)));
    return {o, lse};
}

// dq, dk, dv into the tensors given (any strides with contiguous channels); returns the factors' gradients,
// undefined where nobody asks for them (constant factors; the library then skips them).
std::pair<Tensor, Tensor> attend_backward(const Call &c, const Tensor &o, const Tensor &lse, const Tensor &dout_in, const Tensor &dq,
                                          const Tensor &dk, const Tensor &dv, bool factor_grads) {
    const Tensor dout = channel_contiguous(dout_in);
    fb_params p = block(c);
    p.o = t4(o);
    p.lse = lse.data_ptr<float>();
    p.dout = t4(dout);
    p.dq = t4(dq); p.dk = t4(dk); p.dv = t4(dv);
    Tensor dqb_full, dkb_full;
    factor_grads = factor_grads && p.r;
    // factors shared by a large batch of short sequences: a workgroup walks `group` batch entries (it then loads
    // the factor operand it keeps once), sums their factor gradients itself, and the full-shape tensors shrink by
    // that factor
    // (only for factors saved with a batch of one: a factor expanded over the batch by its caller also has batch
    // stride 0, but autograd wants its gradient in the expanded shape)
    const bool shared = p.r && c.qb.size(0) == 1 && c.kb.size(0) == 1 && p.B > 1;
    const int group = p.bias_grad_group = p.r ? (shared ? fb_suggest_bias_grad_group(&p) : 1) : 0;
    if (factor_grads) {
        const int64_t rows = ((int64_t)p.B + group - 1) / group;
        dqb_full = fresh({rows, p.Lq, p.H, p.r}, c.q.scalar_type(), c.q.device());
        dkb_full = fresh({rows, p.Lk, p.H, p.r}, c.q.scalar_type(), c.q.device());
        p.dq_bias = t4(dqb_full);
        p.dk_bias = t4(dkb_full);
    }
    // scratch of the backward, sized by the library
    Tensor scratch = fresh({(int64_t)(fb_bwd_workspace_bytes(&p) / 4)}, torch::kFloat32, c.q.device());
    p.delta = scratch.data_ptr<float>();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(c.q.device());
    const hipStream_t stream = stream_of(c.q);
    check(fb_bwd(&p, stream));
    if (!factor_grads) return {Tensor(), Tensor()};
    return {reduce_like(dqb_full, c.qb, stream), reduce_like(dkb_full, c.kb, stream)};
}

double scale_or_default(double softmax_scale, const Tensor &q) { return softmax_scale != 0.0 ? softmax_scale : 1.0 / std::sqrt((double)q.size(3)); }

Tensor given(const c10::optional<Tensor> &x) { return x.has_value() && x->defined() ? channel_contiguous(*x) : Tensor(); }

struct FlashBiasFn : public torch::autograd::Function<FlashBiasFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &qb,
                          const c10::optional<Tensor> &kb, const c10::optional<Tensor> &mask, bool causal, double scale) {
        const Call c{q, k, v, qb.value_or(Tensor()), kb.value_or(Tensor()), mask.value_or(Tensor()), causal, scale, 0};
        const auto [o, lse] = attend(c);
        ctx->save_for_backward({q, k, v, o, lse, c.qb, c.kb, c.mask});
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["scale"] = scale;
        return o;
    }

    static tensor_list backward(AutogradContext *ctx, tensor_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Call c{saved[0], saved[1], saved[2], saved[5], saved[6], saved[7], ctx->saved_data["causal"].toBool(), ctx->saved_data["scale"].toDouble(), 0};
        // as the reference, only a backward that is asked for the mask's gradient fails (flash_bias_triton.py:1371).
        // (The graph edges count the tensor arguments that were given: q, k, v, then the factors, then the mask.)
        if (c.mask.defined())
            TORCH_CHECK(!ctx->needs_input_grad(c.qb.defined() ? 5 : 3), "FlashBias does not support mask gradient yet");
        const Tensor dq = fresh_like(c.q), dk = fresh_like(c.k), dv = fresh_like(c.v);
        const bool factor_grads = c.qb.defined() && (ctx->needs_input_grad(3) || ctx->needs_input_grad(4));
        const auto [dqb, dkb] = attend_backward(c, saved[3], saved[4], grads[0], dq, dk, dv, factor_grads);
        return {dq, dk, dv, dqb, dkb, Tensor(), Tensor(), Tensor()};
    }
};

// The attention core of a cosine-attention window block on its packed projection qkv (windows, n, 3 H d).  Where the window kernels
// take the call (fb_window_ready) they normalise q and k themselves and the backward writes the packed gradient: one launch
// forward, one and a sum of the logit scale's shares backward.  Else unit q and k and the logit scale in one pass (fb_cosine_fwd),
// the operator on them and on v where it lies, and backward the operator's gradients written into the packed gradient, where one
// more pass (fb_cosine_bwd) turns dq and dk into those of the projection.  (As tensor operations: about 40 passes over tensors of
// that size, and the split of the packed tensor comes back as three zero-filled copies added up.)  `mask` (nW, n, n) or none, one
// per window of an image.
struct WindowFn : public torch::autograd::Function<WindowFn> {
    static fb_cosine cosine(const Tensor &qkv, const Tensor &logit_scale, int64_t heads, c10::ScalarType type, bool autocast) {
        fb_cosine a;
        std::memset(&a, 0, sizeof(a));
        a.size = sizeof(a);
        a.dtype = dtype_code(type);
        a.in_dtype = dtype_code(qkv.scalar_type());
        a.scale_dtype = dtype_code(logit_scale.scalar_type());
        a.H = (int32_t)heads;
        a.d = (int32_t)(qkv.size(2) / (3 * heads));
        a.tokens = qkv.size(0) * qkv.size(1);
        a.qkv = qkv.data_ptr();
        a.logit_scale = logit_scale.data_ptr();
        a.fp32 = autocast;
        return a;
    }
    // part `which` of a packed tensor, as (windows, n, H, d)
    static Tensor part(const Tensor &packed, int64_t which, int64_t heads) {
        const int64_t B = packed.size(0), n = packed.size(1), dim = packed.size(2) / 3;
        return packed.as_strided({B, n, heads, dim / heads}, {n * 3 * dim, 3 * dim, dim / heads, 1}, packed.storage_offset() + which * dim);
    }

    // c.q and c.k (and c.v, if allocated): the normalised rows in memory
    static void unit_rows(fb_cosine a, Call &c, const Tensor &qkv, c10::ScalarType type, int64_t heads, bool convert) {
        const int64_t B = qkv.size(0), n = qkv.size(1), d = qkv.size(2) / (3 * heads);
        c.q = fresh({B, n, heads, d}, type, qkv.device());
        c.k = fresh({B, n, heads, d}, type, qkv.device());
        a.q = c.q.data_ptr();
        a.k = c.k.data_ptr();
        a.v = convert ? c.v.data_ptr() : nullptr;
        const c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
        check(fb_cosine_fwd(&a, stream_of(qkv)));
    }

    static Tensor forward(AutogradContext *ctx, const Tensor &qkv, const Tensor &logit_scale, const Tensor &qb, const Tensor &kb,
                          const c10::optional<Tensor> &mask_in, int64_t heads, int64_t dtype) {
        const auto type = (c10::ScalarType)dtype;
        const int64_t B = qkv.size(0), n = qkv.size(1), d = qkv.size(2) / (3 * heads);
        // (tensor operations would compute the norm, and with it all that follows, in fp32 there)
        const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
        fb_cosine a = cosine(qkv, logit_scale, heads, type, autocast);
        Call c;
        const bool convert = qkv.scalar_type() != type;
        c.v = convert ? fresh({B, n, heads, d}, type, qkv.device()) : part(qkv, 2, heads);
        c.qb = qb;
        c.kb = kb;
        c.causal = false;
        c.scale = 1.0;
        c.mask_batches = 0;
        if (mask_in.has_value() && mask_in->defined()) {
            c.mask = channel_contiguous(*mask_in).unsqueeze(1);
            TORCH_CHECK(c.mask.dim() == 4 && c.mask.size(0) > 0 && B % c.mask.size(0) == 0, "the windows must be a multiple of the mask's");
            c.mask_batches = (int)c.mask.size(0);
        }
        ctx->saved_data["heads"] = heads;
        ctx->saved_data["autocast"] = autocast;
        ctx->saved_data["dtype"] = dtype;
        // (constant factors: their gradients need the normalised rows in memory)
        if (!convert && !autocast && !qb.requires_grad() && !kb.requires_grad()) {
            c.q = part(qkv, 0, heads);
            c.k = part(qkv, 1, heads);
            fb_params p = block(c);
            const Tensor o = fresh({B, n, heads, d}, type, qkv.device()), lse = fresh({B, heads, n}, torch::kFloat32, qkv.device());
            p.o = t4(o);
            p.lse = lse.data_ptr<float>();
            if (fb_window_ready(&p, &a, 0)) {
                const c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
                check(fb_window_fwd(&p, &a, stream_of(qkv)));
                ctx->save_for_backward({qkv, logit_scale, Tensor(), Tensor(), Tensor(), o, lse, qb, kb, c.mask});
                return o;
            }
        }
        unit_rows(a, c, qkv, type, heads, convert);
        const auto [o, lse] = attend(c);
        ctx->save_for_backward({qkv, logit_scale, c.q, c.k, convert ? c.v : Tensor(), o, lse, qb, kb, c.mask});
        return o;
    }

    static tensor_list backward(AutogradContext *ctx, tensor_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &qkv = saved[0], &logit_scale = saved[1];
        const int64_t heads = ctx->saved_data["heads"].toInt();
        const bool convert = saved[4].defined();
        Call c{saved[2], saved[3], convert ? saved[4] : part(qkv, 2, heads), saved[7], saved[8], saved[9], false, 1.0, 0};
        if (c.mask.defined()) c.mask_batches = (int)c.mask.size(0);
        TORCH_CHECK(!(c.mask.defined() && ctx->needs_input_grad(4)), "FlashBias does not support mask gradient yet");
        Tensor dqkv = fresh_like(qkv);
        Tensor dq, dk, dv;
        if (convert) {
            dq = fresh_like(c.q);
            dk = fresh_like(c.k);
            dv = fresh_like(c.v);
        } else {
            dq = part(dqkv, 0, heads);
            dk = part(dqkv, 1, heads);
            dv = part(dqkv, 2, heads);
        }
        const auto type = (c10::ScalarType)ctx->saved_data["dtype"].toInt();
        fb_cosine a = cosine(qkv, logit_scale, heads, type, ctx->saved_data["autocast"].toBool());
        Tensor dscale = fresh_like(logit_scale);
        if (!c.q.defined()) {
            c.q = part(qkv, 0, heads);
            c.k = part(qkv, 1, heads);
            const Tensor dout = channel_contiguous(grads[0]);
            fb_params p = block(c);
            p.o = t4(saved[5]);
            p.lse = saved[6].data_ptr<float>();
            p.dout = t4(dout);
            p.dq = t4(dq); p.dk = t4(dk); p.dv = t4(dv);
            if (fb_window_ready(&p, &a, 1)) {
                const Tensor partial = fresh({(int64_t)(fb_window_workspace_bytes(&p) / 4)}, torch::kFloat32, qkv.device());
                a.partial = partial.data_ptr<float>();
                a.dlogit_scale = dscale.data_ptr();
                const c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
                check(fb_window_bwd(&p, &a, stream_of(qkv)));
                return {dqkv, dscale, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
            }
            unit_rows(a, c, qkv, type, heads, false); // (a gradient or a saved tensor in rows these kernels do not read)
        }
        const auto [dqb, dkb] = attend_backward(c, saved[5], saved[6], grads[0], dq, dk, dv, ctx->needs_input_grad(2) || ctx->needs_input_grad(3));
        Tensor partial = fresh({(int64_t)(fb_cosine_workspace_bytes(&a) / 4)}, torch::kFloat32, qkv.device());
        a.dq = dq.data_ptr();
        a.dk = dk.data_ptr();
        a.dv = convert ? dv.data_ptr() : nullptr;
        a.grad_stride = dq.stride(1);
        a.dqkv = dqkv.data_ptr();
        a.dlogit_scale = dscale.data_ptr();
        a.partial = partial.data_ptr<float>();
        {
            const c10::hip::HIPGuardMasqueradingAsCUDA guard(qkv.device());
            check(fb_cosine_bwd(&a, stream_of(qkv)));
        }
        return {dqkv, dscale, dqb, dkb, Tensor(), Tensor(), Tensor()};
    }
};

// The attention core on what its kernels take, else nothing: the caller then runs the tensor operations, which take the
// rest (float64 parameters, a projection that is not packed in 16-byte aligned rows, other head dims and ranks) and say
// what is wrong with what nobody takes.
c10::optional<Tensor> window_attention(const Tensor &qkv, const Tensor &logit_scale, const Tensor &qb, const Tensor &kb,
                                       const c10::optional<Tensor> &mask, int64_t heads, py::object dtype) {
    const auto type = torch::python::detail::py_object_to_dtype(dtype);
    auto floating = [](const Tensor &x) { return x.scalar_type() == torch::kFloat16 || x.scalar_type() == torch::kBFloat16 || x.scalar_type() == torch::kFloat32; };
    const int64_t d = heads > 0 && qkv.dim() == 3 && qkv.size(2) % (3 * heads) == 0 ? qkv.size(2) / (3 * heads) : 0;
    const bool ready = d >= 8 && d <= FB_MAX_HEADDIM && (d & (d - 1)) == 0 && qkv.is_cuda() && qkv.is_contiguous() && floating(qkv) &&
                       reinterpret_cast<uintptr_t>(qkv.data_ptr()) % 16 == 0 && logit_scale.device() == qkv.device() &&
                       floating(logit_scale) && logit_scale.numel() == heads && (type == torch::kFloat16 || type == torch::kBFloat16) &&
                       qb.scalar_type() == type && kb.scalar_type() == type && qb.dim() == 4 && qb.size(3) % 8 == 0;
    if (!ready) return c10::nullopt;
    return WindowFn::apply(qkv, logit_scale.contiguous(), channel_contiguous(qb), channel_contiguous(kb), mask, heads, (int64_t)type);
}

// (q_bias, k_bias) of fb_alibi_factors, (1, L, H, rank) in the 16-bit dtype of `like`'s device.
std::pair<Tensor, Tensor> alibi_factors(int64_t Lq, int64_t Lk, int64_t heads, int64_t rank, bool reference_sign, py::object dtype, py::object device) {
    const auto type = torch::python::detail::py_object_to_dtype(dtype);
    const auto where = torch::python::detail::py_object_to_device(device);
    Tensor qb = torch::empty({1, Lq, heads, rank}, torch::TensorOptions().dtype(type).device(where));
    Tensor kb = torch::empty({1, Lk, heads, rank}, torch::TensorOptions().dtype(type).device(where));
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(qb.device());
    check(fb_alibi_factors(qb.data_ptr(), kb.data_ptr(), dtype_code(type), (int)Lq, (int)Lk, (int)heads, (int)rank, reference_sign, stream_of(qb)));
    return {qb, kb};
}

// What a projection's own route needs of the call: nothing that looks at operations or replaces them is active.
bool nothing_watches() {
    // (functorch's thread-local state outlives the thread's first transform; what a running one has included does not)
    return !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !at::autocast::is_autocast_enabled(at::kCUDA) && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing();
}

// ... and of a tensor: memory of its own that holds its values (a tensor that a transform wraps has none)
bool plain_tensor(const Tensor &t, const Tensor &like) {
    return t.is_cuda() && t.scalar_type() == like.scalar_type() && t.device() == like.device() && !t.key_set().has(c10::DispatchKey::Python) &&
           t.layout() == c10::kStrided && t.has_storage() && !t.is_neg() && !t._is_zerotensor() && !t._fw_grad(/*level=*/0).defined();
}

// x w^T + b of plain tensors of one 16-bit type: by the library's kernel (fb_linear) where that is ahead and takes them, else nothing.
Tensor many_tokens(const Tensor &x, const Tensor &w, const c10::optional<Tensor> &b) {
    const int64_t k = x.size(-1), n = w.size(0), tokens = x.numel() / k;
    auto takes = [](const Tensor &t, int align) { return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % align == 0; };
    if (n > (1 << 16) || k > (1 << 16) || !fb_linear_recommended(tokens, (int)n, (int)k) || !takes(x, 16) || !takes(w, 16) || (b.has_value() && !takes(*b, 4)))
        return Tensor();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    auto shape = x.sizes().vec();
    shape.back() = n;
    Tensor y = fresh(shape, x.scalar_type(), x.device());
    check(fb_linear(x.data_ptr(), k, w.data_ptr(), b.has_value() ? b->data_ptr() : nullptr, y.data_ptr(), dtype_code(x.scalar_type()), tokens, (int)n, (int)k,
                    stream_of(x)));
    return y;
}

// Whether dy w is left to the same kernel on the transposed weight (asked before dy is copied into rows that it reads).  Vendor library / this with the 3 us
// of the transpose, us: 147456 tokens of 128 to 128 22.7 / 20.1, of 256 to 256 38.5 / 33.6, of 512 to 512 134 / 92, 262144 of 512 to 512 196 / 147, of 384 to
// 128 59.6 / 44.7; 65536 of 512 to 512 45.9 / 45.1, of 256 to 256 19.0 / 19.9, of 384 to 128 18.3 / 18.2.
bool input_gradient_pays(int64_t tokens, const Tensor &w) {
    const int64_t n = w.size(0), k = w.size(1);
    return tokens >= 100000 && n % 64 == 0 && k % 64 == 0 && n <= (1 << 16) && k <= (1 << 16) && w.is_contiguous() &&
           reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 && fb_linear_recommended(tokens, (int)k, (int)n);
}
Tensor input_gradient(const Tensor &dy, const Tensor &w) {
    const int64_t tokens = dy.size(0), n = w.size(0), k = w.size(1);
    if (dy.stride(0) >= (1 << 22)) return Tensor();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dy.device());
    const Tensor wt = fresh({k, n}, w.scalar_type(), w.device());
    Tensor dx = fresh({tokens, k}, dy.scalar_type(), dy.device());
    check(fb_transpose(w.data_ptr(), wt.data_ptr(), (int)n, (int)k, stream_of(dy)));
    check(fb_linear(dy.data_ptr(), dy.stride(0), wt.data_ptr(), nullptr, dx.data_ptr(), dtype_code(dy.scalar_type()), tokens, (int)k, (int)n, stream_of(dy)));
    return dx;
}

// A projection x w^T + b whose weight and bias gradients come from the library's kernel for long contractions
// (fb_weight_grad); the forward is the library's where it is ahead (many_tokens), and so is the input's gradient (input_gradient).
struct LinearFn : public torch::autograd::Function<LinearFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, const c10::optional<Tensor> &b) {
        // (the weight only where the input's gradient needs it: as long as it is saved nobody may change it before the backward)
        ctx->save_for_backward({x, x.requires_grad() ? w : Tensor()});
        ctx->saved_data["bias"] = b.has_value();
        const Tensor y = many_tokens(x, w, b);
        return y.defined() ? y : at::linear(x, w, b);
    }

    static tensor_list backward(AutogradContext *ctx, tensor_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &w = saved[1];
        const int64_t n = grads[0].size(-1), k = x.size(-1);
        const bool bias = ctx->saved_data["bias"].toBool();
        const Tensor dy = grads[0].reshape({-1, n});
        Tensor dx, dw, db;
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1), want_b = bias && ctx->needs_input_grad(2);
        // (a gradient that is itself differentiated, batched gradients, modes that look at the backward: tensor operations)
        const bool plain = !c10::GradMode::is_enabled() && plain_tensor(x, x) && plain_tensor(dy, x) && nothing_watches();
        auto rows = [](const Tensor &t) { // rows of contiguous, 16-byte aligned elements
            const bool ok = t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 && t.stride(0) < (1 << 24) &&
                            reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
            return ok ? t : t.clone(at::MemoryFormat::Contiguous);
        };
        Tensor y2; // dy in such rows, for whoever reads them: copied at most once, and not for a product of the tensor library
        if (want_x && plain && plain_tensor(w, x) && input_gradient_pays(dy.size(0), w)) dx = input_gradient(y2 = rows(dy), w);
        if (want_x) dx = (dx.defined() ? dx : dy.matmul(w)).reshape(x.sizes());
        if (want_w && plain) {
            if (!y2.defined()) y2 = rows(dy);
            const Tensor x2 = rows(x.reshape({-1, k}));
            dw = fresh({n, k}, x.scalar_type(), x.device());
            if (want_b) db = fresh({n}, x.scalar_type(), x.device());
            const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
            Tensor scratch = fresh({(int64_t)(fb_weight_grad_workspace_bytes(y2.size(0), (int)n, (int)k, want_b) / 4)}, torch::kFloat32, x.device());
            check(fb_weight_grad(y2.data_ptr(), y2.stride(0), x2.data_ptr(), x2.stride(0), dw.data_ptr(), want_b ? db.data_ptr() : nullptr,
                                 scratch.data_ptr<float>(), dtype_code(x.scalar_type()), y2.size(0), (int)n, (int)k, stream_of(x)));
        } else {
            if (want_w) dw = dy.t().matmul(x.reshape({-1, k}));
            if (want_b) db = dy.sum(0);
        }
        return {dx, dw, db};
    }
};

// The projection where its weight gradient is asked for and the library's kernel for it is ahead, or where nothing is differentiated and
// the library's product is, else nothing: the caller then takes the tensor library's own operation, which is also what modes,
// transforms and tracers that look at operations see.
c10::optional<Tensor> linear(const Tensor &x, const Tensor &w, const c10::optional<Tensor> &b) {
    const auto type = x.scalar_type();
    const bool ready = (type == torch::kFloat16 || type == torch::kBFloat16) && plain_tensor(x, x) && plain_tensor(w, x) && x.dim() >= 2 && w.dim() == 2 &&
                       x.size(-1) == w.size(1) && x.numel() > 0 && (!b.has_value() || (plain_tensor(*b, x) && b->dim() == 1 && b->size(0) == w.size(0))) &&
                       nothing_watches();
    if (!ready) return c10::nullopt;
    if (!c10::GradMode::is_enabled()) {
        const Tensor y = many_tokens(x, w, b);
        return y.defined() ? c10::optional<Tensor>(y) : c10::nullopt;
    }
    if (!w.requires_grad() || w.size(0) > (1 << 16) || w.size(1) > (1 << 16) ||
        !fb_weight_grad_recommended(x.numel() / x.size(-1), (int)w.size(0), (int)w.size(1)))
        return c10::nullopt;
    return LinearFn::apply(x, w, b);
}

// x w^T for each of three weights in one launch of the library's kernel, where nothing is differentiated and that kernel is
// ahead, else an empty list (the caller then takes the tensor library's operations, as with `linear`).
std::vector<Tensor> project(const Tensor &x, const std::vector<Tensor> &w) {
    const auto type = x.scalar_type();
    const bool grad_mode = c10::GradMode::is_enabled();
    auto takes = [&](const Tensor &t) {
        return plain_tensor(t, x) && !(grad_mode && t.requires_grad()) && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    };
    if (!(type == torch::kFloat16 || type == torch::kBFloat16) || x.dim() < 2 || w.size() != 3 || !nothing_watches() || !takes(x) || x.numel() == 0)
        return {};
    const int64_t k = x.size(-1), tokens = x.numel() / k;
    const void *ws[3];
    void *ys[3];
    int n[3];
    for (int i = 0; i < 3; ++i) {
        if (w[i].dim() != 2 || w[i].size(1) != k || w[i].size(0) > (1 << 16) || k > (1 << 16) || !takes(w[i])) return {};
        n[i] = (int)w[i].size(0);
        ws[i] = w[i].data_ptr();
    }
    if (!fb_project_recommended(tokens, (int)k, n, 3)) return {};
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    std::vector<Tensor> y(3);
    auto shape = x.sizes().vec();
    for (int i = 0; i < 3; ++i) {
        shape.back() = n[i];
        y[i] = fresh(shape, type, x.device());
        ys[i] = y[i].data_ptr();
    }
    check(fb_project(x.data_ptr(), k, ws, ys, n, 3, dtype_code(type), tokens, (int)k, stream_of(x)));
    return y;
}

// x (..., r) with its last dim zero-padded (or cut) to `rank` columns in one launch of the library; the gradient
// is the same operation the other way.  For contiguous 16-bit GPU tensors (the caller checks).
struct ResizeRankFn : public torch::autograd::Function<ResizeRankFn> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, int64_t rank) {
        TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.element_size() == 2 && x.dim() >= 1 && x.numel() > 0 && rank > 0,
                    "resize_rank wants a contiguous fp16 / bf16 GPU tensor");
        ctx->saved_data["rank_in"] = x.size(-1);
        auto shape = x.sizes().vec();
        shape.back() = rank;
        Tensor out = torch::empty(shape, x.options());
        const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
        check(fb_resize_rank(x.data_ptr(), out.data_ptr(), out.numel() / rank, (int)x.size(-1), (int)rank,
                             c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream()));
        return out;
    }

    static tensor_list backward(AutogradContext *ctx, tensor_list grads) {
        return {ResizeRankFn::apply(grads[0].contiguous(), ctx->saved_data["rank_in"].toInt()), Tensor()};
    }
};

Tensor resize_rank(const Tensor &x, int64_t rank) { return ResizeRankFn::apply(x, rank); }

// An input that a derivative is wanted of.  A forward-mode tangent counts: tensors that carry one need not require a
// gradient, and may do so with gradients off.
bool differentiated(const Tensor &x) {
    return x.defined() && ((c10::GradMode::is_enabled() && x.requires_grad()) || x._fw_grad(/*level=*/0).defined());
}

// Both factors of a call (contiguous 16-bit GPU tensors of one rank) resized: in one launch where neither asks for a
// gradient and both are on one device (constant factors: ALiBi on every call), by one autograd node each otherwise.
std::pair<Tensor, Tensor> resize_ranks(const Tensor &q_bias, const Tensor &k_bias, int64_t rank) {
    if (differentiated(q_bias) || differentiated(k_bias) || q_bias.device() != k_bias.device() || q_bias.scalar_type() != k_bias.scalar_type())
        return {ResizeRankFn::apply(q_bias, rank), ResizeRankFn::apply(k_bias, rank)};
    if (const auto &transforms = at::functorch::functorchTLSAccessor()) transforms->checkSupportsCppAutogradFunction();
    Tensor out[2];
    const Tensor *const in[2] = {&q_bias, &k_bias};
    for (int i = 0; i < 2; ++i) {
        const Tensor &x = *in[i];
        TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.element_size() == 2 && x.dim() >= 1 && x.numel() > 0 && rank > 0 &&
                        x.size(-1) == q_bias.size(-1),
                    "resize_ranks wants contiguous fp16 / bf16 GPU tensors of one rank");
        auto shape = x.sizes().vec();
        shape.back() = rank;
        out[i] = fresh(shape, x.scalar_type(), x.device());
    }
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(q_bias.device());
    check(fb_resize_ranks(q_bias.data_ptr(), out[0].data_ptr(), out[0].numel() / rank, k_bias.data_ptr(), out[1].data_ptr(),
                          out[1].numel() / rank, (int)q_bias.size(-1), (int)rank, stream_of(q_bias)));
    return {out[0], out[1]};
}

Tensor flash_bias(const Tensor &q_in, const Tensor &k_in, const Tensor &v_in, const c10::optional<Tensor> &q_bias,
                  const c10::optional<Tensor> &k_bias, const c10::optional<Tensor> &mask, bool causal, double softmax_scale) {
    const Tensor q = channel_contiguous(q_in), k = channel_contiguous(k_in), v = channel_contiguous(v_in);
    const Tensor qb = given(q_bias), kb = given(k_bias), m = given(mask);
    TORCH_CHECK(!qb.defined() || kb.defined(), "q_bias without k_bias");
    const double scale = scale_or_default(softmax_scale, q);
    // Nothing to differentiate: no graph node either.  What the autograd function refuses stays refused: inputs that
    // carry a forward-mode tangent (they need not require a gradient, and may do so with gradients off; without the
    // refusal their derivative would come out as zero) and calls under a function transform (torch.func).
    if (!(differentiated(q) || differentiated(k) || differentiated(v) || differentiated(qb) || differentiated(kb) || differentiated(m))) {
        if (const auto &transforms = at::functorch::functorchTLSAccessor()) transforms->checkSupportsCppAutogradFunction();
        return attend(Call{q, k, v, qb, kb, m, causal, scale, 0}).first;
    }
    auto maybe = [](const Tensor &x) { return x.defined() ? c10::optional<Tensor>(x) : c10::nullopt; };
    return FlashBiasFn::apply(q, k, v, maybe(qb), maybe(kb), maybe(m), causal, scale);
}

// The operator on arguments that need no preparation and break no rule, else nothing: the caller then takes its own
// way through the checks (which say what is wrong) and the preparations.
c10::optional<Tensor> flash_bias_ready(const Tensor &q, const Tensor &k, const Tensor &v, const c10::optional<Tensor> &q_bias,
                                       const c10::optional<Tensor> &k_bias, const c10::optional<Tensor> &mask, bool causal,
                                       c10::optional<double> softmax_scale) {
    const auto type = q.scalar_type();
    const bool ready = q.dim() == 4 && k.dim() == 4 && q.is_cuda() && k.is_cuda() && v.is_cuda() && (type == torch::kFloat16 || type == torch::kBFloat16) &&
                       k.scalar_type() == type && v.scalar_type() == type && k.size(0) == q.size(0) && k.size(2) == q.size(2) &&
                       k.size(3) == q.size(3) && v.sizes() == k.sizes() && q.size(3) <= FB_MAX_HEADDIM &&
                       !(q_bias.has_value() && (q_bias->dim() != 4 || q_bias->size(3) % 8 != 0)) &&
                       !(mask.has_value() && mask->dim() == 4 && mask->size(2) == 1);
    if (!ready) return c10::nullopt;
    return flash_bias(q, k, v, q_bias, k_bias, mask, causal, softmax_scale.value_or(0.0));
}

} // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "flash_bias_func with its autograd function in C++ (kernel-ready inputs; see flashbias_amd/interface.py)";
    // what this module was compiled against: the caller compares both with the library it loaded
    m.def("abi", []() { return std::make_pair((int)FB_VERSION, (int)sizeof(fb_params)); });
    m.def("flash_bias_ready", &flash_bias_ready, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("q_bias"), py::arg("k_bias"), py::arg("mask"),
          py::arg("causal"), py::arg("softmax_scale"));
    m.def("window_attention", &window_attention, py::arg("qkv"), py::arg("logit_scale"), py::arg("q_bias"), py::arg("k_bias"), py::arg("mask"),
          py::arg("heads"), py::arg("dtype"));
    m.def("alibi_factors", &alibi_factors, py::arg("seqlen_q"), py::arg("seqlen_k"), py::arg("heads"), py::arg("rank"), py::arg("reference_sign"),
          py::arg("dtype"), py::arg("device"));
    m.def("linear", &linear, py::arg("x"), py::arg("weight"), py::arg("bias"));
    m.def("project", &project, py::arg("x"), py::arg("weights"));
    m.def("resize_rank", &resize_rank, py::arg("x"), py::arg("rank"));
    m.def("resize_ranks", &resize_ranks, py::arg("q_bias"), py::arg("k_bias"), py::arg("rank"));
    m.def("flash_bias", &flash_bias, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("q_bias") = py::none(),
          py::arg("k_bias") = py::none(), py::arg("mask") = py::none(), py::arg("causal") = false,
          py::arg("softmax_scale") = 0.0);
}
