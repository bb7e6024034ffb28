"""Module-level drop-ins that call ``flash_bias_func`` the way the reference's application
code does: an ALiBi causal self-attention block
(1_Language_Model/attention_with_alibi_bias.py:18-64) and the attention core of a Swin-V2
window block with SVD bias factors (2_Vision_Transformer/swin_transformer_v2.py:155-207).
They exist for end-to-end layer timing and as usage examples; parameters are randomly
initialised (no checkpoints ship with either repository)."""
import torch
import torch.nn as nn

from . import factors, interface
from .interface import flash_bias_func


# (csrc/fb_wgrad.hip takes no fewer; asked for here because a block of a few hundred tokens is bound by the host, where
# looking at its four layers cost 4 % of a training step: 1822 tokens of 1024 channels, 516 -> 538 us)
_TOKENS_OF_A_LONG_CONTRACTION = 6000


# (a subclass may see or replace operations by ``__torch_function__``, which a call into the extension is not)
_TENSORS = (torch.Tensor, nn.Parameter)


def _plain(layer):
    """Whether ``layer`` is a plain ``nn.Linear`` on plain tensors that nothing hooks into or replaces."""
    return (type(layer) is nn.Linear and type(layer.weight) in _TENSORS and (layer.bias is None or type(layer.bias) in _TENSORS)
            and not torch.compiler.is_compiling()
            and not (layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks or layer._backward_pre_hooks)
            and "forward" not in layer.__dict__ and layer._compiled_call_impl is None
            and not nn.modules.module._has_any_global_hook())


def _project(layer, x):
    """``layer(x)``.  A plain ``nn.Linear`` over many tokens is the library's own product and gets its weight gradient from the
    library's own kernel (``ext.linear``, which says for which calls; a layer that something hooks into or replaces is called)."""
    if type(x) in _TENSORS and x.is_cuda and x.numel() >= _TOKENS_OF_A_LONG_CONTRACTION * x.shape[-1] and _plain(layer):
        ext = interface._extension()
        if ext is not None:
            y = ext.linear(x, layer.weight, layer.bias)
            if y is not None:
                return y
    return layer(x)


def _project_all(layers, x):
    """``[layer(x) for layer in layers]``.  Plain ``nn.Linear`` layers without bias, with gradients off, in one launch of the
    library's own kernel (``ext.project``, which says for which calls)."""
    if type(x) in _TENSORS and x.is_cuda and not torch.is_grad_enabled() and all(_plain(layer) and layer.bias is None for layer in layers):
        ext = interface._extension()
        y = None if ext is None else ext.project(x, [layer.weight for layer in layers])
        if y:
            return y
    return [_project(layer, x) for layer in layers]


class AttentionWithALiBiBias(nn.Module):
    """Causal multi-head self-attention with ALiBi as an exact rank-2 FlashBias.

    Same constructor arguments and forward contract as the reference module
    (x: (batch, seq, dim) -> (batch, seq, dim)).  Two deliberate differences, both switchable:
    the bias follows the standard ALiBi sign, ``-m_h (i - j)``, unless ``reference_sign=True``
    (the reference builds ``+m_h (i - j)``, attention_with_alibi_bias.py:49-52), and the compute
    dtype defaults to bf16 where the reference casts to fp16 (``dtype=torch.float16`` restores
    that).  The factors are the exact rank-4 form of ``factors.alibi_factors``: the bias the
    kernels see is exactly ``-m (i - j)`` with the slope rounded to the dtype, at every position."""

    def __init__(self, dim, heads, dim_head, dropout=0.0, dtype=torch.bfloat16, reference_sign=False):
        super().__init__()
        self.reference_sign = reference_sign
        inner = dim_head * heads
        self.heads, self.dim_head, self.scale, self.dtype = heads, dim_head, dim_head ** -0.5, dtype
        self.to_q = nn.Linear(dim, inner, bias=False)
        self.to_k = nn.Linear(dim, inner, bias=False)
        self.to_v = nn.Linear(dim, inner, bias=False)
        self.to_out = nn.Sequential(nn.Linear(inner, dim), nn.Dropout(dropout))

    def forward(self, x):
        b, n, _ = x.shape
        split = lambda t: t.view(b, n, self.heads, self.dim_head).to(self.dtype)
        q, k, v = (split(t) for t in _project_all((self.to_q, self.to_k, self.to_v), x))
        ext = interface._extension()
        if ext is not None and x.is_cuda and n <= 65536:
            # the same factors in one launch, with the zero columns the operator would append on every call
            q_bias, k_bias = ext.alibi_factors(n, n, self.heads, 16, self.reference_sign, self.dtype, x.device)
        else:
            q_bias, k_bias = factors.alibi_factors(n, n, self.heads, self.dtype, x.device, exact=True,
                                                   reference_sign=self.reference_sign)
        o = flash_bias_func(q, k, v, q_bias, k_bias, None, True, self.scale)
        return self.to_out(o.reshape(b, n, -1).to(x.dtype))


class WindowAttentionCore(nn.Module):
    """The attention core of a Swin-V2 window block: cosine attention with a learned per-head
    logit scale, a relative-position bias given by rank-``rank`` SVD factors shared by all
    windows, and an optional shifted-window mask (num_windows, N, N) of 0 / -100 entries.

    x: (num_windows * B, N, C) -> (num_windows * B, N, C), as WindowAttention.forward
    (swin_transformer_v2.py:155-207); scale 1 is passed to the kernel because q is pre-scaled."""

    def __init__(self, dim, window, heads, rank=16, seed=0, dtype=torch.bfloat16):
        super().__init__()
        self.heads, self.dtype = heads, dtype
        self.qkv = nn.Linear(dim, dim * 3, bias=False)
        self.proj = nn.Linear(dim, dim)
        self.logit_scale = nn.Parameter(torch.log(10 * torch.ones(heads, 1, 1)))
        table = factors.swin_v2_bias_table(window, heads, seed)
        q_bias, k_bias, rel = factors.svd_factors(table, rank, dtype)
        self.register_buffer("q_bias_pos", q_bias)  # (1, N, H, rank)
        self.register_buffer("k_bias_pos", k_bias)
        self.register_buffer("bias_rel_error", rel)

    def forward(self, x, mask=None):
        b_, n, c = x.shape
        qkv = _project(self.qkv, x)
        ext = interface._extension()
        if ext is not None and qkv.is_cuda:
            # normalisation, attention and the packed projection's gradient without passes in between (csrc/fb_torch.cpp)
            m = mask
            if mask is not None:
                m = mask.to(self.dtype)
                if m.dim() != 3 or m.shape[2] != n:  # broadcast over the keys (or the windows), as below
                    m = m[None, :, None].expand(1, m.shape[0], 1, n, n)[0, :, 0]
            o = ext.window_attention(qkv, self.logit_scale, self.q_bias_pos, self.k_bias_pos, m, self.heads, self.dtype)
            if o is not None:
                return _project(self.proj, o.reshape(b_, n, c).to(x.dtype))
        qkv = qkv.view(b_, n, 3, self.heads, c // self.heads)
        q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
        scale = torch.clamp(self.logit_scale, max=4.6052).exp().view(1, 1, self.heads, 1)
        q = (torch.nn.functional.normalize(q, dim=-1) * scale).to(self.dtype)
        k = torch.nn.functional.normalize(k, dim=-1).to(self.dtype)
        if mask is not None:
            nw = mask.shape[0]
            mask = mask.to(self.dtype)[None, :, None].expand(b_ // nw, nw, 1, n, n).reshape(b_, 1, n, n)
        o = flash_bias_func(q, k, v.to(self.dtype), self.q_bias_pos, self.k_bias_pos, mask, False, 1.0)
        return _project(self.proj, o.reshape(b_, n, c).to(x.dtype))
