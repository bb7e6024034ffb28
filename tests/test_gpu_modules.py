"""The one-pass kernels of the module drop-ins (csrc/fb_cosine.hip, the ALiBi factor builder) against the tensor
operations they replace."""
import ctypes

import pytest
import torch

from flashbias_amd import _lib, factors, interface, modules

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,heads,sign", [(1, 1, False), (257, 3, True), (700, 50, False), (64, 128, True)])
def test_alibi_factors_in_one_launch(gpu_device, dtype, n, heads, sign):
    want = factors.alibi_factors(n, n + 5, heads, dtype, gpu_device, exact=True, reference_sign=sign)
    for rank in (8, 16):
        got = interface._extension().alibi_factors(n, n + 5, heads, rank, sign, dtype, gpu_device)
        for g, w in zip(got, want):
            assert torch.equal(g[..., :4], w) and not g[..., 4:].any()


# param dtype = dtype of the packed projection; 1 head of 8 channels: 1 chunk a token, fewer than a workgroup has
# lanes; 3 heads of 128: 48 chunks, which do not divide 256; windows shared by images through the mask's period
@pytest.mark.parametrize("dtype,param", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("window,heads,hd,windows,types", [(3, 1, 8, 1, 0), (8, 2, 32, 6, 3), (7, 3, 128, 4, 4), (16, 5, 16, 8, 2), (12, 2, 64, 3, 1),
                                                           (16, 8, 32, 64, 0)])
def test_window_block_against_tensor_operations(gpu_device, monkeypatch, dtype, param, window, heads, hd, windows, types):
    torch.manual_seed(1)
    n, dim = window * window, heads * hd
    mod = modules.WindowAttentionCore(dim, window, heads, rank=8, dtype=dtype).to(gpu_device, param)
    mod.q_bias_pos, mod.k_bias_pos = mod.q_bias_pos.to(dtype), mod.k_bias_pos.to(dtype)
    with torch.no_grad():
        mod.logit_scale[0] = 6.0  # clamped: no gradient
    x = torch.randn(windows, n, dim, device=gpu_device, dtype=param, requires_grad=True)
    dy = torch.randn(windows, n, dim, device=gpu_device, dtype=param)
    mask = (torch.rand(types, n, n, device=gpu_device) < 0.2).float() * -100.0 if types else None
    leaves = [x] + list(mod.parameters())
    def grads():
        y = mod(x, mask)
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]
    got = grads()
    monkeypatch.setattr(interface, "_ext", None)  # the tensor operations and the Python autograd function
    want = grads()
    # (q and k have the same bits on both ways: test_cosine_forward_has_the_bits_of_tensor_operations)  What is left is the backward's own rounding (2^-8 per product of
    # bf16 tensor operations, of which the fused pass has fewer) and the summation orders
    bound = 3e-2
    for name, g, w in zip(["y", "x"] + [k for k, _ in mod.named_parameters()], got, want):
        assert torch.isfinite(g).all() and g.shape == w.shape and g.dtype == w.dtype, name
        if w.float().abs().max() == 0:
            assert g.abs().max() == 0, name
        else:
            assert (g.float() - w.float()).norm() <= bound * w.float().norm(), name
    assert got[2].flatten()[0] == 0


class FbCosine(ctypes.Structure):  # fb_cosine of include/flashbias.h
    _fields_ = ([("size", ctypes.c_uint32)] + [(n, ctypes.c_int32) for n in ("dtype", "in_dtype", "scale_dtype", "H", "d")]
                + [("tokens", ctypes.c_int64)] + [(n, ctypes.c_void_p) for n in ("qkv", "logit_scale", "q", "k", "v", "dq", "dk", "dv")]
                + [("grad_stride", ctypes.c_int64)] + [(n, ctypes.c_void_p) for n in ("dqkv", "dlogit_scale", "partial")]
                + [("fp32", ctypes.c_int32), ("reserved", ctypes.c_int32)])


CODES = {torch.float16: _lib.FB_F16, torch.bfloat16: _lib.FB_BF16, torch.float32: _lib.FB_F32}


def _cosine_block(qkv, logit_scale, heads, dtype):
    a = FbCosine()
    a.size = ctypes.sizeof(FbCosine)
    a.dtype, a.in_dtype, a.scale_dtype = CODES[dtype], CODES[qkv.dtype], CODES[logit_scale.dtype]
    a.H, a.d, a.tokens = heads, qkv.shape[1] // (3 * heads), qkv.shape[0]
    a.qkv, a.logit_scale = qkv.data_ptr(), logit_scale.data_ptr()
    return a


def _cosine_inputs(dev, in_dtype, scale_dtype, heads, d, tokens=333):
    g = torch.Generator().manual_seed(4)
    qkv = (torch.randn(tokens, 3 * heads * d, generator=g) * torch.logspace(-3, 3, tokens, dtype=torch.float32)[:, None]).to(in_dtype)
    qkv[7] = 0  # rows without a direction
    scale = (torch.randn(heads, generator=g) * 0.5 + 2.3).to(scale_dtype)
    scale[0] = 7.0  # clamped
    return qkv.to(dev), scale.to(dev)


def _cosine_exact(qkv, logit_scale, heads):
    """q, k, v of (tokens, 3 H d) as float64 tensor operations; the clamp's bound is a number of the parameter's type."""
    x = qkv.double().view(qkv.shape[0], 3, heads, -1)
    top = torch.tensor(4.6052).to(logit_scale.dtype).double().item()
    s = logit_scale.double().clamp(max=top).exp()[None, :, None]
    unit = lambda t: torch.nn.functional.normalize(t, dim=-1)
    return unit(x[:, 0]) * s, unit(x[:, 1]), x[:, 2]


COSINE_TYPES = [(torch.bfloat16, torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.bfloat16, torch.float32),
                (torch.float16, torch.float16, torch.float32), (torch.float16, torch.bfloat16, torch.float32),
                (torch.float32, torch.bfloat16, torch.float32), (torch.float32, torch.float16, torch.bfloat16)]


@pytest.mark.parametrize("in_dtype,dtype,scale_dtype", COSINE_TYPES)
@pytest.mark.parametrize("heads,d", [(1, 8), (3, 16), (5, 32), (2, 128)])
def test_cosine_forward_in_fp32_rounds_once(gpu_device, in_dtype, dtype, scale_dtype, heads, d):
    """Unit q (times the logit scale) and unit k with fp32 steps are the float64 values rounded once to the attention's
    type, whatever types the projection and the scale have."""
    lib = _lib.load()
    qkv, scale = _cosine_inputs(gpu_device, in_dtype, scale_dtype, heads, d)
    got = [torch.full((qkv.shape[0], heads, d), float("nan"), device=gpu_device, dtype=dtype) for _ in range(3)]
    a = _cosine_block(qkv, scale, heads, dtype)
    a.q, a.k, a.v = (t.data_ptr() for t in got)
    a.fp32 = 1
    _lib.check_status(lib.fb_cosine_fwd(ctypes.byref(a), ctypes.c_void_p(interface._stream())))
    torch.cuda.synchronize()
    # half a unit in the last place of the result's 8 or 11 significant bits (fp16: subnormals below 2^-14) on top of the
    # fp32 arithmetic: 8 + log2(d / 8) additions halved by the root, the root, the division, the product, 2 units of exp
    bits, low = (8, -125) if dtype == torch.bfloat16 else (11, -13)
    for name, g, w in zip("qkv", got, _cosine_exact(qkv, scale, heads)):
        half = torch.ldexp(torch.ones_like(w), torch.frexp(w).exponent.clamp(min=low) - 1 - bits)
        excess = (g.double() - w).abs() - half - w.abs() * 12 * 2.0 ** -24
        assert (excess <= 0).all(), (name, float((excess / half).max()))
    assert not got[0][7].any() and not got[1][7].any()


@pytest.mark.parametrize("in_dtype,dtype,scale_dtype", [t for t in COSINE_TYPES if t[0] != torch.float32])
@pytest.mark.parametrize("heads,d", [(1, 8), (3, 16), (5, 32), (2, 128)])
def test_cosine_forward_has_the_bits_of_tensor_operations(gpu_device, in_dtype, dtype, scale_dtype, heads, d):
    """With steps in the projection's type q and k are those of the tensor operations, also from a block that ends before
    the field that says so."""
    lib = _lib.load()
    qkv, scale = _cosine_inputs(gpu_device, in_dtype, scale_dtype, heads, d)
    qkv[7] = 1  # (a row of zeros in fp16 is 0 / 0 on both ways)
    x = qkv.view(qkv.shape[0], 3, heads, d)
    unit = lambda t: torch.nn.functional.normalize(t, dim=-1)
    s = torch.clamp(scale, max=4.6052).exp().view(1, heads, 1)
    want = [(unit(x[:, 0]) * s).to(dtype), unit(x[:, 1]).to(dtype), x[:, 2].to(dtype)]
    for size in (ctypes.sizeof(FbCosine), FbCosine.fp32.offset):
        got = [torch.full_like(w, float("nan")) for w in want]
        a = _cosine_block(qkv, scale, heads, dtype)
        a.size = size
        a.q, a.k, a.v = (t.data_ptr() for t in got)
        _lib.check_status(lib.fb_cosine_fwd(ctypes.byref(a), ctypes.c_void_p(interface._stream())))
        torch.cuda.synchronize()
        for name, g, w in zip("qkv", got, want):
            # (the two sum squares in fp32 in orders of their own: up to 12 x 2^-24 apart, which puts one norm in
            # 2^12 / 12 (fp16; bf16 2^15 / 12) on the other side of a rounding: at most two of the 333 to 1665 here, twice d elements)
            assert int((g != w).any(-1).sum()) <= (0 if name == "v" else 2), name
            assert (g.float() - w.float()).abs().max() <= 2.0 ** -6 * w.float().abs().max(), name


def _window_params(qkv, qb, kb, mask, heads, o, lse):
    """fb_params of the attention of a window block whose q, k, v are the parts of the packed projection (windows, n, 3 H d)."""
    windows, n, dim = qkv.shape[0], qkv.shape[1], qkv.shape[2] // 3
    p = _lib.new_params()
    p.dtype, p.B, p.H, p.Lq, p.Lk, p.d, p.r, p.scale = CODES[qkv.dtype], windows, heads, n, n, dim // heads, qb.shape[3], 1.0
    packed = lambda t, i: _lib.FbTensor(t.data_ptr() + 2 * dim * i, 3 * n * dim, dim // heads, 3 * dim)
    p.q, p.k, p.v = (packed(qkv, i) for i in range(3))
    p.q_bias, p.k_bias = (_lib.FbTensor(t.data_ptr(), 0, t.stride(2), t.stride(1)) for t in (qb, kb))
    if mask is not None:
        p.mask_type, p.mask_dtype, p.mask_batches = 2, CODES[mask.dtype], mask.shape[0]
        p.mask = _lib.FbTensor(mask.data_ptr(), n * n, 0, n)
    p.o = _lib.FbTensor(o.data_ptr(), n * dim, dim // heads, dim)
    p.lse = lse.data_ptr()
    return p, packed


# edges: one query, one block, blocks of 32 and of 64 keys with a remainder, one and two halves of 128 queries, workgroups that walk
# several windows (2048 x 8), four waves and eight (up to 512 pairs), grids below those where the operator takes these kernels
@pytest.mark.parametrize("dtype,scale_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("windows,n,heads,rank,types", [(2048, 8, 1, 8, 0), (1030, 1, 1, 8, 0), (2050, 49, 8, 16, 0), (260, 64, 4, 16, 4), (130, 72, 8, 8, 2), (344, 144, 3, 16, 0),
                                                        (512, 144, 2, 16, 8), (128, 256, 8, 8, 0), (1024, 256, 1, 16, 4), (520, 200, 2, 16, 1), (3, 256, 5, 16, 3)])
def test_window_block_in_the_attention_kernels(gpu_device, dtype, scale_dtype, windows, n, heads, rank, types):
    """fb_window_fwd and fb_window_bwd have the bits of the normalisation, the operator and the normalisation's backward one after
    the other; the logit scale's gradient is another order of the same sum."""
    lib, s = _lib.load(), ctypes.c_void_p(interface._stream())
    g = torch.Generator(device=gpu_device).manual_seed(n)
    dim = 32 * heads
    rand = lambda *shape: torch.randn(*shape, generator=g, device=gpu_device)
    qkv = (rand(windows, n, 3 * dim) * torch.exp2(rand(windows, n, 1))).to(dtype)
    if dtype == torch.bfloat16:
        qkv[1, 0, :dim] = 0  # a row without a direction (fp16: 0 / 0)
        qkv[2, n // 2, dim:2 * dim] = 1e20  # a norm beyond fp32: zeros
    qb, kb = (rand(1, n, heads, rank).to(dtype) * 0.3 for _ in range(2))
    scale = (rand(heads) * 0.5 + 2).to(scale_dtype)
    scale[-1] = 5.0  # clamped
    mask = ((rand(types, n, n) < -0.5).to(dtype) * -100.0) if types else None
    dout = rand(windows, n, dim).to(dtype)
    full = lambda *shape, dt=dtype: torch.full(shape, float("nan"), device=gpu_device, dtype=dt)

    def outputs():
        return full(windows, n, dim), full(windows, heads, n, dt=torch.float32), full(windows, n, 3 * dim), full(heads, dt=scale_dtype)

    def one():
        o, lse, dqkv, dscale = outputs()
        p, packed = _window_params(qkv, qb, kb, mask, heads, o, lse)
        a = _cosine_block(qkv.view(windows * n, -1), scale, heads, dtype)
        assert lib.fb_window_ready(ctypes.byref(p), ctypes.byref(a), 0), lib.fb_last_error()
        _lib.check_status(lib.fb_window_fwd(ctypes.byref(p), ctypes.byref(a), s))
        p.dout = _lib.FbTensor(dout.data_ptr(), n * dim, 32, dim)
        p.dq, p.dk, p.dv = (packed(dqkv, i) for i in range(3))
        partial = full(lib.fb_window_workspace_bytes(ctypes.byref(p)) // 4, dt=torch.float32)
        a.partial, a.dlogit_scale = partial.data_ptr(), dscale.data_ptr()
        assert lib.fb_window_ready(ctypes.byref(p), ctypes.byref(a), 1), lib.fb_last_error()
        _lib.check_status(lib.fb_window_bwd(ctypes.byref(p), ctypes.byref(a), s))
        return o, lse, dqkv, dscale

    def parts():
        o, lse, dqkv, dscale = outputs()
        q, k = full(windows, n, dim), full(windows, n, dim)
        a = _cosine_block(qkv.view(windows * n, -1), scale, heads, dtype)
        a.q, a.k = q.data_ptr(), k.data_ptr()
        _lib.check_status(lib.fb_cosine_fwd(ctypes.byref(a), s))
        p, packed = _window_params(qkv, qb, kb, mask, heads, o, lse)
        p.q, p.k = (_lib.FbTensor(t.data_ptr(), n * dim, 32, dim) for t in (q, k))
        _lib.check_status(lib.fb_fwd(ctypes.byref(p), s))
        p.dout = _lib.FbTensor(dout.data_ptr(), n * dim, 32, dim)
        p.dq, p.dk, p.dv = (packed(dqkv, i) for i in range(3))
        scratch = full(lib.fb_bwd_workspace_bytes(ctypes.byref(p)) // 4, dt=torch.float32)
        p.delta = scratch.data_ptr()
        _lib.check_status(lib.fb_bwd(ctypes.byref(p), s))
        lib.fb_cosine_workspace_bytes.restype = ctypes.c_size_t
        partial = full(lib.fb_cosine_workspace_bytes(ctypes.byref(a)) // 4, dt=torch.float32)
        a.dq, a.dk, a.grad_stride = p.dq.ptr, p.dk.ptr, 3 * dim
        a.dqkv, a.dlogit_scale, a.partial = dqkv.data_ptr(), dscale.data_ptr(), partial.data_ptr()
        _lib.check_status(lib.fb_cosine_bwd(ctypes.byref(a), s))
        return o, lse, dqkv, dscale

    got, want = one(), parts()
    torch.cuda.synchronize()
    same = windows * heads >= 1024  # (below, the operator's backward is not the ring kernel: other summation orders)
    for name, x, w in zip(("o", "lse", "dqkv", "dlogit_scale"), got, want):
        assert torch.isfinite(x).all(), name
        if name == "dlogit_scale":
            # sums of 32 windows n products each, any order: 2^-24 sqrt(their number) of the root of their sum of squares, which
            # is that of random signs, and one rounding to the parameter's type
            terms = 32 * windows * n
            eps = 2.0 ** -24 if scale_dtype == torch.float32 else 2.0 ** -8 if scale_dtype == torch.bfloat16 else 2.0 ** -11
            big = float(w.float().abs().max())
            assert (x.float() - w.float()).abs().max() <= (eps + 2.0 ** -24 * terms ** 0.5 * 8 + (0 if same else 2.0 ** -8)) * max(big, 1.0), name
            assert float(x[-1]) == 0
        elif name == "dqkv" and same and dtype == torch.float16:
            # (the compiler sums products of fp16 pairs by v_dot2_f32_f16 in one of the two and by fma in the other: fp32 roundings of
            # a row's sums, 2^-21 of its largest value, and what of them reaches the result's 11 bits)
            row = w.float().abs().view(windows, n, 3 * heads, 32).amax(-1, keepdim=True).expand(-1, -1, -1, 32).reshape(w.shape)
            off = x != w
            assert int(off.sum()) <= x.numel() * 2.0 ** -12, name
            assert ((x.float() - w.float()).abs() <= w.float().abs() * 2.0 ** -10 + row * 2.0 ** -20 + 2.0 ** -24).all(), name
        elif same or (name == "o" and windows * heads >= 512):
            assert torch.equal(x, w), name
        else:
            assert (x.float() - w.float()).norm() <= 2.0 ** -7 * w.float().norm(), name
    again = one()
    assert all(torch.equal(x, y) for x, y in zip(got, again))


class Given(torch.nn.Module):
    """In the place of a projection: its result."""

    def __init__(self, y):
        super().__init__()
        self.y = y

    def forward(self, x):
        return self.y


def _window_core_exact(mod, qkv, logit_scale, heads, mask=None):
    """Attention of a window block on its projection, in float64 tensor operations."""
    windows, n, dim = qkv.shape[0], qkv.shape[1], qkv.shape[2] // 3
    q, k, v = (t.view(windows, n, heads, dim // heads).transpose(1, 2).contiguous()
               for t in _cosine_exact(qkv.view(windows * n, -1), logit_scale, heads))
    bias = mod.q_bias_pos.double()[0].transpose(0, 1) @ mod.k_bias_pos.double()[0].permute(1, 2, 0).contiguous()
    logits = q @ k.transpose(-1, -2).contiguous() + bias
    o = torch.softmax(logits if mask is None else logits + mask[:, None], dim=-1) @ v
    return o.transpose(1, 2).reshape(windows, n, dim)


@pytest.mark.parametrize("dtype,autocast", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("param", [torch.float32, torch.bfloat16])
def test_window_block_under_autocast(gpu_device, monkeypatch, dtype, autocast, param):
    """Under torch.autocast the projection comes in 16 bits while norm, quotient, exponential and product are computed in
    fp32: output and the projection's gradient are no further from float64 than the tensor operations'."""
    torch.manual_seed(2)
    window, heads, hd, windows = 8, 4, 32, 16
    n, dim = window * window, heads * hd
    mod = modules.WindowAttentionCore(dim, window, heads, rank=8, dtype=dtype).to(gpu_device, param)
    mod.q_bias_pos, mod.k_bias_pos = mod.q_bias_pos.to(dtype), mod.k_bias_pos.to(dtype)
    x = torch.randn(windows, n, dim, device=gpu_device, dtype=param)
    dy = torch.randn(windows, n, dim, device=gpu_device, dtype=param)
    with torch.no_grad(), torch.autocast("cuda", dtype=autocast):
        qkv = mod.qkv(x)
    assert qkv.dtype == autocast
    qkv.requires_grad_(True)
    mod.qkv, mod.proj = Given(qkv), torch.nn.Identity()  # (the attention itself)

    def run():
        with torch.autocast("cuda", dtype=autocast):
            y = mod(x)
        return [y.detach().double(), torch.autograd.grad(y, qkv, dy)[0].double()]
    got = run()
    monkeypatch.setattr(interface, "_ext", None)
    ops = run()
    leaf = qkv.detach().double().requires_grad_(True)
    y = _window_core_exact(mod, leaf, mod.logit_scale.detach().flatten(), heads)
    exact = [y.detach(), torch.autograd.grad(y, leaf, dy.double())[0]]
    for name, g, o, w in zip(("y", "dqkv"), got, ops, exact):
        error = lambda t: float((t - w).norm() / w.norm())
        # (131072 and 393216 values with roundings of their own: the two errors are measured to less than 2 %)
        assert error(g) <= 1.05 * error(o), (name, error(g), error(o))


def _both_ways(monkeypatch, mod, x, mask):
    """Output and input gradient of the module from the one-pass kernels and from the tensor operations; an error in the
    place of a result that there is none of."""
    out = []
    for ext in (interface._extension(), None):
        with monkeypatch.context() as m:
            m.setattr(interface, "_ext", ext)
            try:
                y = mod(x, mask)
                out.append([y.detach().double(), torch.autograd.grad(y.double().square().sum(), x)[0].double()])
            except (RuntimeError, AssertionError) as e:
                out.append(e)
    return out


# windows of 16 tokens, 8 of them, 4 to an image; what expands to (4, 16, 16), then what does not
@pytest.mark.parametrize("shape,accepted", [
    ((4, 16, 16), True), ((4, 16, 1), True), ((4, 1, 16), True), ((4, 1, 1), True), ((8, 16, 1), True), ((1, 16, 16), True),
    ((1, 16), True), ((1, 1), True), ((1,), True), ((4, 16), False), ((3, 16, 16), False), ((4, 8, 16), False), ((4, 16, 8), False),
    ((16, 16, 16), False), ((4, 1, 16, 16), False)])
def test_window_masks_that_broadcast(gpu_device, monkeypatch, shape, accepted):
    torch.manual_seed(3)
    mod = modules.WindowAttentionCore(64, 4, 2, rank=8).to(gpu_device)
    x = torch.randn(8, 16, 64, device=gpu_device, requires_grad=True)
    mask = torch.randn(shape, device=gpu_device) * 2
    one, ops = _both_ways(monkeypatch, mod, x, mask)
    if not accepted:
        assert isinstance(one, Exception) and isinstance(ops, Exception)
        return
    for name, a, b in zip(("y", "dx"), one, ops):
        # (fp32 projection: q and k differ by the last bit where fp32 sums in another order fall on the other side of a
        # rounding, P and dS by 2^-9 relative; outputs rounded to bf16)
        assert (a - b).norm() <= 2.0 ** -7 * b.norm(), name


@pytest.mark.parametrize("what", ["float64", "float64 scale", "strided scale", "flat scale", "misaligned projection", "fp16 in bf16 out",
                                  "head dim 24", "rank 12"])
def test_window_block_takes_what_the_tensor_operations_take(gpu_device, monkeypatch, what):
    """Parameters and projections that the one-pass kernels have no form for, or not the obvious one."""
    torch.manual_seed(4)
    hd, rank = 24 if what == "head dim 24" else 32, 12 if what == "rank 12" else 8
    mod = modules.WindowAttentionCore(2 * hd, 4, 2, rank=rank).to(gpu_device)
    q_bias, k_bias = mod.q_bias_pos, mod.k_bias_pos
    mod = mod.to({"float64": torch.float64, "fp16 in bf16 out": torch.float16}.get(what, torch.float32))
    mod.q_bias_pos, mod.k_bias_pos = q_bias, k_bias  # (bf16 still)
    if what == "float64 scale":
        mod.logit_scale = torch.nn.Parameter(mod.logit_scale.double())
    if what == "strided scale":
        mod.logit_scale = torch.nn.Parameter(torch.tensor([[2.0, 9.0], [2.5, 9.0]], device=gpu_device)[:, :1, None])
        assert not mod.logit_scale.is_contiguous()
    if what == "flat scale":
        mod.logit_scale = torch.nn.Parameter(torch.tensor([2.0, 2.5], device=gpu_device))
    x = torch.randn(6, 16, 2 * hd, device=gpu_device, dtype=mod.qkv.weight.dtype, requires_grad=True)
    if what == "misaligned projection":
        store = torch.randn(6 * 16 * 6 * hd + 1, device=gpu_device)
        mod.qkv = Given(store.requires_grad_(True)[1:].view(6, 16, 6 * hd))
        assert mod.qkv.y.data_ptr() % 16
        x = x.detach()
    target = mod.qkv.y if isinstance(mod.qkv, Given) else x
    results = []
    for ext in (interface._extension(), None):
        with monkeypatch.context() as m:
            m.setattr(interface, "_ext", ext)
            y = mod(x)
            results.append([y.detach().double()] + [t.double() for t in torch.autograd.grad(y.double().square().sum(), [target, mod.logit_scale])])
    for name, a, b in zip(("y", "input", "scale"), *results):
        # (as test_window_masks_that_broadcast; the scale's gradient is a sum over all scores: as the module's other tests)
        assert (a - b).norm() <= (3e-2 if name == "scale" else 2.0 ** -7) * b.norm(), name


def _requested(fn):
    """fn(), and the bytes that it asked the allocator for."""
    torch.cuda.synchronize()
    before = torch.cuda.memory_stats()["requested_bytes.all.allocated"]
    out = fn()
    return out, torch.cuda.memory_stats()["requested_bytes.all.allocated"] - before


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("windows,window,heads,types", [(264, 16, 4, 0), (264, 12, 4, 4), (8, 16, 4, 2), (6, 8, 2, 0)])
def test_window_block_with_a_gradient_in_unaligned_rows(gpu_device, dtype, windows, window, heads, types):
    """The forward normalised q and k inside its kernel and kept neither, and the backward kernel that would do so again does not read these
    rows: the normalised rows are formed then, and the gradients are those of the same gradient in aligned rows."""
    torch.manual_seed(8)
    n, dim = window * window, 32 * heads
    mod = modules.WindowAttentionCore(dim, window, heads, rank=8, dtype=dtype).to(gpu_device, dtype)
    qkv = torch.randn(windows, n, 3 * dim, device=gpu_device).to(dtype).requires_grad_(True)
    mod.qkv, mod.proj = Given(qkv), torch.nn.Identity()
    x = torch.zeros(windows, n, dim, device=gpu_device, dtype=dtype)
    mask = (torch.rand(types, n, n, device=gpu_device) < 0.2).to(dtype) * -100.0 if types else None
    dy = torch.zeros(windows, n, dim + 8, device=gpu_device, dtype=dtype)[..., 4:dim + 4].copy_(torch.randn(windows, n, dim, device=gpu_device))
    assert dy.data_ptr() % 16
    y, asked = _requested(lambda: mod(x, mask))
    size = windows * n * dim * 2
    assert asked == size + windows * heads * n * 4  # (o and lse alone)
    gradients = lambda d: torch.autograd.grad(y, [qkv, mod.logit_scale], d, retain_graph=True)
    gradients(dy)
    want, few = _requested(lambda: gradients(dy.contiguous()))
    got, more = _requested(lambda: gradients(dy))
    assert more >= few - size + 2 * size  # (less the copy of dy, and q and k)
    for name, g, w in zip(("dqkv", "scale"), got, want):
        # other kernels with other orders of their sums, dq and dk rounded before the normalisation's part on both ways (the scale's
        # gradient is a sum over all scores: as the module's other tests)
        assert torch.isfinite(g).all() and (g.double() - w.double()).norm() <= (3e-2 if name == "scale" else 2.0 ** -7) * w.double().norm(), name


@pytest.mark.parametrize("dtype,param", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("window,heads,hd,windows,types", [(8, 2, 32, 6, 3), (7, 3, 128, 4, 0), (16, 8, 32, 64, 4), (12, 4, 32, 66, 6)])
def test_window_block_against_float64(gpu_device, monkeypatch, dtype, param, window, heads, hd, windows, types):
    """The module's attention on its projection, forward and backward, against float64, and beside the error that the tensor
    operations have there (64 x 8 windows of 256 and 66 x 4 of 144: one workgroup per window and head in the backward, masks
    that repeat over the images)."""
    torch.manual_seed(5)
    n, dim = window * window, heads * hd
    mod = modules.WindowAttentionCore(dim, window, heads, rank=8, dtype=dtype).to(gpu_device, param)
    mod.q_bias_pos, mod.k_bias_pos = mod.q_bias_pos.to(dtype), mod.k_bias_pos.to(dtype)
    qkv = torch.randn(windows, n, 3 * dim, device=gpu_device).to(param).requires_grad_(True)
    mod.qkv, mod.proj = Given(qkv), torch.nn.Identity()
    x = torch.zeros(windows, n, dim, device=gpu_device, dtype=param)
    dy = torch.randn(windows, n, dim, device=gpu_device).to(param)
    mask = (torch.rand(types, n, n, device=gpu_device) < 0.2).float() * -100.0 if types else None

    def run():
        y = mod(x, mask)
        return [y.detach()] + list(torch.autograd.grad(y, [qkv, mod.logit_scale], dy))
    got = run()
    monkeypatch.setattr(interface, "_ext", None)
    ops = run()
    leaf, scale = qkv.detach().double().requires_grad_(True), mod.logit_scale.detach().double().flatten().requires_grad_(True)
    exact = [[], [], 0]
    for at in range(0, windows, 8):  # (dense)
        part = slice(at, min(at + 8, windows))
        m = None if mask is None else mask[torch.arange(at, part.stop, device=gpu_device) % types].double()
        y = _window_core_exact(mod, leaf[part], scale, heads, m)
        g = torch.autograd.grad(y, [leaf, scale], dy[part].double())
        exact[0].append(y.detach())
        exact[1].append(g[0][part])
        exact[2] = exact[2] + g[1]
    exact = [torch.cat(exact[0]), torch.cat(exact[1]), exact[2].view_as(mod.logit_scale)]
    for name, g, o, w in zip(("y", "dqkv", "dscale"), got, ops, exact):
        error = lambda t: float((t.double() - w).norm() / w.norm())
        # y and dqkv: independent roundings of thousands of values, the two errors are measured to a percent or two; dscale:
        # `heads` values, each the rest of a sum that cancels, where two errors of one size differ by a factor
        assert torch.isfinite(g).all() and error(g) <= (3 if name == "dscale" else 1.05) * error(o), (name, error(g), error(o))


# tiles of 256 and 128 and their ragged edges; fewer stages of 32 tokens than the pipeline is deep, a ragged last one, one
# share and many; rows inside wider tensors
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k", [(1, 8, 8), (31, 264, 136), (64, 128, 384), (97, 248, 256), (129, 256, 504), (300, 1000, 248), (4100, 384, 128),
                                        (20000, 768, 256)])
def test_weight_gradient(gpu_device, dtype, tokens, n, k):
    lib = _lib.load()
    g = torch.Generator(device=gpu_device).manual_seed(tokens)
    dy_all = torch.randn(tokens, n + 24, generator=g, device=gpu_device).to(dtype)
    x_all = torch.randn(tokens, k + 8, generator=g, device=gpu_device).to(dtype)
    dy, x = dy_all[:, 8:8 + n], x_all[:, :k]
    # (nothing outside the rows may count: what lies beside them is not finite)
    dy_all[:, :8] = dy_all[:, 8 + n:] = x_all[:, k:] = float("nan")
    for bias in (True, False):
        dw = torch.full((n, k), float("nan"), device=gpu_device, dtype=dtype)
        db = torch.full((n,), float("nan"), device=gpu_device, dtype=dtype)
        scratch = torch.full((lib.fb_weight_grad_workspace_bytes(tokens, n, k, bias) // 4,), float("nan"), device=gpu_device)
        _lib.check_status(lib.fb_weight_grad(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), dw.data_ptr(), db.data_ptr() if bias else None,
                                             scratch.data_ptr(), CODES[dtype], tokens, n, k, interface._stream()))
        # rounded once to 8 / 11 significant bits: at most half a unit of the last place of every element, whose sums in
        # 32 bits are far closer
        bound = 1.01 * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
        want = dy.double().t().contiguous() @ x.double()
        assert (dw.double() - want).norm() <= bound * want.norm()
        if bias:
            assert (db.double() - dy.double().sum(0)).norm() <= bound * dy.double().sum(0).norm()


# one step of 64 columns, fewer steps than the pipeline has stages, and many; the three tiles (128 x 64 up to 512 of them, 128 x 128
# where up to 256 of them are enough for more than 256 small ones, 256 x 128) with ragged edges along tokens and channels; one to three weights of different sizes; rows inside a wider tensor
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k", [(1, (8,), 64), (63, (136, 64), 128), (65, (128, 8, 264), 192), (300, (1000, 72, 512), 320),
                                        (1500, (1000, 1032, 264), 192), (4099, (520, 136, 1288), 128), (2600, (776, 1032, 776), 1600)])
def test_projections(gpu_device, dtype, tokens, n, k):
    lib = _lib.load()
    g = torch.Generator(device=gpu_device).manual_seed(tokens)
    x_all = torch.randn(tokens, k + 24, generator=g, device=gpu_device).to(dtype)
    x = x_all[:, 8:8 + k]
    x_all[:, :8] = x_all[:, 8 + k:] = float("nan")  # (nothing outside the rows may count)
    w = [torch.randn(m, k, generator=g, device=gpu_device).to(dtype) for m in n]
    whole = [torch.full((tokens * m + 64,), 7.0, device=gpu_device, dtype=dtype) for m in n]  # (nor be written)
    y = [t[:tokens * m].view(tokens, m) for t, m in zip(whole, n)]
    pointers = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    sizes = (ctypes.c_int * len(n))(*n)
    _lib.check_status(lib.fb_project(x.data_ptr(), x.stride(0), pointers(w), pointers(y), sizes, len(n), CODES[dtype], tokens, k, interface._stream()))
    # rounded once to 8 / 11 significant bits: at most half a unit of the last place of every element, plus its sum in 32 bits
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for got, weight, full, m in zip(y, w, whole, n):
        want = x.double() @ weight.double().t().contiguous()
        size = x.double().abs() @ weight.double().abs().t().contiguous()
        assert ((got.double() - want).abs() <= 1.01 * unit * want.abs() + k * 2.0 ** -24 * size).all()
        assert (full[tokens * m:] == 7.0).all()
    assert lib.fb_project(x.data_ptr(), x.stride(0), pointers(w), pointers(y), sizes, len(n), CODES[dtype], tokens, k - 8, interface._stream()) != 0


# one step of 64 columns, fewer steps than a tile has stages, and many; tiles of 128 and of 256 channels, one and several a workgroup, results
# through the caches and past them (200 MiB and more), ragged edges along tokens and channels, a bias on 4 bytes, rows inside a wider tensor
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k", [(1, 8, 64), (257, 136, 128), (300, 1000, 1600), (9001, 1000, 192), (33000, 512, 64), (70144, 512, 128),
                                        (140001, 264, 64), (20001, 776, 512), (202001, 520, 64), (137000, 776, 128)])
def test_linear(gpu_device, dtype, tokens, n, k):
    lib = _lib.load()
    g = torch.Generator(device=gpu_device).manual_seed(tokens)
    x_all = torch.randn(tokens, k + 24, generator=g, device=gpu_device).to(dtype)
    x = x_all[:, 8:8 + k]
    x_all[:, :8] = x_all[:, 8 + k:] = float("nan")  # (nothing outside the rows may count)
    w = torch.randn(n, k, generator=g, device=gpu_device).to(dtype)
    bias = torch.randn(n + 2, generator=g, device=gpu_device).to(dtype)[2:]
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for b in (bias, None):
        whole = torch.full((tokens * n + 64,), 7.0, device=gpu_device, dtype=dtype)  # (nor be written)
        y = whole[:tokens * n].view(tokens, n)
        _lib.check_status(lib.fb_linear(x.data_ptr(), x.stride(0), w.data_ptr(), None if b is None else b.data_ptr(), y.data_ptr(), CODES[dtype], tokens,
                                        n, k, interface._stream()))
        for rows in torch.arange(tokens, device=gpu_device).split(32768):
            part = x[rows].double()
            want = part @ w.double().t().contiguous() + (0 if b is None else b.double())
            size = part.abs() @ w.double().abs().t().contiguous() + (0 if b is None else b.double().abs())
            # rounded once: at most half a unit of the last place of every element, plus its sum in 32 bits
            assert ((y[rows].double() - want).abs() <= 1.01 * unit * want.abs() + (k + 1) * 2.0 ** -24 * size).all()
        assert (whole[tokens * n:] == 7.0).all()
    assert lib.fb_linear(x.data_ptr(), x.stride(0), w.data_ptr(), None, y.data_ptr(), CODES[dtype], tokens, n, k - 8, interface._stream()) != 0


@pytest.mark.parametrize("rows,cols", [(64, 64), (512, 1536), (192, 128)])
def test_transpose(gpu_device, rows, cols):
    lib = _lib.load()
    x = torch.randint(0, 1 << 15, (rows, cols), device=gpu_device, dtype=torch.int16)
    whole = torch.full((rows * cols + 64,), 7, device=gpu_device, dtype=torch.int16)
    _lib.check_status(lib.fb_transpose(x.data_ptr(), whole.data_ptr(), rows, cols, interface._stream()))
    assert torch.equal(whole[:rows * cols].view(cols, rows), x.t()) and (whole[rows * cols:] == 7).all()
    assert lib.fb_transpose(x.data_ptr(), whole.data_ptr(), rows - 8, cols, interface._stream()) != 0


@pytest.mark.parametrize("n,bias", [(384, False), (128, True)])
def test_projection_of_many_tokens_takes_the_product_and_leaves_the_rest(gpu_device, n, bias):
    torch.manual_seed(4)
    layer = torch.nn.Linear(128, n, bias=bias).to(gpu_device, torch.bfloat16)
    x = torch.randn(1025, 128, 128, device=gpu_device, dtype=torch.bfloat16)
    ext, many = interface._extension(), 1.01 * 2.0 ** -8
    want = layer(x).double()
    with torch.no_grad():
        got = ext.linear(x, layer.weight, layer.bias)
        assert got is not None and (got.double() - want).norm() <= 2 * many * want.norm()
        assert torch.equal(got, modules._project(layer, x))
        # few tokens, rows that are not contiguous, long rows and other types are left to the tensor library
        assert ext.linear(x[:2], layer.weight, layer.bias) is None and ext.linear(x.transpose(0, 1), layer.weight, layer.bias) is None
        assert ext.linear(x.view(-1, 1024), torch.zeros(n, 1024, device=gpu_device, dtype=torch.bfloat16), layer.bias) is None
        assert ext.linear(x.float(), layer.weight.float(), None) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert ext.linear(x, layer.weight, layer.bias) is None
    y = modules._project(layer, x)
    assert "LinearFn" in y.grad_fn.name() and torch.equal(y.detach(), got)
    # the input's gradient, by the same kernel, from rows of a wider tensor and from rows that it has to copy
    x.requires_grad_(True)
    y = modules._project(layer, x)
    wide = torch.randn(1025, 128, n + 8, device=gpu_device, dtype=torch.bfloat16)
    for dy in (wide[..., :n].contiguous(), wide[..., 8:], wide[..., 4:n + 4], wide[:1, :1, :n].expand(1025, 128, n)):
        (dx,) = torch.autograd.grad(y, [x], dy, retain_graph=True)
        want = dy.double() @ layer.weight.double()
        assert dx.shape == x.shape and (dx.double() - want).norm() <= many * want.norm()


# few tokens, whose input gradient is left to the tensor library, and many, which the library's product takes
@pytest.mark.parametrize("tokens", [20000, 110000])
def test_projection_backward_copies_a_gradient_once(gpu_device, tokens):
    """A gradient in rows that the kernels do not read is copied where one of them takes it, and once for both."""
    torch.manual_seed(7)
    layer = torch.nn.Linear(256, 256).to(gpu_device, torch.bfloat16)
    x = torch.randn(tokens, 256, device=gpu_device, dtype=torch.bfloat16, requires_grad=True)
    wide = torch.randn(tokens, 256 + 8, device=gpu_device, dtype=torch.bfloat16)
    aligned, shifted = wide[:, :256], wide[:, 4:260]
    assert shifted.data_ptr() % 16
    y = modules._project(layer, x)
    assert "LinearFn" in y.grad_fn.name()

    def allocated(dy, leaves):
        for _ in range(2):  # (the first call may set up the tensor library)
            torch.cuda.synchronize()
            before = torch.cuda.memory_stats()["requested_bytes.all.allocated"]
            grads = torch.autograd.grad(y, leaves, dy, retain_graph=True)
            bytes_ = torch.cuda.memory_stats()["requested_bytes.all.allocated"] - before
        return bytes_, grads
    copy = tokens * 256 * 2
    for leaves, copies in (([x], 1 if tokens >= 100000 else 0), ([layer.weight, layer.bias], 1), ([x, layer.weight, layer.bias], 1)):
        few, _ = allocated(aligned, leaves)
        more, grads = allocated(shifted, leaves)
        assert more - few == copies * copy, (len(leaves), (more - few) / copy)
        d = shifted.double()
        for name, g in zip(("weight", "bias") if len(leaves) == 2 else ("x", "weight", "bias"), grads):
            want = d @ layer.weight.double() if name == "x" else d.t().contiguous() @ x.detach().double() if name == "weight" else d.sum(0)
            assert (g.double() - want).norm() <= 1.01 * 2.0 ** -8 * want.norm(), name


def test_block_projections_take_the_kernel_and_leave_the_rest(gpu_device):
    torch.manual_seed(3)
    layers = [torch.nn.Linear(128, 136, bias=False).to(gpu_device, torch.bfloat16) for _ in range(3)]
    x = torch.randn(5, 130, 128, device=gpu_device, dtype=torch.bfloat16)
    weights = [layer.weight for layer in layers]
    exact = [x.double() @ w.detach().double().t().contiguous() for w in weights]
    with torch.no_grad():
        assert len(interface._extension().project(x, weights)) == 3
        for got, want in zip(modules._project_all(layers, x), exact):
            assert got.shape == want.shape and (got.double() - want).norm() <= 1.01 * 2.0 ** -8 * want.norm()
        # no rows of 16-byte aligned chunks, another type, nothing to do, more work than the kernel is ahead for: not taken
        assert not interface._extension().project(x.transpose(0, 1), weights) and not interface._extension().project(x[..., :72], weights)
        assert not interface._extension().project(x.float(), weights) and not interface._extension().project(x[:0], weights)
        big = torch.empty(1, 256 * 128 + 1, 128, device=gpu_device, dtype=torch.bfloat16)
        assert not interface._extension().project(big, weights) and interface._extension().project(big[:, 1:], weights)
        # (a sum of many columns is not split)
        row, narrow = torch.randn(1, 3, 8192, device=gpu_device, dtype=torch.bfloat16), [torch.randn(64, 8192, device=gpu_device, dtype=torch.bfloat16)] * 3
        short = row[..., :4096].contiguous(), [w[:, :4096].contiguous() for w in narrow]
        assert not interface._extension().project(row, narrow) and len(interface._extension().project(*short)) == 3
        seen = []
        handle = layers[1].register_forward_hook(lambda *a: seen.append(1))
        modules._project_all(layers, x)
        handle.remove()
        assert seen
        with torch.autocast("cuda", dtype=torch.float16):
            assert all(t.dtype == torch.float16 for t in modules._project_all(layers, x))
        per_sample = torch.func.vmap(lambda t: modules._project_all(layers, t)[2])(x)
        assert (per_sample.double() - exact[2]).norm() <= 1.01 * 2.0 ** -8 * exact[2].norm()
    assert all(t.grad_fn is not None for t in modules._project_all(layers, x))


def test_projection_takes_the_kernel_and_leaves_the_rest(gpu_device):
    torch.manual_seed(2)
    layer = torch.nn.Linear(128, 136).to(gpu_device, torch.bfloat16)
    x = torch.randn(5, 1300, 128, device=gpu_device, dtype=torch.bfloat16, requires_grad=True)
    leaves = [x, layer.weight, layer.bias]
    dy = torch.randn(5, 1300, 136, device=gpu_device, dtype=torch.bfloat16)
    y, want_y = modules._project(layer, x), torch.nn.functional.linear(x, layer.weight, layer.bias)
    assert "LinearFn" in type(y.grad_fn).__name__ + y.grad_fn.name() and torch.equal(y, want_y)
    for out in (dy, dy[:1, :1].expand(5, 1300, 136), dy.transpose(0, 1).contiguous().transpose(0, 1)):
        got = torch.autograd.grad(y, leaves, out, retain_graph=True)
        want = torch.autograd.grad(want_y, leaves, out, retain_graph=True)
        for g, w in zip(got, want):  # (the same products, rounded once each: two units of the last place in norm)
            assert g.shape == w.shape and g.dtype == w.dtype and (g.float() - w.float()).norm() <= 2.0 ** -7 * w.float().norm()
    # a gradient of a gradient is that of the tensor operations
    for out in (y, want_y):
        (gw,) = torch.autograd.grad((out.float() ** 2).sum(), [layer.weight], create_graph=True)
        out.second = torch.autograd.grad(gw.float().square().sum(), [x], retain_graph=True)[0].float()
    assert (y.second - want_y.second).norm() <= 2e-2 * want_y.second.norm()
    # what else looks at or replaces the operation still does
    seen = []
    handle = layer.register_forward_hook(lambda *a: seen.append(1))
    assert "LinearFn" not in modules._project(layer, x).grad_fn.name() and seen
    handle.remove()
    with torch.no_grad():
        assert modules._project(layer, x).grad_fn is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert modules._project(layer, x).dtype == torch.float16
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        assert torch.autograd.forward_ad.unpack_dual(modules._project(layer, dual)).tangent is not None
    per_sample = torch.func.vmap(lambda t: modules._project(layer, t))(x)
    assert torch.allclose(per_sample.float(), want_y.float(), atol=2e-2)


def _projection_case(dev):
    torch.manual_seed(6)
    layer = torch.nn.Linear(128, 136).to(dev, torch.bfloat16)
    x = torch.randn(5, 1300, 128, device=dev, dtype=torch.bfloat16, requires_grad=True)
    return layer, x, torch.randn(3, 5, 1300, 136, device=dev, dtype=torch.bfloat16)


@pytest.mark.parametrize("what", ["batched gradients", "counted operations", "autocast"])
def test_projection_backward_that_something_watches(gpu_device, what):
    """What wraps the gradients or looks at the operations of a backward, around a forward that took the kernel's route."""
    from torch.utils.flop_counter import FlopCounterMode
    layer, x, dy = _projection_case(gpu_device)
    leaves = [layer.weight, layer.bias, x]
    results = []
    for y in (modules._project(layer, x), layer(x)):
        if what == "batched gradients":
            results.append(torch.autograd.grad(y, leaves, dy, is_grads_batched=True))
        elif what == "counted operations":
            with FlopCounterMode(display=False) as counter:
                torch.autograd.grad(y, leaves, dy[0])
            results.append([torch.tensor(float(counter.get_total_flops()))])
        else:
            with torch.autocast("cuda", dtype=torch.float16):
                results.append(torch.autograd.grad(y, leaves, dy[0]))
    for got, want in zip(*results):  # (the same products, rounded once each: two units of the last place in norm)
        assert got.shape == want.shape and got.dtype == want.dtype and (got.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


def test_projection_of_an_input_without_gradient_keeps_no_weight(gpu_device):
    """Nothing of the backward needs the weight then: it may change before it (an optimizer's step between two losses)."""
    layer, x, dy = _projection_case(gpu_device)
    x = x.detach()
    want = torch.autograd.grad(layer(x), [layer.weight, layer.bias], dy[0])
    y = modules._project(layer, x)
    assert "LinearFn" in y.grad_fn.name()
    with torch.no_grad():
        layer.weight.mul_(0.5)
    for got, w in zip(torch.autograd.grad(y, [layer.weight, layer.bias], dy[0]), want):
        assert (got.float() - w.float()).norm() <= 2.0 ** -7 * w.float().norm()
    y = modules._project(layer, x.requires_grad_(True))
    with torch.no_grad():
        layer.weight.mul_(0.5)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, [x], dy[0])


class Watching(torch.Tensor):
    """A tensor type that sees operations without a dispatch key of its own."""
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(func)
        return super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.parametrize("what", ["input", "weight"])
@pytest.mark.parametrize("grad", [True, False])
def test_projections_of_tensor_subclasses(gpu_device, what, grad):
    """An input or a weight of a type that overrides operations sees its projection, as F.linear shows it."""
    torch.manual_seed(7)
    layers = [torch.nn.Linear(128, 136, bias=False).to(gpu_device, torch.bfloat16) for _ in range(3)]
    x = torch.randn(5, 1300, 128, device=gpu_device, dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad):
        want = modules._project_all(layers, x)
        if what == "input":
            x = x.as_subclass(Watching)
        else:
            layers[1].weight = torch.nn.Parameter(layers[1].weight.detach().as_subclass(Watching))
        Watching.seen.clear()
        got = modules._project_all(layers, x)
    assert Watching.seen.count(torch.nn.functional.linear) == (3 if what == "input" else 1)
    for i, (a, b) in enumerate(zip(got, want)):
        assert type(a) is (Watching if what == "input" or i == 1 else torch.Tensor)
        assert (a.as_subclass(torch.Tensor).float() - b.float()).norm() <= 2.0 ** -7 * b.float().norm()
