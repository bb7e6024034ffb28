"""The one-pass kernels of the module drop-ins (csrc/fb_cosine.hip, the ALiBi factor builder) against the tensor
operations they replace."""
import pytest
import torch

from flashbias_amd import factors, interface, modules

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
    # q and k have the same bits on both ways; what is left is the backward's own rounding (2^-8 per product of
    # bf16 tensor operations, of which the fused pass has fewer) and the summation orders
    bound = 3e-2
    for name, g, w in zip(["y", "x"] + [k for k, _ in mod.named_parameters()], got, want):
        assert torch.isfinite(g).all() and g.shape == w.shape and g.dtype == w.dtype, name
        if w.float().abs().max() == 0:
            assert g.abs().max() == 0, name
        else:
            assert (g.float() - w.float()).norm() <= bound * w.float().norm(), name
    assert got[2].flatten()[0] == 0
