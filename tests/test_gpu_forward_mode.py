"""What the operator cannot differentiate it refuses: forward-mode derivatives and function transforms, also where no
argument requires a gradient and the call makes no graph node."""
import pytest
import torch
import torch.autograd.forward_ad as fwad

from _util import make_inputs
from flashbias_amd import flash_bias_func, interface, modules

pytestmark = pytest.mark.gpu

NAMES = ["q", "k", "v", "q_bias", "k_bias", "mask"]


def _args(dev, r, mask):
    q, k, v, qb, kb, _ = make_inputs(1, 40, 40, 2, 32, r, torch.bfloat16, seed=9)
    m = {"none": None, "vector": torch.zeros(1, 1, 1, 40, dtype=torch.bfloat16), "matrix": torch.zeros(1, 1, 40, 40, dtype=torch.bfloat16)}[mask]
    return [None if t is None else t.to(dev) for t in (q, k, v, qb, kb, m)]


# rank 8 without a vector mask goes straight to the extension, rank 4 and vector masks through the preparations
@pytest.mark.parametrize("r,mask,folded", [(8, "none", False), (8, "matrix", False), (8, "vector", False), (8, "vector", True), (4, "none", False),
                                           (0, "none", False)])
@pytest.mark.parametrize("grad_enabled", [True, False])
def test_forward_mode_derivatives_are_refused(gpu_device, monkeypatch, r, mask, grad_enabled, folded):
    assert interface._extension() is not None
    if folded:
        monkeypatch.setattr(interface, "_FOLD_MIN_PAIRS", 1)
    args = _args(gpu_device, r, mask)
    with torch.set_grad_enabled(grad_enabled):
        assert flash_bias_func(*args, False, None).isfinite().all()
        for i, name in enumerate(NAMES):
            if args[i] is None:
                continue
            with fwad.dual_level():
                duals = list(args)
                duals[i] = fwad.make_dual(args[i], torch.ones_like(args[i]))
                with pytest.raises((RuntimeError, NotImplementedError), match="jvp is not implemented"):
                    flash_bias_func(*duals, False, None)
            # the tangent belongs to the dual, not to the tensor: afterwards the same call is taken again
            assert flash_bias_func(*args, False, None).isfinite().all(), name


def test_function_transforms_are_refused(gpu_device):
    q, k, v, qb, kb, _ = _args(gpu_device, 8, "none")
    call = lambda x: flash_bias_func(x, k, v, qb, kb, None, False, None)
    with torch.no_grad():
        want = call(q)
        for transformed in (lambda: torch.func.jvp(call, (q,), (torch.ones_like(q),)),
                            lambda: torch.func.vmap(call)(q[None]),
                            # nothing the operator sees is wrapped here
                            lambda: torch.func.vmap(lambda x: x + call(q))(q[None])):
            with pytest.raises(RuntimeError):
                transformed()
        assert torch.equal(call(q), want)


@pytest.mark.parametrize("which", ["alibi", "window"])
def test_modules_refuse_forward_mode(gpu_device, which):
    if which == "alibi":
        mod, x = modules.AttentionWithALiBiBias(64, 2, 32), torch.randn(1, 40, 64)
    else:
        mod, x = modules.WindowAttentionCore(64, 8, 2, rank=8), torch.randn(2, 64, 64)
    mod, x = mod.to(gpu_device).requires_grad_(False), x.to(gpu_device)
    with torch.no_grad(), fwad.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError), match="jvp is not implemented"):
            mod(fwad.make_dual(x, torch.ones_like(x)))
