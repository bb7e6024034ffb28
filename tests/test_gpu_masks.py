"""Additive masks through the C ABI: masks that repeat over the batch, and parameter blocks from before that."""
import ctypes

import pytest
import torch

from _util import make_inputs
from flashbias_amd import _lib
from flashbias_amd.interface import _params, _stream, _tensor

pytestmark = pytest.mark.gpu


def _call(inputs, mask, do, scale=None, mask_batches=0, mask_strides=None, group=1, grads=True, bwd="fb_bwd", old_block=None):
    """o, lse and the gradients of one forward and backward call.  mask_strides: (batch, head) element strides of the mask
    where they are not those of the tensor; old_block: the left-over value at the end of a version 3 block."""
    q, k, v, qb, kb = inputs
    lib = _lib.load()
    p, keep = _params(q, k, v, qb, kb, mask if mask_strides is None else mask[:1, :1].expand(q.shape[0], *mask.shape[1:]), False, scale)
    if mask_strides is not None:
        p.mask = _lib.FbTensor(mask.data_ptr(), *mask_strides, p.mask.stride_s)
    p.mask_batches = mask_batches
    rows = -(-p.B // group)
    nan = lambda *shape: torch.full(shape, float("nan"), device=q.device, dtype=q.dtype)
    out = dict(o=nan(*q.shape), lse=torch.empty((p.B, p.H, p.Lq), device=q.device, dtype=torch.float32), dq=nan(*q.shape), dk=nan(*k.shape),
               dv=nan(*v.shape))
    scratch = torch.empty(lib.fb_bwd_workspace_bytes(p) // 4, device=q.device, dtype=torch.float32)
    p.o, p.lse, p.dout, p.delta = _tensor(out["o"]), out["lse"].data_ptr(), _tensor(do), scratch.data_ptr()
    p.dq, p.dk, p.dv = _tensor(out["dq"]), _tensor(out["dk"]), _tensor(out["dv"])
    if p.r and grads:
        out["dq_bias"], out["dk_bias"] = nan(rows, p.Lq, p.H, p.r), nan(rows, p.Lk, p.H, p.r)
        p.dq_bias, p.dk_bias = _tensor(out["dq_bias"]), _tensor(out["dk_bias"])
    p.bias_grad_group = group if p.r else 0
    block = p
    if old_block is not None:
        p.size, p.reserved0 = _lib.FbParams.mask_batches.offset, old_block
        buf = (ctypes.c_char * p.size)()
        ctypes.memmove(buf, ctypes.byref(p), p.size)
        block = ctypes.cast(buf, ctypes.POINTER(_lib.FbParams))
    _lib.check_status(lib.fb_fwd(block, _stream()))
    for fn in ([bwd] if isinstance(bwd, str) else bwd):
        _lib.check_status(getattr(lib, fn)(block, _stream()))
    torch.cuda.synchronize()
    del keep
    return out


@pytest.mark.parametrize("left_over", [1, 3, -1])
def test_a_block_of_version_3_has_a_mask_per_batch_entry(gpu_device, left_over):
    """What lies behind bias_grad_group in a version 3 block is padding: it does not become mask_batches."""
    q, k, v, qb, kb, do = [t.to(gpu_device) for t in make_inputs(5, 70, 90, 2, 32, 8, torch.bfloat16, seed=6)]
    mask = torch.randn(5, 1, 70, 90, generator=torch.Generator().manual_seed(7)).bfloat16().to(gpu_device)
    want = _call((q, k, v, qb, kb), mask, do)
    for bwd in ("fb_bwd", "fb_bwd_static"):
        got = _call((q, k, v, qb, kb), mask, do, bwd=bwd, old_block=left_over)
        for name in want:
            assert torch.equal(got[name], want[name]), name
