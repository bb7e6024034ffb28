"""Additive masks through the C ABI: masks that repeat over the batch, and parameter blocks from before that."""
import ctypes

import pytest
import torch

from _util import GRAD_TOL, O_TOL, errors, make_inputs, oracle
from flashbias_amd import _lib
from flashbias_amd.interface import _params, _stream, _tensor

pytestmark = pytest.mark.gpu


def _call(inputs, mask, do, scale=None, mask_batches=0, group=1, grads=True, bwd="fb_bwd", old_block=None):
    """o, lse and the gradients of one forward and backward call.  mask_batches = n: the mask has n batch entries, which
    repeat; old_block: the left-over value at the end of a version 3 block."""
    q, k, v, qb, kb = inputs
    lib = _lib.load()
    at = torch.arange(q.shape[0], device=q.device) % mask.shape[0]
    p, keep = _params(q, k, v, qb, kb, mask[at] if mask_batches else mask, False, scale)
    if mask_batches:
        p.mask = _lib.FbTensor(mask.data_ptr(), mask.stride(0), mask.stride(1) if mask.shape[1] == q.shape[2] else 0, p.mask.stride_s)
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


# (dtype, B, H, Lq, Lk, d, r, mask rows, mask per head, masks, mask dtype, batch entries per factor gradient, factor gradients)
REPEATING = [
    # the window backward: grids that fill the chip, a batch that the masks do not divide, a mask per head, groups of entries,
    # several entries per workgroup without groups, constant factors
    (torch.bfloat16, 66, 4, 256, 256, 32, 16, "matrix", False, 4, None, 1, True),
    (torch.float16, 130, 4, 144, 200, 32, 32, "matrix", True, 7, None, 2, True),
    (torch.bfloat16, 66, 4, 100, 130, 32, 0, "vector", True, 5, None, 1, True),
    (torch.float16, 520, 4, 64, 64, 32, 8, "vector", False, 3, None, 8, True),
    (torch.bfloat16, 1101, 4, 160, 129, 32, 8, "matrix", False, 64, None, 1, False),
    # the general kernels and those of large head dims; more masks than batch entries
    (torch.bfloat16, 5, 3, 70, 90, 32, 8, "matrix", True, 2, None, 1, True),
    (torch.bfloat16, 5, 2, 96, 72, 32, 16, "matrix", False, 3, torch.float32, 1, True),
    (torch.bfloat16, 3, 2, 64, 64, 32, 8, "vector", False, 5, torch.float32, 1, True),
    (torch.float16, 5, 2, 96, 150, 64, 16, "vector", False, 3, None, 1, True),
    (torch.bfloat16, 5, 2, 64, 190, 128, 16, "vector", True, 2, None, 1, True),
    (torch.bfloat16, 3, 2, 130, 97, 128, 8, "matrix", False, 2, None, 1, True),
    (torch.bfloat16, 3, 1, 33, 41, 20, 5, "matrix", False, 2, None, 1, True),
]


@pytest.mark.parametrize("dtype,B,H,Lq,Lk,d,r,kind,per_head,masks,mdtype,group,grads", REPEATING)
def test_repeating_masks(gpu_device, dtype, B, H, Lq, Lk, d, r, kind, per_head, masks, mdtype, group, grads):
    """fb_params.mask_batches = n: batch entry b takes mask b % n.  The same bits as the masks written out for every batch
    entry, from fb_bwd and from its phases; and attention under those masks."""
    shared = group > 1
    cpu = make_inputs(B, Lq, Lk, H, d, r, dtype, seed=B + Lk, bq=(shared, False), bk=(shared, False))
    q, k, v, qb, kb, do = [None if t is None else t.to(gpu_device) for t in cpu]
    g = torch.Generator().manual_seed(8)
    mask = torch.randn(masks, H if per_head else 1, Lq if kind == "matrix" else 1, Lk, generator=g) * 2
    mask[..., Lk - Lk // 5:] = -100.0
    mask = mask.to(mdtype or dtype)
    dev_mask = mask.to(gpu_device)
    at = torch.arange(B) % masks
    first = None
    for bwd in ("fb_bwd", ("fb_bwd_preprocess", "fb_bwd_dkv", "fb_bwd_dq")):
        got = _call((q, k, v, qb, kb), dev_mask, do, mask_batches=masks, group=group, grads=grads, bwd=bwd)
        want = _call((q, k, v, qb, kb), dev_mask[at.to(gpu_device)], do, group=group, grads=grads, bwd=bwd)
        for name in want:
            assert torch.isfinite(got[name]).all() and torch.equal(got[name], want[name]), (name, bwd)
        first = first or got
    few = slice(0, min(B, 2 * masks + 1))  # (the oracle is dense)
    ref = oracle(*[t[few] if t is not None and t.shape[0] == B else t for t in cpu[:5]], mask[at[few]], False, None, cpu[5][few])
    for name, want in zip(("o", "dq", "dk", "dv"), (ref[0],) + tuple(ref[2:5])):
        err, rel = errors(first[name][few].float().cpu(), want)
        assert (err <= O_TOL[dtype] if name == "o" else rel <= GRAD_TOL), (name, err, rel)
