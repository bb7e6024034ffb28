"""The calls that performance is measured on: what users of the operator and of the two modules have them do.

A case is one pass: a forward (inference, gradients off), or a forward and a backward as a training step makes them
(``"grad"``: ``"inputs"`` for constant factors, whose gradients nobody asks for, ``"all"`` for learned ones).
Sizes are those of the benchmark configurations, of ``bench.py`` and of the reference's applications, from calls of a
few microseconds to the largest, with lengths that no tile divides among them.

``listed()`` are the ones looked at one by one, ``draw()`` takes others from the same ranges."""
import math

import torch

from flashbias_amd import factors, flash_bias_func, modules

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _op(name, B, H, Lq, Lk, d, r, bias, dtype="bf16", causal=False, mask="none", grad="none"):
    c = dict(kind="op", B=B, H=H, Lq=Lq, Lk=Lk, d=d, r=r, bias=bias, dtype=dtype, causal=causal, mask=mask, grad=grad)
    return dict(c, name=name) if name else c


def _alibi_block(name, B, L, H, d, grad):
    c = dict(kind="alibi block", B=B, L=L, H=H, d=d, grad=grad)
    return dict(c, name=name) if name else c


def _window_block(name, images, side, window, H, shifted, grad):
    """`images` feature maps of side x side windows of window x window tokens, H heads of 32 channels."""
    c = dict(kind="window block", images=images, side=side, window=window, H=H, shifted=shifted, grad=grad)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one inference call on the shortest sequences of the benchmark sweep: latency and launches
        _op("call 256", 2, 4, 256, 256, 32, 8, "learned"),
        # a training step at the sweep's configured lengths: short ...
        _op("step 1024", 2, 4, 1024, 1024, 32, 8, "learned", grad="all"),
        # ... and the longest, the headline of the benchmark
        _op("step 16384", 2, 4, 16384, 16384, 32, 8, "learned", grad="all"),
        # causal language model with ALiBi as constant rank-2 factors: training step
        _op("alibi step 4096", 1, 50, 4096, 4096, 32, 2, "alibi", causal=True, grad="inputs"),
        # the module around it, prefill of a prompt of no round length
        _alibi_block("alibi block prefill 1500", 1, 1500, 50, 32, "none"),
        # Swin-V2 windows with the SVD factors of the relative position table, shared by all windows: training step
        _op("swin step 4096 x 256", 4096, 16, 256, 256, 32, 16, "table", grad="inputs"),
        # the module around it in a shifted-window block: 16 images of 8 x 8 windows, training step
        _window_block("swin shifted block", 16, 8, 16, 16, True, "all"),
        # neural PDE solver over a point cloud of 32186 points, constant distance factors shared by the heads
        _op("pde step 32186", 1, 8, 32186, 32186, 32, 8, "distance", grad="inputs"),
        # triangle attention over 768 tokens with a learned pair bias shared by the rows: training step
        _op("pair step 768", 768, 4, 768, 768, 32, 32, "pair", grad="all"),
        # the same at inference on a padded crop of 384 tokens
        _op("pair padded 384", 384, 4, 384, 384, 32, 32, "pair", mask="padding"),
        # causal language model with heads of 128 channels and a learned bias: training step
        _op("causal d128 step 4096", 4, 32, 4096, 4096, 128, 8, "learned", causal=True, grad="all"),
        # cross attention, fp16, heads of 64 channels, ragged lengths, padded keys: training step
        _op("cross d64 padded step", 8, 8, 1000, 1500, 64, 16, "learned", dtype="fp16", mask="padding", grad="all"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A length spread over the logarithm of the range; half of them as they come, half rounded to a multiple of 64."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.5 else max(lo, n // 64 * 64)


def _drawn(rng):
    family = rng.choice(["learned", "learned", "learned", "alibi", "alibi block", "windows", "window block", "distance", "pair"])
    grad = rng.choice(["none", "step"])
    if family == "learned":
        d = rng.choice([32, 32, 64, 128])
        causal = rng.random() < 0.3
        Lq = _length(rng, 256, 16384)
        Lk = Lq if causal or rng.random() < 0.7 else _length(rng, 256, 16384)
        return _op(None, rng.choice([1, 2, 4, 8]), rng.choice([4, 8, 16, 32]), Lq, Lk, d, rng.choice([8, 8, 16, 32]), "learned",
                   dtype=rng.choice(["bf16", "bf16", "fp16"]), causal=causal, mask="padding" if not causal and rng.random() < 0.3 else "none",
                   grad="all" if grad == "step" else "none")
    if family == "alibi":
        L = _length(rng, 512, 8192)
        return _op(None, rng.choice([1, 2]), rng.choice([8, 16, 32, 50]), L, L, rng.choice([32, 32, 64]), 2, "alibi",
                   causal=True, grad="inputs" if grad == "step" else "none")
    if family == "alibi block":
        return _alibi_block(None, rng.choice([1, 2]), _length(rng, 256, 4096), rng.choice([16, 32, 50]), rng.choice([32, 64]),
                            "all" if grad == "step" else "none")
    if family == "windows":
        window = rng.choice([8, 12, 16])
        return _op(None, _log_int(rng, 64, 4096), rng.choice([4, 8, 16]), window * window, window * window, 32, 16, "table",
                   dtype=rng.choice(["bf16", "fp16"]), mask="windows" if rng.random() < 0.4 else "none",
                   grad="inputs" if grad == "step" else "none")
    if family == "window block":
        return _window_block(None, rng.choice([1, 2, 4, 8, 16]), rng.choice([4, 8]), rng.choice([8, 12, 16]), rng.choice([4, 8, 16]),
                             rng.random() < 0.5, "all" if grad == "step" else "none")
    if family == "distance":
        N = _length(rng, 1024, 32186)
        return _op(None, 1, 8, N, N, 32, 8, "distance", grad="inputs" if grad == "step" else "none")
    N = _length(rng, 128, 768)
    return _op(None, N, 4, N, N, 32, 32, "pair", mask="padding" if rng.random() < 0.5 else "none", grad="all" if grad == "step" else "none")


def draw(rng):
    most = [work(c) for c in listed()]
    flops, bytes_ = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    while True:
        c = _drawn(rng)
        w = work(c)
        if w["flops"] <= flops and w["bytes"] <= bytes_:
            return c


def _randn(g, shape, dtype, by=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(by).to(dtype)


def _shift_mask(side, window, dtype):
    """The 0 / -100 mask of a shifted-window block, (side * side, n, n): a feature map of side x side windows rolled by
    half a window, tokens that were not neighbours before do not see each other."""
    edge, shift = side * window, window // 2
    line = torch.zeros(edge, dtype=torch.int64)
    line[edge - window:edge - shift] = 1
    line[edge - shift:] = 2
    region = line[:, None] * 3 + line[None, :]
    w = region.view(side, window, side, window).permute(0, 2, 1, 3).reshape(side * side, window * window)
    return ((w[:, None, :] != w[:, :, None]).to(torch.float32) * -100.0).to("cuda", dtype)


def _prepare_op(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[c["dtype"]]
    B, H, Lq, Lk, d, r = (c[n] for n in ("B", "H", "Lq", "Lk", "d", "r"))
    q, k, v = (_randn(g, (B, L, H, d), dtype) for L in (Lq, Lk, Lk))
    do = _randn(g, (B, Lq, H, d), dtype)
    if c["bias"] == "learned":
        qb, kb = (_randn(g, (B, L, H, r), dtype, 1 / math.sqrt(r)) for L in (Lq, Lk))
    elif c["bias"] == "pair":
        qb, kb = (_randn(g, (1, L, H, r), dtype, 1 / math.sqrt(r)) for L in (Lq, Lk))
    elif c["bias"] == "alibi":
        qb, kb = factors.alibi_factors(Lq, Lk, H, dtype, device="cuda")
    elif c["bias"] == "distance":
        x = torch.rand(B, Lq, 3, generator=g, device="cuda")
        # (terms of at most 2 alpha: padded to rank 8 once by their owner, as workloads.pde does)
        qb, kb = factors.pad_rank(*factors.distance_factors(x, x, 10.0, dtype), 8)
    else:
        qb, kb, _ = factors.svd_factors(factors.swin_v2_bias_table(math.isqrt(Lq), H, seed), r, dtype)
        qb, kb = qb.cuda(), kb.cuda()
    mask = None
    if c["mask"] == "padding":  # the last keys of every batch entry are padding, an eighth of them at most
        seen = Lk - torch.randint(0, max(1, Lk // 8), (B,), generator=g, device="cuda")
        mask = ((torch.arange(Lk, device="cuda")[None, :] >= seen[:, None]).to(dtype) * -1e4)[:, None, None, :]
    elif c["mask"] == "windows":  # one mask per window of an image, repeated over the images
        n = _shift_mask(8, math.isqrt(Lq), dtype)
        mask = n[torch.arange(B, device="cuda") % n.shape[0]][:, None]
    leaves = []
    if c["grad"] != "none":
        leaves = [q, k, v] + ([qb, kb] if c["grad"] == "all" else [])
        for t in leaves:
            t.requires_grad_(True)
    return dict(args=(q, k, v, qb, kb, mask, c["causal"], 1.0 / math.sqrt(d)), leaves=leaves, do=do)


def _prepare_block(c, seed):
    torch.manual_seed(seed)
    if c["kind"] == "alibi block":
        dim, rows, n = c["H"] * c["d"], c["B"], c["L"]
        module, mask = modules.AttentionWithALiBiBias(dim, c["H"], c["d"]), None
    else:
        dim, rows, n = c["H"] * 32, c["images"] * c["side"] ** 2, c["window"] ** 2
        module = modules.WindowAttentionCore(dim, c["window"], c["H"], rank=16, seed=seed)
        mask = _shift_mask(c["side"], c["window"], torch.bfloat16) if c["shifted"] else None
    module = module.to("cuda", torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(seed)
    x, dy = _randn(g, (rows, n, dim), torch.bfloat16), _randn(g, (rows, n, dim), torch.bfloat16)
    leaves = []
    if c["grad"] == "all":
        leaves = [x.requires_grad_(True)] + list(module.parameters())
    return dict(module=module, args=(x,) if c["kind"] == "alibi block" else (x, mask), leaves=leaves, do=dy)


def prepare(case, seed):
    return _prepare_op(case, seed) if case["kind"] == "op" else _prepare_block(case, seed)


def run(state):
    f = state.get("module", flash_bias_func)
    if not state["leaves"]:
        with torch.no_grad():
            return f(*state["args"])
    out = f(*state["args"])
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["do"])]


def _attention(B, H, Lq, Lk, d, r, rb, rh, causal, mask_elements, grad):
    """(bytes, flops) of the operator with 16-bit tensors; rb, rh: batch entries and heads that the factors are given
    for.  Forward: q, k, v, factors and mask in, o out; the backward has them all and o, dO in, the gradients out, and
    needs the scores once more."""
    pairs = B * H * (Lq * (Lq + 1) // 2 if causal else Lq * Lk)
    qo, kv, fac = 2 * B * H * Lq * d, 2 * B * H * Lk * d, 2 * rb * rh * (Lq + Lk) * r
    bytes_, flops = 2 * qo + 2 * kv + fac + 2 * mask_elements, 2 * pairs * (2 * d + r)
    if grad != "none":
        bytes_ += 4 * qo + 4 * kv + fac + 2 * mask_elements + (fac if grad == "all" else 0)
        flops += 2 * pairs * (5 * d + r + (2 * r if grad == "all" else 0))
    return bytes_, flops


def work(case):
    c = case
    if c["kind"] == "op":
        B, H, Lq, Lk, r = c["B"], c["H"], c["Lq"], c["Lk"], c["r"]
        r = 5 if c["bias"] == "distance" else r
        rb = B if c["bias"] in ("learned", "distance") else 1
        rh = 1 if c["bias"] == "distance" else H
        m = {"none": 0, "padding": B * Lk, "windows": B * Lq * Lk}[c["mask"]]
        bytes_, flops = _attention(B, H, Lq, Lk, c["d"], r, rb, rh, c["causal"], m, c["grad"])
        return {"bytes": bytes_, "flops": flops}
    # the modules: four (three and one) projections of dim x dim around the operator; q, k, v and o need not
    # leave the chip in principle, x and y (and their gradients) do
    step = 3 if c["grad"] == "all" else 1
    grad = "inputs" if c["grad"] == "all" else "none"
    if c["kind"] == "alibi block":
        dim, tokens = c["H"] * c["d"], c["B"] * c["L"]
        flops = _attention(c["B"], c["H"], c["L"], c["L"], c["d"], 2, 0, 0, True, 0, grad)[1]
        m = 0
    else:
        dim, n, windows = c["H"] * 32, c["window"] ** 2, c["images"] * c["side"] ** 2
        tokens = windows * n
        flops = _attention(windows, c["H"], n, n, 32, 16, 0, 0, False, 0, grad)[1]
        m = c["side"] ** 2 * n * n if c["shifted"] else 0
    return {"bytes": 2 * (2 if step == 3 else 1) * (2 * tokens * dim + 4 * dim * dim) + 2 * m, "flops": flops + step * 8 * tokens * dim * dim}


def tolerance(case):
    """Operands and results of 8 (bf16) or 11 (fp16) significant bits, probabilities and score gradients rounded to them
    between the products, sums in 32 bits.  The window module also rounds its normalised q and k, whose cosines are then
    multiplied by 10: an error of 2^-9 in either is one of about a hundredth in the probabilities, and the gradient of
    logit_scale is one sum over all of them."""
    if case["kind"] == "window block":
        return {"rel": 3e-2}
    return {"rel": 2e-3 if case.get("dtype") == "fp16" else 1e-2}
