"""Performance cases of the fused deformable multi-view SDPA operator.

Every case is one pass through the public operator, ``deform_sdpa_triton(q, k, v, coords, WIDTH, HEIGHT, sm_scale)``
with its optional eighth argument, as a program that holds the inputs on the GPU calls it:

``what``     "forward" (inference, no graph), "step" (forward and backward), "coords" (a step that asks for the
             gradient of the sampling positions too, as a trained deformable attention does), "deterministic" (a step
             under ``torch.use_deterministic_algorithms``)
``coords``   where the samples lie, as in ``workloads.py``: "unit" over the whole image, "border" over a tenth of
             the image more on every side, "clustered" around a centre drawn per query, "coherent" around the
             query's own place in the other view
``layout``   "packed": q, k, v contiguous; "projection": as a linear layer leaves them, (batch, view, pixel, head, dim),
             permuted for the call
"""
import importlib
import math
import os

import torch

_PACKAGE = "fused-deform-multi-head-scaled-dot-product-attention-triton_amd"
if not os.path.isdir(os.path.join(os.getcwd(), _PACKAGE)):
    raise ImportError("perf/cases.py runs with the repository's root as the working folder")
deform_sdpa_triton = importlib.import_module(_PACKAGE + ".ops.triton").deform_sdpa_triton

_DTYPE = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, what, dtype, B, V, H, D, W, Himg, P, coords, scale, layout="packed"):
    return {"name": name, "what": what, "dtype": dtype, "B": B, "V": V, "H": H, "D": D, "W": W, "Himg": Himg, "P": P,
            "coords": coords, "scale": scale, "layout": layout}


def listed():
    return [
        # the smallest point of the views x samples sweep (sweep.py's defaults: batch 2, 32 heads, 18x18): a call
        # whose time is launches and host work, once at inference and once as a training step
        _case("sweep-2x2-forward", "forward", "fp32", 2, 2, 32, 32, 18, 18, 2, "unit", 0.5),
        _case("sweep-2x2-step", "step", "fp32", 2, 2, 32, 32, 18, 18, 2, "unit", 0.5),
        # the middle of the same sweep in 16-bit storage
        _case("sweep-6x6-step-bf16", "step", "bf16", 2, 6, 32, 32, 18, 18, 6, "unit", 0.5),
        # its largest point, the headline figure of the sweep
        _case("sweep-12x12-forward", "forward", "fp32", 2, 12, 32, 32, 18, 18, 12, "unit", 0.5),
        # the README example (workload C1): small images, many samples
        _case("readme-step", "step", "fp32", 2, 8, 16, 32, 14, 14, 32, "unit", 0.5),
        # workload C2 as a reproducible training run calls it
        _case("square18-deterministic", "deterministic", "fp32", 2, 6, 8, 32, 18, 18, 32, "unit", 1.0 / math.sqrt(32)),
        # workload C3: larger maps, a quarter of the taps outside the image
        _case("border-step", "step", "fp32", 1, 6, 8, 64, 32, 32, 16, "border", 0.125),
        # workload C4: 16-bit storage, maps too large for on-chip memory, samples everywhere
        _case("uniform-step-bf16", "step", "bf16", 2, 6, 8, 64, 48, 48, 32, "unit", 0.125),
        # workload C5, the largest: every query's samples around one place, all of them in the middle of the image
        _case("clustered-step-bf16", "step", "bf16", 2, 4, 8, 128, 64, 64, 64, "clustered", 1.0 / math.sqrt(128)),
        # workload C5c at inference: neighbouring queries look at neighbouring places
        _case("coherent-forward-bf16", "forward", "bf16", 2, 4, 8, 128, 64, 64, 64, "coherent", 1.0 / math.sqrt(128)),
        # deformable attention as it is trained: few samples per view around the query's place, offsets learned
        # (gradient of the positions), q, k, v straight from their projections
        _case("coherent-coords-fp16", "coords", "fp16", 2, 4, 8, 64, 40, 28, 8, "coherent", 0.125, "projection"),
        # nothing a multiple of anything
        _case("ragged-step", "step", "fp32", 1, 3, 5, 128, 37, 23, 7, "border", 1.0 / math.sqrt(128)),
    ]


_MOST, _LEAST = 2.0e9, 2.0e6        # multiply-adds (samples x head dimension) of a drawn case


def draw(rng):
    """A case of the same ranges: maps of 8 to 64 pixels a side, 1 to 12 views, 2 to 64 samples, all head dimensions."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while True:
        D = rng.choice([16, 32, 32, 64, 64, 128, 256])
        B, V, H = rng.choice([1, 2]), log(1, 12), log(2, 32)
        W, Himg, P = log(8, 64), log(8, 64), log(2, 64)
        if _LEAST <= B * V * H * W * Himg * V * P * D <= _MOST:
            break
    r = rng.random()
    what = "forward" if r < 0.4 else "step" if r < 0.75 else "coords" if r < 0.9 else "deterministic"
    dtype = rng.choice(["fp32", "fp32", "bf16", "bf16", "fp16"])
    coords = rng.choice(["unit", "border", "clustered", "coherent"])
    case = _case("", what, dtype, B, V, H, D, W, Himg, P, coords, 1.0 / math.sqrt(D), rng.choice(["packed", "packed", "projection"]))
    del case["name"]
    return case


def _coords(case, gen):
    B, V, P, W, Himg = (case[n] for n in ("B", "V", "P", "W", "Himg"))
    L, dev, kind = W * Himg, "cuda", case["coords"]
    shape = (B, V, L, V, P, 2)
    if kind == "unit":
        return torch.rand(shape, generator=gen, device=dev)
    if kind == "border":
        return torch.rand(shape, generator=gen, device=dev) * 1.2 - 0.1
    around = torch.randn(shape, generator=gen, device=dev) * 0.03
    if kind == "clustered":
        centre = torch.rand((B, V, L, V, 1, 2), generator=gen, device=dev) * 0.2 + 0.4
    else:
        ys, xs = torch.meshgrid(torch.arange(Himg, device=dev), torch.arange(W, device=dev), indexing="ij")
        own = torch.stack([xs.reshape(-1) / max(W - 1, 1), ys.reshape(-1) / max(Himg - 1, 1)], -1)
        centre = own.view(1, 1, L, 1, 1, 2) * 0.6 + 0.2 + 0.02 * torch.randn((B, V, 1, V, 1, 2), generator=gen, device=dev)
    return (centre + around).clamp_(0.0, 1.0)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, V, H, D, L = case["B"], case["V"], case["H"], case["D"], case["W"] * case["Himg"]
    dtype, train = _DTYPE[case["dtype"]], case["what"] != "forward"
    shape = (B, V, L, H, D) if case["layout"] == "projection" else (B, V, H, L, D)
    qkv = [torch.randn(shape, generator=gen, device="cuda").to(dtype).requires_grad_(train) for _ in range(3)]
    coords = _coords(case, gen).requires_grad_(case["what"] == "coords")
    dout = torch.randn((B, V, H, L, D), generator=gen, device="cuda").to(dtype) if train else None
    return {"case": case, "qkv": qkv, "coords": coords, "dout": dout}


def run(state):
    case, coords = state["case"], state["coords"]
    leaves = state["qkv"]
    q, k, v = (t.permute(0, 1, 3, 2, 4) for t in leaves) if case["layout"] == "projection" else leaves
    W, Himg, scale, what = case["W"], case["Himg"], case["scale"], case["what"]
    if what == "forward":
        with torch.no_grad():
            return deform_sdpa_triton(q, k, v, coords, W, Himg, scale)
    for t in leaves:
        t.grad = None
    if what == "coords":
        coords.grad = None
        out = deform_sdpa_triton(q, k, v, coords, W, Himg, scale, True)
        out.backward(state["dout"])
        return [out.detach()] + [t.grad for t in leaves] + [coords.grad]
    if what == "deterministic":
        torch.use_deterministic_algorithms(True)
        try:
            out = deform_sdpa_triton(q, k, v, coords, W, Himg, scale)
            out.backward(state["dout"])
        finally:
            torch.use_deterministic_algorithms(False)
    else:
        out = deform_sdpa_triton(q, k, v, coords, W, Himg, scale)
        out.backward(state["dout"])
    return [out.detach()] + [t.grad for t in leaves]


def work(case):
    """q, k, v and coords read, out written, each once; a step reads those and dout and writes the gradients. The
    operations are those of the operator's definition, per sample: two bilinear blends of four taps (8 D
    multiply-adds), the logit and the weighted sum (2 D); backward recomputes the blends and the logit (9 D), has one
    product for dp and one for dq (2 D) and spreads two rows over four taps (8 D)."""
    B, V, H, D, P, L = case["B"], case["V"], case["H"], case["D"], case["P"], case["W"] * case["Himg"]
    rows = B * V * H * L
    tensor = rows * D * (4 if case["dtype"] == "fp32" else 2)
    coords = B * V * L * V * P * 2 * 4
    samples = rows * V * P
    nbytes, flops = 4 * tensor + coords, 2 * 10 * D * samples
    if case["what"] != "forward":
        # one step as a whole: q, k, v, coords, dout in; out, dq, dk, dv out
        nbytes = 8 * tensor + coords * (2 if case["what"] == "coords" else 1)
        flops += 2 * 19 * D * samples
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # fp32 throughout: sums in another order. 16-bit storage: the outputs' own rounding (bf16 2^-9, fp16 2^-12) and that
    # of the saved output, from which the backward takes its row sums.
    return {"rel": {"fp32": 1e-5, "bf16": 1e-2, "fp16": 2e-3}[case["dtype"]]}
