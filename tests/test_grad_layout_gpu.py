"""Gradients in the layout of permuted inputs: every dq and dk/dv kernel against the same call on contiguous copies. The values are
the same sums; where dk and dv are added by float atomics their order is not fixed (fp32: 1e-5 of the largest), and 16-bit
storage rounds such a sum to one of two neighbours, a step apart: up to 2^-7 of an element in bf16 (8 bits), 2^-10 in fp16 (11)."""
import ctypes
import math

import pytest
import torch

from ops import _native
from ops.triton import deform_sdpa_triton

CASES = [
    # B, V, H, Himg, Wimg, D, P, how the samples lie           which kernels
    (2, 2, 3, 6, 5, 32, 2, "unit"),                          # rows, cells
    (2, 2, 32, 10, 9, 32, 2, "unit"),                        # rows, patches
    (1, 3, 2, 9, 7, 64, 12, "unit"),                         # staged planes, cells
    (1, 2, 24, 13, 21, 32, 4, "border"),                     # staged planes, patches
    (2, 3, 16, 23, 21, 16, 4, "point"),                      # patches left to the cells behind them
    (1, 2, 2, 32, 32, 64, 16, "border"),                     # slabs (fp32)
    (1, 2, 1, 37, 23, 128, 40, "border"),                    # a wave per row
    (1, 2, 1, 34, 36, 128, 64, "point"),                     # windows
    (1, 1, 1, 1, 1, 256, 1, "unit"),
]


def layouts(kind, t):
    """(leaf, the (B, V, H, L, D) tensor that the operator is given) of the same values"""
    if kind == "projection":                                 # (B, V, L, H, D)
        leaf = t.permute(0, 1, 3, 2, 4).contiguous().requires_grad_(True)
        return leaf, leaf.permute(0, 1, 3, 2, 4)
    if kind == "pixels first":                               # (B, L, V, H, D)
        leaf = t.permute(0, 3, 1, 2, 4).contiguous().requires_grad_(True)
        return leaf, leaf.permute(0, 2, 3, 1, 4)
    if kind == "sliced":                                     # heads of a wider tensor: holes, gradients stay contiguous
        leaf = torch.cat([t, t], 2).requires_grad_(True)
        return leaf, leaf[:, :, :t.shape[2]]
    leaf = t.clone().requires_grad_(True)
    return leaf, leaf


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["plain", "coords", "deterministic"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("case", CASES, ids=[f"{c[3]}x{c[4]}-D{c[5]}-P{c[6]}" for c in CASES])
def test_gradients_follow_the_inputs_layout(case, dtype, mode):
    B, V, H, Himg, Wimg, D, P, where = case
    L = Himg * Wimg
    print(f"[case] gradient layout {case} {dtype} {mode}", flush=True)
    g = torch.Generator().manual_seed(L + P)
    q, k, v, dout = (torch.randn(B, V, H, L, D, generator=g).to(dtype).cuda() for _ in range(4))
    coords = torch.rand(B, V, L, V, P, 2, generator=g)
    coords = (coords * 1.2 - 0.1 if where == "border" else coords * 0.1 + 0.4 if where == "point" else coords).cuda()
    results = {}
    torch.use_deterministic_algorithms(mode == "deterministic")
    try:
        for kq, kk in (("contiguous", "contiguous"), ("projection", "projection"), ("pixels first", "contiguous"),
                       ("contiguous", "pixels first"), ("sliced", "projection")):
            ql, qv = layouts(kq, q)
            kl, kv = layouts(kk, k)
            vl, vv = layouts(kk, v)
            c = coords.clone().requires_grad_(mode == "coords")
            out = deform_sdpa_triton(qv, kv, vv, c, Wimg, Himg, 1.0 / math.sqrt(D), mode == "coords")
            assert out.is_contiguous()
            grads = torch.autograd.grad(out, (qv, kv, vv) + ((c,) if mode == "coords" else ()), dout)
            if "sliced" not in (kq, kk):
                for t, d in ((qv, grads[0]), (kv, grads[1]), (vv, grads[2])):
                    assert all(s == u for s, u, n in zip(t.stride(), d.stride(), t.shape) if n > 1)
            results[kq, kk] = [x.contiguous() for x in grads]
    finally:
        torch.use_deterministic_algorithms(False)
    ref = results.pop(("contiguous", "contiguous"))
    step = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    for name, got in results.items():
        assert torch.equal(got[0], ref[0]), name
        for a, b in zip(got[1:], ref[1:]):
            if mode == "deterministic":
                assert torch.equal(a, b), name
            else:
                a, b = a.double(), b.double()
                assert ((a - b).abs() <= 1e-5 * b.abs().max() + step * b.abs()).all(), name


@pytest.mark.gpu
def test_leaf_gradients_are_not_copied():
    """A projection's gradients reach it as they are: the only new memory of a backward is theirs and the workspace."""
    B, V, H, Himg, Wimg, D, P = 1, 2, 4, 24, 24, 64, 4
    leaves = [torch.randn(B, V, Himg * Wimg, H, D, device="cuda").requires_grad_(True) for _ in range(3)]
    coords = torch.rand(B, V, Himg * Wimg, V, P, 2, device="cuda")
    out = deform_sdpa_triton(*(t.permute(0, 1, 3, 2, 4) for t in leaves), coords, Wimg, Himg, 0.125)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        out.backward(torch.ones_like(out))
    assert not any(e.key in ("aten::copy_", "aten::clone") for e in prof.key_averages())
    for t in leaves:
        assert t.grad.is_contiguous()


def test_strides_that_do_not_fill_a_block_are_refused():
    lib = _native.load()
    fake = ctypes.c_void_p(0x1000)   # never dereferenced: validation fails first
    ll8 = ctypes.c_longlong * 8
    V, H, L, D = 2, 2, 12, 32
    dense = (V * L * H * D, L * H * D, D, H * D)             # (B, V, L, H, D) as (B, V, H, L, D)
    holes = (2 * V * L * H * D, 2 * L * H * D, D, 2 * H * D)
    shared = (V * L * H * D, 0, D, H * D)
    call = [fake] * 10 + [None, fake, 1, V, H, 3, 4, D, 2, 0.5]
    for q, kv in ((holes, dense), (dense, holes), (shared, dense)):
        assert lib.dsdpa_bwd_f32(*call, ll8(*q, *kv), _native.FLAG_GRADS_AS_INPUTS, None) == _native.ERR_BAD_STRIDES
