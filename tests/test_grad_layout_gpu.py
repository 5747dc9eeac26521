"""Gradients in the layout of permuted inputs: every dq and dk/dv kernel against the same call on contiguous copies. The values are
the same sums; where dk and dv are added by float atomics their order is not fixed (fp32: 1e-5 of the largest), and 16-bit
storage rounds such a sum to one of two neighbours, a step apart: up to 2^-7 of an element in bf16 (8 bits), 2^-10 in fp16 (11)."""
import ctypes
import math

import pytest
import torch

from ops import _native
from ops.triton import deform_sdpa_triton
from parity_util import kernels_of

CASES = [
    # B, V, H, Himg, Wimg, D, P, how the samples lie, dq and dk/dv kernels (slabs: fp32; deterministic: cells)
    (2, 2, 3, 6, 5, 32, 2, "unit", "rows", "cell"),
    (2, 2, 32, 10, 9, 32, 2, "unit", "rows", "patch"),
    (1, 3, 2, 9, 7, 64, 12, "unit", "slot", "cell"),
    (1, 2, 24, 13, 21, 32, 4, "border", "slot", "patch"),
    (2, 3, 16, 23, 21, 16, 4, "point", "slot", "patch"),     # left to the cells behind them
    (1, 2, 2, 32, 32, 64, 16, "border", "slab", "cell"),
    (1, 2, 1, 37, 23, 128, 40, "border", "gather", "cell"),
    (1, 2, 1, 34, 36, 128, 64, "point", "gather", "cell"),   # windows
    (1, 1, 1, 1, 1, 256, 1, "unit", "rows", "cell"),
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


def as_given(kind, grad, H):
    """a leaf's gradient as one of the operator's (B, V, H, L, D) argument"""
    return (grad.permute(0, 1, 3, 2, 4) if kind == "projection" else grad.permute(0, 2, 3, 1, 4) if kind == "pixels first"
            else grad[:, :, :H] if kind == "sliced" else grad)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["plain", "coords", "deterministic"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("case", CASES, ids=[f"{c[3]}x{c[4]}-D{c[5]}-P{c[6]}" for c in CASES])
def test_gradients_follow_the_inputs_layout(case, dtype, mode):
    B, V, H, Himg, Wimg, D, P, where, dq_kernel, dkdv_kernel = case
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
            names = kernels_of(lambda: out.backward(dout))
            grads = [as_given(kind, leaf.grad, H) for kind, leaf in ((kq, ql), (kk, kl), (kk, vl))]
            results[kq, kk] = [x.contiguous() for x in grads] + ([c.grad] if mode == "coords" else [])
            dq_by = "gather" if dq_kernel == "slab" and dtype != torch.float32 else dq_kernel
            dkdv_by = "cell" if mode == "deterministic" else dkdv_kernel
            assert all(any(n.startswith(by) for n in names) for by in (f"bwd_dq_{dq_by}_kernel", f"bwd_dkdv_{dkdv_by}_kernel")), names
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


# Only a gradient that nobody sees lies as its tensor does. Whoever is shown that of q, or what the permutation's backward makes of it,
# gets it contiguous as (B, V, H, L, D), whatever q's strides are.
@pytest.mark.gpu
@pytest.mark.parametrize("who", ["grad", "hook", "retain", "prehook", "node", "own node", "leaf grad", "leaf hook", "behind", "permuted leaf", "nobody"])
def test_gradients_that_are_shown_are_contiguous(who):
    print(f"[case] shown gradients: {who}", flush=True)
    B, V, H, Himg, Wimg, D, P = 1, 2, 4, 10, 9, 32, 2
    seen = []

    def see(g):
        seen.append(g.detach())
    leaf = torch.randn(B, V, Himg * Wimg, H, D, device="cuda").requires_grad_(True)
    back = lambda g: g.permute(0, 1, 3, 2, 4)
    q = back(leaf + 1.0) if who == "behind" else back(leaf)
    if who == "permuted leaf":
        q = back(leaf.detach()).requires_grad_(True)
    k, v = torch.randn(2, B, V, H, Himg * Wimg, D, device="cuda").requires_grad_(True).unbind(0)
    out = deform_sdpa_triton(q, k, v, torch.rand(B, V, Himg * Wimg, V, P, 2, device="cuda"), Wimg, Himg, 0.2)
    dout = torch.randn(out.shape, device="cuda")
    if who in ("grad", "permuted leaf"):
        see(torch.autograd.grad(out, q, dout)[0])
    elif who == "leaf grad":
        see(back(torch.autograd.grad(out, leaf, dout)[0]))
    else:
        if who == "hook":
            q.register_hook(see)
        elif who == "retain":
            q.retain_grad()
        elif who == "prehook":
            q.grad_fn.register_prehook(lambda go: see(go[0]))
        elif who == "node":
            q.grad_fn.register_hook(lambda gi, go: see(go[0]))
        elif who == "own node":
            out.grad_fn.register_hook(lambda gi, go: see(gi[0]))
        elif who == "leaf hook":
            leaf.register_hook(lambda g: see(back(g)))
        elif who == "behind":
            q.grad_fn.next_functions[0][0].register_prehook(lambda go: see(back(go[0])))
        out.backward(dout)
        if who == "retain":
            see(q.grad)
    if who == "nobody":
        assert leaf.grad.is_contiguous() and not seen
    else:
        assert len(seen) == 1 and seen[0].is_contiguous()
        seen[0].view(-1)


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


# 2^34 elements and more are addressed like fewer. (Where there is no GPU, what passes the checks ends at the first launch.)
@pytest.mark.skipif(torch.cuda.device_count() > 0, reason="the pointers are made up")
def test_size_is_no_reason_to_refuse_the_layout():
    lib = _native.load()
    fake, ll8 = ctypes.c_void_p(0x1000), ctypes.c_longlong * 8
    B, V, H, side, D = 8200, 1, 2, 64, 256
    strides = ll8(*2 * (V * H * side * side * D, H * side * side * D, D, H * D))
    call = [fake] * 10 + [None, fake, B, V, H, side, side, D, 2, 0.5, strides]
    rc = [lib.dsdpa_bwd_bf16(*call, flags, None) for flags in (0, _native.FLAG_GRADS_AS_INPUTS)]
    assert rc[0] == rc[1], rc
