"""Calls that the operator's native side hands back to Python to be mended (coordinates of another type, layouts the
kernels cannot read, sizes that are not plain ints) give what the mended arguments give, gradients included."""
import numpy as np
import pytest
import torch

from ops.triton import deform_sdpa_triton

pytestmark = pytest.mark.gpu

B, V, H, HIMG, WIMG, D, P = 2, 2, 3, 4, 5, 32, 3


def inputs():
    g = torch.Generator().manual_seed(5)
    L = HIMG * WIMG
    q, k, v = (torch.randn(B, V, H, L, D, generator=g).cuda() for _ in range(3))
    return q, k, v, torch.rand(B, V, L, V, P, 2, generator=g).cuda(), torch.randn(B, V, H, L, D, generator=g).cuda()


def step(q, k, v, c, do, w, h):
    leaves = [t.detach().requires_grad_(True) for t in (q, k, v, c)]       # (detach keeps a layout)
    out = deform_sdpa_triton(*leaves, w, h, 0.3, True)
    out.backward(do)
    return [out.detach()] + [t.grad for t in leaves]


@pytest.mark.parametrize("what", ["coords_double", "coords_half", "head_dim_strided", "k_v_unlike", "numpy_sizes"])
def test_mended_call(what):
    print(f"[case] {what}", flush=True)
    q, k, v, c, do = inputs()
    if what == "coords_half":
        c = c.half().float()
    want = step(q, k, v, c, do, WIMG, HIMG)
    w, h = WIMG, HIMG
    if what == "coords_double":
        c = c.double()
    elif what == "coords_half":
        c = c.half()
    elif what == "head_dim_strided":
        q = q.transpose(3, 4).contiguous().transpose(3, 4)
    elif what == "k_v_unlike":
        k = k.transpose(2, 3).contiguous().transpose(2, 3)
    else:
        w, h = np.int64(WIMG), np.int32(HIMG)
    got = step(q, k, v, c, do, w, h)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    for a, b in zip(got[2:4], want[2:4]):               # float atomics: the order of the sums is not fixed
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    bound = 1e-3 if what == "coords_half" else 1e-5      # the gradient of half coordinates is rounded to 2^-11
    assert got[4].dtype == c.dtype
    assert (got[4].double() - want[4].double()).abs().max() <= bound * want[4].abs().max()
