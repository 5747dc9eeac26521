"""dk/dv by patches of 4x4 pixels, where the cell lists are short: images whose sides end inside a patch, every lane split of
the head dimension, entries on the patch borders, lists too long for patches in one key view, and non-finite
rows, which may reach the pixels they touch only. Against the CPU oracle at the bars of the other gradient tests
(sums in another order 1e-3 in fp32, the storage type's rounding 2e-2 in 16 bits)."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle_bwd
from ops.triton import deform_sdpa_triton
from parity_util import rel

pytestmark = pytest.mark.gpu
BAR = {torch.float32: 1e-3, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def inputs(B, V, H, Himg, Wimg, D, P, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    L = Himg * Wimg
    assert B * V * H * ((Himg + 3) // 4) * ((Wimg + 3) // 4) >= 1024 and B * V * H * L * V * P >= 1 << 15     # the patches' range
    t = [torch.randn(B, V, H, L, D, generator=g).to(dtype) for _ in range(4)]
    return (*t, torch.rand(B, V, L, V, P, 2, generator=g) * 1.2 - 0.1)


def gradients(q, k, v, coords, dout, W, Himg):
    scale = 1.0 / math.sqrt(q.shape[-1])
    print(f"[case] patches {tuple(q.shape)} {Himg}x{W} P{coords.shape[-2]} {q.dtype}", flush=True)
    leaves = [t.to("cuda:0").requires_grad_(True) for t in (q, k, v)]
    deform_sdpa_triton(*leaves, coords.to("cuda:0"), W, Himg, scale).backward(dout.to("cuda:0"))
    torch.cuda.synchronize()
    want = oracle_bwd(*(t.float().numpy() for t in (q, k, v, coords, dout)), W, Himg, scale)
    return [t.grad for t in leaves], want


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("B,V,H,Himg,Wimg,D,P", [(1, 2, 256, 5, 6, 16, 2), (2, 2, 64, 7, 9, 32, 3), (1, 3, 40, 9, 11, 64, 2),
                                                 (1, 2, 33, 13, 14, 128, 2), (1, 1, 64, 17, 18, 256, 2), (2, 1, 128, 1, 16, 32, 8)])
def test_patches_against_the_oracle(B, V, H, Himg, Wimg, D, P, dtype):
    q, k, v, dout, coords = inputs(B, V, H, Himg, Wimg, D, P, dtype, 7)
    got, want = gradients(q, k, v, coords, dout, Wimg, Himg)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# mean list length up to 48 in 16 bits and 12 in fp32: lists of several blocks of 64 entries a patch, two and four waves
@pytest.mark.parametrize("P,dtype", [(7, torch.float32), (40, torch.bfloat16), (40, torch.float16)], ids=str)
def test_several_blocks_a_patch(P, dtype):
    q, k, v, dout, coords = inputs(1, 1, 114, 11, 9, 32, P, dtype, 8)
    got, want = gradients(q, k, v, coords, dout, 9, 11)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# samples of one key view in one cell: its lists are left to the cell kernel, the other views' are not
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
def test_one_view_clustered(dtype):
    q, k, v, dout, coords = inputs(2, 3, 12, 20, 18, 64, 2, dtype, 9)
    coords[:, :, :, 1] = (coords[:, :, :, 1] + 0.1) / 1.2 / 40 + 0.5
    got, want = gradients(q, k, v, coords, dout, 18, 20)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_non_finite_rows_stay_with_their_pixels(bad, dtype):
    q, k, v, dout, coords = inputs(1, 2, 64, 9, 10, 32, 2, dtype, 11)
    dout[0, 1, 3, 17, 5] = bad                               # a column of dv at the taps of one query; its dp, so its ds: all columns of dk
    got, want = gradients(q, k, v, coords, dout, 10, 9)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        a = a.float().cpu().numpy()
        assert np.array_equal(np.isfinite(a), np.isfinite(b)), name
        assert 0 < (~np.isfinite(b)).sum() < 2000, name
        ok = np.isfinite(b)
        assert np.abs(a[ok] - b[ok]).max() < BAR[dtype] * np.abs(b[ok]).max(), name


# Coefficients (weight times p) to fp32's precision: three queries look at one place, with different p, and the rows of dout
# cancel down to 2^-13 of their size. What is left takes the storage type's rounding (1.7e-3 in bf16) and that of p and the sums (2^-23 of the
# terms, a few of them: 2^-10 of the rest); coefficients good to 2^-17 would leave 2^-4 times a third of it (1.5e-2).
@pytest.mark.parametrize("dtype,kept", [(torch.bfloat16, 2.0 ** -4), (torch.float16, 0.5)], ids=str)
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_coefficients_are_not_rounded_to_16_bits(D, dtype, kept):
    H, W = 64, 16
    L, T, scale = W * W, W * W // 3, 1.0 / math.sqrt(D)
    g = torch.Generator().manual_seed(D)
    q, k, v, d = (torch.randn(1, 1, H, L, D, generator=g).to(dtype) for _ in range(4))
    coords = torch.full((1, 1, L, 1, 2, 2), -1.0)                # the second sample: outside, its logit 0
    place = torch.rand(T, 2, generator=g) * 0.9 + 0.05
    coords[0, 0, :3 * T, 0, 0] = place.repeat_interleave(3, 0)
    x, y = (place.double() * (W - 1)).unbind(-1)
    x0, y0 = x.floor().long(), y.floor().long()
    fx, fy = x - x0, y - y0
    taps = [((y0 + j) * W + x0 + i, (fx if i else 1 - fx) * (fy if j else 1 - fy)) for j in (0, 1) for i in (0, 1)]
    at = sum(w[:, None] * k[0, 0].double()[:, p] for p, w in taps)                                   # (H, T, D): k at the places
    p = torch.sigmoid(scale * (q[0, 0, :, :3 * T].double().view(H, T, 3, D) * at[:, :, None]).sum(-1))
    p = [p[..., m, None] for m in range(3)]
    rows = d[0, 0, :, :3 * T].double().view(H, T, 3, D)[:, :, 0]
    second = (-p[0] / p[1] * rows).to(dtype)
    left = p[0] * rows + p[1] * second.double()
    third = (-(1 - kept) * left / p[2]).to(dtype)
    left = left + p[2] * third.double()
    dout = torch.zeros_like(d)
    dout[0, 0, :, :3 * T] = torch.stack([rows.to(dtype), second, third], 2).view(H, 3 * T, D)
    want = torch.zeros(H, L, D, dtype=torch.float64)
    for pix, w in taps:
        want.index_add_(1, pix, w[:, None] * left)
    print(f"[case] cancelling rows D{D} {dtype}", flush=True)
    vd = v.cuda().requires_grad_(True)
    deform_sdpa_triton(q.cuda(), k.cuda(), vd, coords.cuda(), W, W, scale).backward(dout.cuda())
    torch.cuda.synchronize()
    err = float((vd.grad[0, 0].double().cpu() - want).norm() / want.norm())
    print("error", err, "of", float(left.norm() / rows.norm()))
    assert err < 8e-3, err
