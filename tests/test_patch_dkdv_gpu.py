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
from parity_util import kernels_of, oracle_on_slices, rel

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


# mean list length up to 48 in 16 bits and 12 in fp32: lists of several blocks of 64 entries a patch, one and two waves
@pytest.mark.parametrize("P,dtype", [(7, torch.float32), (40, torch.bfloat16), (40, torch.float16)], ids=str)
def test_several_blocks_a_patch(P, dtype):
    q, k, v, dout, coords = inputs(1, 1, 114, 11, 9, 32, P, dtype, 8)
    got, want = gradients(q, k, v, coords, dout, 9, 11)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# 16 columns: C in LDS by halves of a block; lists that end in a first half, in a second one and behind one
@pytest.mark.parametrize("P,dtype", [(3, torch.float32), (7, torch.float32), (3, torch.bfloat16), (20, torch.bfloat16)], ids=str)
def test_half_blocks(P, dtype):
    q, k, v, dout, coords = inputs(1, 1, 114, 11, 9, 16, P, dtype, 16)
    got, want = gradients(q, k, v, coords, dout, 9, 11)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# C in LDS by halves of a block, every entry at the same four pixels: what one lane clears, the lane 32 places on writes next. (Few samples,
# binned in one launch, are the patches' wherever they lie in 16-bit storage. They are spread over their cell: at one point dp - delta, and
# with it ds, cancels down to what the rounding of the saved output, 2^-9 of delta, leaves of it.)
@pytest.mark.parametrize("D,P", [(16, 3), (16, 20), (32, 3), (32, 20)])
def test_half_blocks_of_one_cell(D, P):
    q, k, v, dout, coords = inputs(1, 1, 114, 11, 9, D, P, torch.bfloat16, 18)
    coords = 0.5 + (coords + 0.1) / 1.2 * torch.tensor([0.124, 0.099])
    got, want = gradients(q, k, v, coords, dout, 9, 11)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[torch.bfloat16], name


# 1350 visits a patch: four waves
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_four_waves_a_patch(dtype):
    B, V, H, side, D, P = 1, 6, 7, 20, 32, 9
    assert V * side * side * P * 25 // 16 // (side // 4) ** 2 > 1280
    q, k, v, dout, coords = inputs(B, V, H, side, side, D, P, dtype, 15)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    print(f"[case] four waves a patch {dtype}", flush=True)
    out = deform_sdpa_triton(*leaves, coords.cuda(), side, side, 0.18)
    names = kernels_of(lambda: out.backward(dout.cuda()))
    assert any(n.startswith("bwd_dkdv_patch_kernel") for n in names), names
    want = oracle_bwd(*(t.float().numpy() for t in (q, k, v, coords, dout)), side, side, 0.18)
    for leaf, b, name in zip(leaves, want, ("dq", "dk", "dv")):
        assert rel(leaf.grad, b) < BAR[dtype], name


# samples of one key view in one cell: its lists are left to the cell kernel, the other views' are not
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
def test_one_view_clustered(dtype):
    q, k, v, dout, coords = inputs(2, 3, 12, 20, 18, 64, 2, dtype, 9)
    coords[:, :, :, 1] = (coords[:, :, :, 1] + 0.1) / 1.2 / 40 + 0.5
    got, want = gradients(q, k, v, coords, dout, 18, 20)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# few cells hold samples and one of them many: left to the cell kernel by the longest list, at a mean that is the patches'
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=str)
def test_few_cells_and_a_long_list(dtype):
    q, k, v, dout, coords = inputs(1, 2, 45, 19, 21, 16, 2, dtype, 10)
    coords = 0.5 + 0.07 * torch.randn(coords.shape, generator=torch.Generator().manual_seed(10))
    at = (coords[0, :, :, 0].reshape(-1, 2) * torch.tensor([20, 18])).floor().long()
    lists = torch.unique(at[:, 1] * 22 + at[:, 0], return_counts=True)[1]
    assert len(lists) * 90 < 16384 and lists.double().mean() < 31 and lists.max() > 40, lists
    got, want = gradients(q, k, v, coords, dout, 21, 19)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


# samples of two key views of three in a few cells each: the third one's lists are left to the cell kernel too, although they are short
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
def test_most_views_clustered(dtype):
    q, k, v, dout, coords = inputs(2, 3, 12, 20, 18, 32, 2, dtype, 14)
    coords[:, :, :, :2] = (coords[:, :, :, :2] + 0.1) / 1.2 / 40 + 0.5
    got, want = gradients(q, k, v, coords, dout, 18, 20)
    for a, b, name in zip(got, want, ("dq", "dk", "dv")):
        assert rel(a, b) < BAR[dtype], name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
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


# What leaves the pairs: the staged dq kernel (narrow, and eight fp32 elements a lane), with the coordinate gradient, and the row
# kernel, which takes few samples and planes beyond LDS; q, k, v as projections leave them
@pytest.mark.parametrize("B,V,H,Himg,Wimg,D,P,dtype,coords_grad,dq", [
    (2, 2, 32, 18, 18, 32, 4, torch.float32, False, "bwd_dq_slot_kernel<F32, 32, 8, false, 1, true>"),
    (2, 2, 32, 12, 13, 64, 4, torch.float32, False, "bwd_dq_slot_kernel<F32, 64, 8, false, 1, true>"),
    (2, 2, 32, 18, 18, 32, 4, torch.float32, True, "bwd_dq_slot_kernel<F32, 32, 4, true, 1, true>"),
    (2, 2, 32, 18, 18, 32, 4, torch.bfloat16, True, "bwd_dq_slot_kernel<BF16, 32, 8, true, 1, true>"),
    (2, 2, 32, 18, 17, 64, 5, torch.float16, True, "bwd_dq_slot_kernel<F16, 64, 8, true, 1, true>"),
    (1, 4, 64, 9, 10, 256, 4, torch.bfloat16, True, "bwd_dq_slot_kernel<BF16, 256, 16, true, 1, true>"),
    (1, 2, 12, 23, 29, 128, 2, torch.float32, True, "bwd_dq_rows_kernel<F32, 128, "),
    (1, 2, 12, 23, 29, 128, 5, torch.float16, False, "bwd_dq_rows_kernel<F16, 128, "),
    (1, 2, 12, 23, 29, 256, 3, torch.bfloat16, True, "bwd_dq_rows_kernel<BF16, 256, "),
], ids=str)
@pytest.mark.parametrize("projection", [False, True])
def test_patches_behind_every_dq_kernel(B, V, H, Himg, Wimg, D, P, dtype, coords_grad, dq, projection):
    q, k, v, dout, coords = inputs(B, V, H, Himg, Wimg, D, P, dtype, 12)
    scale = 1.0 / math.sqrt(D)
    print(f"[case] patches behind {dq} B{B} V{V} H{H} {Himg}x{Wimg} D{D} P{P} {projection}", flush=True)
    turn = (lambda t: t.permute(0, 1, 3, 2, 4)) if projection else (lambda t: t)
    leaves = [turn(t).contiguous().cuda().requires_grad_(True) for t in (q, k, v)]
    cdev = coords.cuda().requires_grad_(coords_grad)
    out = deform_sdpa_triton(*(turn(t) for t in leaves), cdev, Wimg, Himg, scale, coords_grad)
    names = kernels_of(lambda: out.backward(dout.cuda()))
    assert any(n.startswith(dq) for n in names) and any(n.startswith("bwd_dkdv_patch_kernel") for n in names), names
    want = oracle_bwd(*(t.float().numpy() for t in (q, k, v, coords, dout)), Wimg, Himg, scale, with_coords=coords_grad)
    got = [turn(t.grad) for t in leaves] + ([cdev.grad] if coords_grad else [])
    for a, b, name in zip(got, want, ("dq", "dk", "dv", "dcoords")):
        assert rel(a, b) < BAR[dtype], name


# 138 MB of pairs, 128 at a time: two groups of (batch, head) pairs
def test_patches_in_groups_of_pairs():
    q, k, v, dout, coords = inputs(1, 4, 270, 20, 20, 32, 10, torch.bfloat16, 13)
    assert 4 * 270 * 400 * 40 * 8 > 128 << 20
    print("[case] patches in two groups", flush=True)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    out = deform_sdpa_triton(*leaves, coords.cuda(), 20, 20, 0.25)
    names = kernels_of(lambda: out.backward(dout.cuda()))
    assert any(n.startswith("bwd_dkdv_patch_kernel") for n in names), names
    slices = [(0, 0), (0, 134), (0, 135), (0, 269)]
    for (b, h), (_, *want) in oracle_on_slices(q, k, v, coords, dout, 20, 20, 0.25, slices, forward=False).items():
        for leaf, w, name in zip(leaves, want, ("dq", "dk", "dv")):
            assert rel(leaf.grad[b:b + 1, :, h:h + 1], w) < BAR[torch.bfloat16], (name, h)
