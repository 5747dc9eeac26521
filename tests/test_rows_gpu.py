"""Row kernels (one query row per slot of lanes, taps from memory): every lane split, query rows that end inside a wave, a last pass
of one sample, of an odd number and of a whole pass, strided inputs, the coordinate gradient and the pairs handed on to
dk/dv. Against the CPU oracle at the bars of the other parity tests."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle_bwd, oracle_fwd
from ops.triton import deform_sdpa_triton
from parity_util import kernels_of, oracle_on_slices, rel

pytestmark = pytest.mark.gpu
BAR = {torch.float32: (1e-4, 1e-3), torch.bfloat16: (2e-2, 2e-2), torch.float16: (2e-2, 2e-2)}


def check(B, V, H, Himg, Wimg, D, P, dtype, coords_grad=False, projection=False):
    print(f"[case] rows B{B} V{V} H{H} {Himg}x{Wimg} D{D} P{P} {dtype} {coords_grad} {projection}", flush=True)
    g = torch.Generator().manual_seed(V * P + D)
    L, scale = Himg * Wimg, 1.0 / math.sqrt(D)
    shape = (B, V, L, H, D) if projection else (B, V, H, L, D)
    leaves = [torch.randn(shape, generator=g).to(dtype) for _ in range(3)]
    coords = torch.rand(B, V, L, V, P, 2, generator=g) * 1.2 - 0.1
    dout = torch.randn(B, V, H, L, D, generator=g).to(dtype)
    dev = [t.to("cuda:0").requires_grad_(True) for t in leaves]
    cdev = coords.to("cuda:0").requires_grad_(coords_grad)
    view = (lambda t: t.permute(0, 1, 3, 2, 4)) if projection else (lambda t: t)
    out = deform_sdpa_triton(*(view(t) for t in dev), cdev, Wimg, Himg, scale, coords_grad)
    out.backward(dout.to("cuda:0"))
    torch.cuda.synchronize()
    n = [view(t).float().contiguous().numpy() for t in leaves]
    assert rel(out, oracle_fwd(*n, coords.numpy(), Wimg, Himg, scale)[0]) < BAR[dtype][0]
    want = oracle_bwd(*n, coords.numpy(), dout.float().numpy(), Wimg, Himg, scale, with_coords=coords_grad)
    got = [view(t.grad) for t in dev] + ([cdev.grad] if coords_grad else [])
    for a, b, name in zip(got, want, ("dq", "dk", "dv", "dcoords")):
        if V * P == 1 and name in ("dq", "dk", "dcoords"):       # one sample: p = 1, the others are zero
            continue
        assert rel(a, b) < BAR[dtype][1], name


# 23x29: planes too large for LDS from D = 64 fp32 on, below that few samples of a staged shape
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("V,P", [(1, 1), (3, 2), (2, 3), (3, 5)])
def test_rows_against_the_oracle(V, P, D, dtype):
    check(1, V, 3, 23, 29, D, P, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=str)
@pytest.mark.parametrize("D,P", [(32, 3), (64, 8), (128, 2), (256, 5)])
def test_rows_with_the_coordinate_gradient(D, P, dtype):
    check(2, 2, 3, 23, 29, D, P, dtype, coords_grad=True, projection=True)


# more than 16 and more than 32 samples a row, from 2048 and 4096 waves of rows on
@pytest.mark.parametrize("V,H,P,dtype", [(2, 10, 12, torch.float32), (2, 20, 10, torch.bfloat16), (3, 14, 21, torch.bfloat16)], ids=str)
def test_many_rows(V, H, P, dtype):
    check(1, V, H, 30, 31, 64, P, dtype)


# the binning of few samples beside the rows of dq: all its places taken, two short of it, more groups than XCDs, a workgroup's threads
# and one more; 2052 samples, and rows of 1 KB with the coordinate gradient, are binned in launches of their own
@pytest.mark.parametrize("coords_grad", [False, True], ids=["plain", "coords"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("B,V,H,Himg,Wimg,D,P", [(1, 2, 3, 16, 32, 64, 2), (5, 2, 1, 11, 31, 32, 3), (1, 1, 2, 16, 16, 128, 1),
                                                 (1, 1, 2, 1, 257, 16, 1), (2, 2, 2, 10, 12, 256, 3), (1, 2, 2, 19, 18, 64, 3)])
def test_binning_beside_the_rows(B, V, H, Himg, Wimg, D, P, dtype, coords_grad):
    names = kernels_of(lambda: check(B, V, H, Himg, Wimg, D, P, dtype, coords_grad))
    beside = V * Himg * Wimg * P <= 2048 and not (coords_grad and D == 256 and dtype == torch.float32)
    rows = [n for n in names if n.startswith("bwd_dq_rows_kernel")]
    assert len(rows) == 1 and rows[0].endswith("true>" if beside else "false>"), names      # (last argument: bins)
    assert any(n.startswith("bin_") for n in names) == (not beside), names


# 5.94 workgroups of rows a CU, and 5.03, which leave a sixth of the last one's time empty: rows and a wave per row
@pytest.mark.parametrize("H,kernels", [(13, ("fwd_rows_kernel", "bwd_dq_rows_kernel")), (11, ("fwd_gather_kernel", "bwd_dq_gather_kernel"))])
def test_rows_where_their_workgroups_fill_the_cus(H, kernels):
    print(f"[case] rows or a wave per row, H {H}", flush=True)
    g = torch.Generator().manual_seed(H)
    L, dev = 30 * 31, [torch.randn(1, 2, H, 30 * 31, 64, generator=g).cuda().requires_grad_(True) for _ in range(3)]
    coords, dout = torch.rand(1, 2, L, 2, 20, 2, generator=g), torch.randn(1, 2, H, L, 64, generator=g)
    out = []
    names = kernels_of(lambda: out.append(deform_sdpa_triton(*dev, coords.cuda(), 31, 30, 0.125)))
    names |= kernels_of(lambda: out[0].backward(dout.cuda()))
    assert all(any(n.startswith(k) for n in names) for k in kernels), names
    slices = [(0, 0), (0, H - 1)]
    for (b, h), (ro, *want) in oracle_on_slices(*(t.detach().cpu() for t in dev), coords, dout, 31, 30, 0.125, slices).items():
        for a, w, bar in zip([out[0]] + [t.grad for t in dev], [ro] + want, (1e-4, 1e-3, 1e-3, 1e-3)):
            assert rel(a[b:b + 1, :, h:h + 1], w) < bar, h


# infinite V at the taps of a row's last sample, rows of an odd number of samples: infinite, not NaN
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize("V,P", [(1, 1), (3, 1), (1, 5)])
def test_infinite_values(V, P, dtype):
    print(f"[case] rows, infinite V, {V} x {P} {dtype}", flush=True)
    g = torch.Generator().manual_seed(V + P)
    L = 18 * 17
    q, k, v = (torch.randn(1, V, 2, L, 32, generator=g).to(dtype) for _ in range(3))
    coords = torch.rand(1, V, L, V, P, 2, generator=g) * 0.9 + 0.05            # (no tap outside)
    v[0, V - 1, :, 3 * 17 + 5] = float("inf")
    out = deform_sdpa_triton(*(t.cuda() for t in (q, k, v, coords)), 17, 18, 0.2).double().cpu().numpy()
    want = oracle_fwd(*(t.float().numpy() for t in (q, k, v, coords)), 17, 18, 0.2)[0]
    assert 0 < np.isinf(want).sum() < want.size // 4 and not np.isnan(want).any()
    assert np.array_equal(np.isinf(out), np.isinf(want)) and not np.isnan(out).any()
