"""dk/dv by cell lists, at list lengths where a block of 64 entries, a trip or a piece ends, and the scan of the list
lengths beyond one pass over 4096 keys: against the CPU oracle, at the bars of the other gradient tests (atomic order
1e-3 in fp32, the storage type's rounding 2e-2 in 16 bits)."""
import math

import pytest
import torch

from oracle import oracle_bwd
from ops.triton import deform_sdpa_triton
from parity_util import rel

pytestmark = pytest.mark.gpu
BAR = {torch.float32: 1e-3, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def check(q, k, v, coords, dout, W, Himg):
    scale = 1.0 / math.sqrt(q.shape[-1])
    leaves = [t.to("cuda:0").requires_grad_(True) for t in (q, k, v)]
    deform_sdpa_triton(*leaves, coords.to("cuda:0"), W, Himg, scale).backward(dout.to("cuda:0"))
    torch.cuda.synchronize()
    want = oracle_bwd(*(t.float().numpy() for t in (q, k, v, coords, dout)), W, Himg, scale)
    for t, w, name in zip(leaves, want, ("dq", "dk", "dv")):
        if coords.shape[3] * coords.shape[4] == 1 and name != "dv":      # one sample: p = 1, the others are zero
            continue
        assert rel(t.grad, w) < BAR[q.dtype], name


# lists of the cell (1, 2) only: plane kernels (recomputing), gather kernels (pairs handed over), and the ring of
# merged entries (D = 128, 16-bit)
@pytest.mark.parametrize("n", [1, 8, 9, 63, 64, 65, 128, 129, 800])
@pytest.mark.parametrize("D,side,dtype", [(16, 5, torch.float32), (32, 5, torch.float32), (32, 5, torch.bfloat16),
                                          (64, 5, torch.float16), (128, 5, torch.bfloat16), (16, 36, torch.float32), (16, 52, torch.bfloat16),
                                          (64, 24, torch.float32), (64, 24, torch.bfloat16), (128, 17, torch.bfloat16)],
                         ids=str)
def test_one_list_of_n_entries(D, side, dtype, n):
    g = torch.Generator().manual_seed(n)
    L = side * side
    P = max(2, (800 + L - 1) // L)                            # (two at least: with one sample dq and dk are zero)
    print(f"[case] one list D{D} {side}x{side} {dtype} n={n}", flush=True)
    q, k, v, dout = (torch.randn(1, 1, 2, L, D, generator=g).to(dtype) for _ in range(4))
    coords = torch.full((L * P, 2), -5.0)                      # outside: in no list
    at = torch.randperm(L * P, generator=g)[:n]
    coords[at] = (torch.rand(n, 2, generator=g) * 0.9 + 0.05 + torch.tensor([2.0, 1.0])) / (side - 1)
    check(q, k, v, coords.view(1, 1, L, 1, P, 2), dout, side, side)


@pytest.mark.parametrize("Himg,Wimg", [(62, 64), (63, 63), (64, 65), (90, 92)])
def test_scan_over_more_keys_than_one_pass(Himg, Wimg):      # (Himg+1)*(Wimg+1) = 4095, 4096, 4290, 8463 keys
    g = torch.Generator().manual_seed(Himg)
    L = Himg * Wimg
    print(f"[case] scan {Himg}x{Wimg}", flush=True)
    q, k, v, dout = (torch.randn(1, 1, 1, L, 16, generator=g) for _ in range(4))
    check(q, k, v, torch.rand(1, 1, L, 1, 2, 2, generator=g) * 1.1 - 0.05, dout, Wimg, Himg)


# one workgroup bins a (batch, key view) up to 2048 samples: the least, the most and one
# more, more keys than one turn of the scan, more than one batch item and view
@pytest.mark.parametrize("B,V,Himg,Wimg,P,dtype", [(1, 1, 2, 2, 2, torch.float32), (2, 2, 16, 16, 4, torch.float32),
                                                   (1, 3, 1, 683, 1, torch.bfloat16), (2, 2, 10, 17, 6, torch.float16),
                                                   (1, 1, 1, 2048, 1, torch.float32), (2, 1, 11, 17, 10, torch.float32)])
def test_binning_of_few_samples(B, V, Himg, Wimg, P, dtype):
    g = torch.Generator().manual_seed(P)
    L = Himg * Wimg
    print(f"[case] few samples B{B} V{V} {Himg}x{Wimg} P{P} {dtype}", flush=True)
    q, k, v, dout = (torch.randn(B, V, 2, L, 16, generator=g).to(dtype) for _ in range(4))
    check(q, k, v, torch.rand(B, V, L, V, P, 2, generator=g) * 1.2 - 0.1, dout, Wimg, Himg)
