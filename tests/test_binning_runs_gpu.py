"""Binning of dk/dv by runs of samples of one key view: a last run of one sample, runs over several query views, four and
eight samples a thread, more cells than samples, lists in several groups of query views (their rows beyond an XCD's L2),
samples that lie outside, the ordered lists of the deterministic backward, and images with more cells than the counters
in LDS hold. Against the CPU oracle at the bar of the other fp32 gradient tests (sums in another order)."""
import pytest
import torch

from oracle import oracle_bwd
from ops.triton import deform_sdpa_triton
from parity_util import rel

pytestmark = pytest.mark.gpu


def check(B, V, H, Himg, Wimg, D, P, dtype=torch.float32, bar=1e-3):
    print(f"[case] runs B{B} V{V} H{H} {Himg}x{Wimg} D{D} P{P} {dtype}", flush=True)
    g = torch.Generator().manual_seed(V * P + Himg)
    L = Himg * Wimg
    q, k, v, dout = (torch.randn(B, V, H, L, D, generator=g).to(dtype) for _ in range(4))
    coords = torch.rand(B, V, L, V, P, 2, generator=g) * 1.4 - 0.2
    coords[0, 0, 0, 0, 0, 0] = float("nan")
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    deform_sdpa_triton(*leaves, coords.cuda(), Wimg, Himg, 0.25).backward(dout.cuda())
    torch.cuda.synchronize()
    want = oracle_bwd(*(t.float().numpy() for t in (q, k, v, coords, dout)), Wimg, Himg, 0.25)
    for a, b, name in zip((t.grad for t in leaves), want, ("dq", "dk", "dv")):
        assert rel(a, b) < bar, name


# 2049 samples: a run and one more; 6 x 343 = 2058 and 3 x 1365 = 4095: runs across query views; 130x150 = 19781 cells
@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("B,V,Himg,Wimg,P", [(1, 1, 1, 683, 3), (2, 3, 7, 7, 14), (1, 3, 13, 35, 3), (1, 1, 130, 150, 2)])
def test_ends_of_runs(B, V, Himg, Wimg, P, deterministic):
    torch.use_deterministic_algorithms(deterministic)
    try:
        check(B, V, 2, Himg, Wimg, 16, P)
    finally:
        torch.use_deterministic_algorithms(False)


def test_eight_samples_a_thread():
    check(1, 5, 1, 41, 43, 16, 97)                 # 4.3 M samples


def test_groups_of_query_views():
    check(1, 3, 1, 60, 61, 256, 50, torch.bfloat16, 2e-2)        # 11 MB of query rows: three groups of a view each


def test_more_cells_than_the_counters_hold():
    check(1, 2, 1, 150, 160, 16, 2)                # 24311 cells: an atomic per sample
