"""Staged forward and dq with eight fp32 elements a lane (D = 32 and 64, launches of many query rows): query rows that end inside a
wave and a workgroup, passes that end inside a run of samples, strided inputs. (These lists are long: the form that hands its
pairs on is among the tests of dk/dv by patches.) Against the CPU oracle at the bars of the other fp32 parity tests."""
import math

import pytest
import torch

from oracle import oracle_bwd, oracle_fwd
from ops.triton import deform_sdpa_triton
from parity_util import kernels_of, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("projection", [False, True])
@pytest.mark.parametrize("B,V,H,Himg,Wimg,D,P", [(2, 4, 32, 18, 17, 32, 5), (2, 3, 64, 9, 11, 32, 8), (2, 6, 16, 13, 12, 64, 8), (1, 3, 96, 11, 13, 64, 9)])
def test_wide_split_against_the_oracle(B, V, H, Himg, Wimg, D, P, projection):
    print(f"[case] wide B{B} V{V} H{H} {Himg}x{Wimg} D{D} P{P} {projection}", flush=True)
    g = torch.Generator().manual_seed(D + P)
    L, scale = Himg * Wimg, 1.0 / math.sqrt(D)
    shape = (B, V, L, H, D) if projection else (B, V, H, L, D)
    leaves = [torch.randn(shape, generator=g) for _ in range(3)]
    coords = torch.rand(B, V, L, V, P, 2, generator=g) * 1.2 - 0.1
    dout = torch.randn(B, V, H, L, D, generator=g)
    dev = [t.to("cuda:0").requires_grad_(True) for t in leaves]
    view = (lambda t: t.permute(0, 1, 3, 2, 4)) if projection else (lambda t: t)
    out = deform_sdpa_triton(*(view(t) for t in dev), coords.to("cuda:0"), Wimg, Himg, scale)
    names = kernels_of(lambda: out.backward(dout.to("cuda:0")))
    assert f"bwd_dq_slot_kernel<F32, {D}, 8, false, 1, false>" in names, names
    n = [view(t).contiguous().numpy() for t in leaves]
    assert rel(out, oracle_fwd(*n, coords.numpy(), Wimg, Himg, scale)[0]) < 1e-4
    want = oracle_bwd(*n, coords.numpy(), dout.numpy(), Wimg, Himg, scale)
    for a, b, name in zip(dev, want, ("dq", "dk", "dv")):
        assert rel(view(a.grad), b) < 1e-3, name
