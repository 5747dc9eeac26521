"""Fused deformable multi-view SDPA: the autograd front-end over libdsdpa.so.

Drop-in for the reference operator ``deform_sdpa_triton`` (``ops/triton.py:466``;
the module and function names are kept so ``from ops.triton import
deform_sdpa_triton`` keeps working -- there is no Triton here, the kernels are
hand-written HIP for gfx950 reached through a C ABI).

Contract mirrored from ``_fused_deform_sdpa`` (``ops/triton.py:377-466``):

* ``deform_sdpa_triton(q, k, v, coords, WIDTH, HEIGHT, sm_scale) -> out``,
  positional; q/k/v ``(B, N_VIEWS, N_HEADS, H*W, D)``, coords
  ``(B, N_VIEWS, H*W, N_VIEWS, N_SAMPLES, 2)`` normalised ``(x, y)``;
* gradients for q, k, v only; coords/WIDTH/HEIGHT/sm_scale get ``None``;
* ``AssertionError`` for unequal head dims, ``D`` outside {16,32,64,128,256},
  ``q.shape[3] != WIDTH*HEIGHT``, non-contiguous coords;
  ``NotImplementedError`` for an unsupported dtype;
* fp32 storage, or bf16/fp16 storage with fp32 accumulation.

The call itself -- checks, allocations, the autograd node -- is native (``csrc/dsdpa_torch.cpp``); what follows here
is what it does not take as it is: the errors, and the layouts and types that are copied first.

Differences, all on purpose: coords are not cloned or pre-scaled (the kernels
un-normalise), ``out``/``dq`` are not zero-filled first, no scaled copy of K is
made, out-of-image taps follow the eager operator's per-tap zero padding
(``ops/torch.py:14-15``) rather than ``ops/triton.py:129,135-136``, strided
q/k/v are read in place where the head dimension is contiguous (and copied
otherwise) instead of asserted, dout is made contiguous, and only the
log-sum-exp is saved on top of the inputs and output.
"""
import operator

import torch

from . import _native

_DTYPES = (torch.float32, torch.bfloat16, torch.float16)

# The backward runs its dk/dv side beside the dq side on a second stream of the library's (forked from and joined
# to the caller's stream inside the call). True keeps every launch on the caller's stream (same results).
SINGLE_STREAM = False

_apply = None


def _check_inputs(q, k, v, coords, WIDTH, HEIGHT):
    """Raises what the reference raises (``ops/triton.py:367-375,385-388``), and this build's own errors."""
    if q.dtype not in _DTYPES:
        raise NotImplementedError(f"unsupported dtype {q.dtype}")
    assert q.dim() == 5 and k.shape == q.shape and v.shape == q.shape, "q, k, v must share (B, V, H, L, D)"
    assert q.shape[-1] == k.shape[-1] == v.shape[-1]
    assert q.shape[-1] in {16, 32, 64, 128, 256}
    assert q.shape[3] == WIDTH * HEIGHT
    assert coords.is_contiguous()
    B, V, H, L, D = q.shape
    if coords.dim() != 6 or coords.shape[:4] != (B, V, L, V) or coords.shape[-1] != 2:
        raise RuntimeError(f"coords must be (B, V, L, V, P, 2) = ({B}, {V}, {L}, {V}, P, 2), got {tuple(coords.shape)}")
    if k.dtype != q.dtype or v.dtype != q.dtype:
        raise RuntimeError("q, k, v must share one dtype")
    if not q.is_cuda:
        raise RuntimeError("deform_sdpa_triton runs on the GPU only (HIP kernels); "
                           "use ops.torch.deform_sdpa_torch for an eager operator")
    if not (k.device == q.device and v.device == q.device and coords.device == q.device):
        raise RuntimeError("q, k, v, coords must be on one device")
    if B < 1 or V < 1 or H < 1 or L < 1 or coords.shape[4] < 1:
        _native.check(_native.ERR_BAD_SHAPE)


def _mend_and_apply(q, k, v, coords, WIDTH, HEIGHT, sm_scale, *extra):
    _check_inputs(q, k, v, coords, WIDTH, HEIGHT)
    # strided q, k, v are read in place where the kernels can (the reference's forward takes their strides,
    # ops/triton.py:396-405): head dimension contiguous, rows 16-byte aligned, k and v laid out alike
    if _native.strides_arg(q, k, v) is False:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if coords.dtype != torch.float32:
        coords = coords.float()
    out = _apply(SINGLE_STREAM, q, k, v, coords, operator.index(WIDTH), operator.index(HEIGHT), float(sm_scale), *extra)
    if out is None:
        raise RuntimeError("deform_sdpa_triton: the arguments are not ones the library takes")
    return out


def deform_sdpa_triton(*args):
    """``deform_sdpa_triton(q, k, v, coords, WIDTH, HEIGHT, sm_scale[, coords_grad]) -> out``, positional.

    ``coords_grad`` is an argument the reference does not have. Left out (or False) coords get no gradient, as in the
    reference (``ops/triton.py:464``); True asks for it, the one the eager operator gets through grid_sample
    (``ops/torch.py:14-15``)."""
    global _apply
    if _apply is None:
        _apply = _native.load_torch().apply
    if not 7 <= len(args) <= 8:
        raise TypeError("deform_sdpa_triton takes 7 arguments and an optional coords_grad flag")
    out = _apply(SINGLE_STREAM, *args)
    if out is None:
        out = _mend_and_apply(*args)
    if isinstance(out, int):
        _native.check(out)
    return out
