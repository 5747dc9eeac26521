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

An ordinary call -- checks, allocations, the autograd node -- is native (``csrc/dsdpa_torch.cpp``). Every other call
takes the ``torch.autograd.Function`` below, the general route: the errors, and the callers that PyTorch follows or
refuses by way of that class (``torch.jit.trace``, which records it; forward-mode AD and the ``torch.func``
transforms, for which the operator has no rule; dispatch modes and tensor subclasses).

Differences, all on purpose: coords are not cloned or pre-scaled (the kernels
un-normalise), ``out``/``dq`` are not zero-filled first, no scaled copy of K is
made, out-of-image taps follow the eager operator's per-tap zero padding
(``ops/torch.py:14-15``) rather than ``ops/triton.py:129,135-136``, strided
q/k/v are read in place where the head dimension is contiguous (and copied
otherwise) instead of asserted, dout is made contiguous, and only the
log-sum-exp is saved on top of the inputs and output.
"""
import contextlib

import torch

from . import _native

_SUFFIX = {torch.float32: "f32", torch.bfloat16: "bf16", torch.float16: "f16"}
_DTYPE_CODE = {torch.float32: _native.DSDPA_F32, torch.bfloat16: _native.DSDPA_BF16,
               torch.float16: _native.DSDPA_F16}

# The backward runs its dk/dv side beside the dq side on a second stream of the library's (forked from and joined
# to the caller's stream inside the call). True keeps every launch on the caller's stream (same results);
# read when a backward runs.
SINGLE_STREAM = False

_apply = None


def _check_inputs(q, k, v, coords, WIDTH, HEIGHT):
    """Raises what the reference raises (``ops/triton.py:367-375,385-388``), and this build's own errors."""
    if q.dtype not in _SUFFIX:
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


def _packed(t, align=16):
    """Contiguous, and at an address that the kernels' vector loads take (a contiguous view may begin at any element)."""
    t = t.contiguous()
    return t if t.data_ptr() % align == 0 else t.clone(memory_format=torch.contiguous_format)


def _check_saved(q, k, v, coords, out, lse, do):
    """Saved-tensor hooks may bring back other tensors than were saved. What does not fit the gradient's shape and device
    is refused: the kernels would read beyond it."""
    if q.dim() != 5 or q.shape[4] not in {16, 32, 64, 128, 256}:
        _native.check(_native.ERR_HEAD_DIM)
    B, V, H, L, D = q.shape
    if not (all(t.shape == do.shape and t.dtype == q.dtype for t in (q, k, v, out)) and q.dtype in _SUFFIX
            and lse.shape == (B, V, H, L) and coords.dim() == 6 and coords.shape[:4] == (B, V, L, V)
            and coords.shape[4] >= 1 and coords.shape[5] == 2 and lse.dtype == coords.dtype == torch.float32
            and all(t.device == do.device for t in (q, k, v, coords, out, lse))):
        raise RuntimeError("deform_sdpa_triton: a tensor saved for the backward came back with another shape, type or device")


@contextlib.contextmanager
def _not_traced():
    """Inside, sizes are plain ints also while ``torch.jit.trace`` records the caller. (It records the Function as a
    node that calls it again, so nothing depends on a size having been read. The buffers are made outside: the output has
    to be one that the tracer knows.)"""
    state = torch._C._get_tracing_state()
    torch._C._set_tracing_state(None)
    try:
        yield
    finally:
        torch._C._set_tracing_state(state)


class _fused_deform_sdpa(torch.autograd.Function):
    """The general route. Every buffer comes from ``torch.empty``, so that dispatch modes see it."""

    @staticmethod
    def forward(ctx, q, k, v, coords, WIDTH, HEIGHT, sm_scale, *extra):
        if len(extra) > 1:
            raise TypeError("deform_sdpa_triton takes 7 arguments and an optional coords_grad flag")
        ctx.n_inputs = 7 + len(extra)
        ctx.coords_grad = bool(extra[0]) if extra else False
        lib = _native.load()
        with _not_traced():
            _check_inputs(q, k, v, coords, WIDTH, HEIGHT)
            B, V, H, L, D = q.shape
            P = coords.shape[-2]
            # strided q, k, v are read in place where the kernels can (the reference's forward takes their strides,
            # ops/triton.py:396-405): head dimension contiguous, rows 16-byte aligned, k and v laid out alike
            strides = _native.strides_arg(q, k, v)
        if strides is False:
            q, k, v = _packed(q), _packed(k), _packed(v)
            strides = None
        if coords.dtype != torch.float32:
            coords = coords.float()
        coords = _packed(coords, 8)                                         # (read as pairs)
        out = torch.empty((B, V, H, L, D), device=q.device, dtype=q.dtype)  # contiguous whatever q's layout
        lse = torch.empty((B, V, H, L), device=q.device, dtype=torch.float32)
        ws_bytes = lib.dsdpa_fwd_workspace_bytes(_DTYPE_CODE[q.dtype], B, V, H, HEIGHT, WIDTH, D, P)
        ws = torch.empty(ws_bytes, device=q.device, dtype=torch.uint8)     # scratch, not saved for backward
        with torch.cuda.device(q.device):
            rc = getattr(lib, "dsdpa_fwd_" + _SUFFIX[q.dtype])(
                q.data_ptr(), k.data_ptr(), v.data_ptr(), coords.data_ptr(), out.data_ptr(), lse.data_ptr(),
                ws.data_ptr() if ws_bytes else None, B, V, H, HEIGHT, WIDTH, D, P, float(sm_scale), strides,
                torch.cuda.current_stream(q.device).cuda_stream)
        _native.check(rc)
        ctx.save_for_backward(q, k, v, coords, out, lse)
        ctx.sm_scale = float(sm_scale)
        ctx.WIDTH, ctx.HEIGHT = WIDTH, HEIGHT
        return out

    @staticmethod
    def backward(ctx, do):
        q, k, v, coords, out, lse = ctx.saved_tensors
        lib = _native.load()
        with _not_traced():
            _check_saved(q, k, v, coords, out, lse, do)
            B, V, H, L, D = q.shape
            P = coords.shape[-2]
            strides = _native.strides_arg(q, k, v)
        do = _packed(do if do.dtype == q.dtype else do.to(q.dtype))
        dq, dk, dv = (torch.empty((B, V, H, L, D), device=q.device, dtype=q.dtype) for _ in range(3))
        if strides is False:                            # (from a hook: forward saves contiguous, or readable in place)
            q, k, v = _packed(q), _packed(k), _packed(v)
            strides = None
        coords, out, lse = _packed(coords, 8), _packed(out), _packed(lse)
        dcoords = torch.empty_like(coords) if ctx.coords_grad and ctx.needs_input_grad[3] else None
        # torch.use_deterministic_algorithms(True) selects the bitwise reproducible backward
        flags = _native.FLAG_DETERMINISTIC if torch.are_deterministic_algorithms_enabled() else 0
        if flags and dcoords is not None:
            raise RuntimeError("deform_sdpa_triton: the coordinate gradient has no deterministic implementation "
                               "(it sums over heads with float atomics); turn one of the two off")
        if dcoords is not None:
            flags |= _native.FLAG_COORDS_GRAD
        if SINGLE_STREAM:
            flags |= _native.FLAG_SINGLE_STREAM
        ws_bytes = lib.dsdpa_bwd_workspace_bytes(_DTYPE_CODE[q.dtype], B, V, H, ctx.HEIGHT, ctx.WIDTH, D, P, flags)
        ws = torch.empty(ws_bytes, device=q.device, dtype=torch.uint8)
        with torch.cuda.device(q.device):
            rc = getattr(lib, "dsdpa_bwd_" + _SUFFIX[q.dtype])(
                q.data_ptr(), k.data_ptr(), v.data_ptr(), coords.data_ptr(), out.data_ptr(), lse.data_ptr(),
                do.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                dcoords.data_ptr() if dcoords is not None else None, ws.data_ptr(), B, V, H, ctx.HEIGHT, ctx.WIDTH, D, P,
                ctx.sm_scale, strides, flags, torch.cuda.current_stream(q.device).cuda_stream)
        _native.check(rc)
        return (dq, dk, dv, dcoords) + (None,) * (ctx.n_inputs - 4)


def deform_sdpa_triton(*args):
    """``deform_sdpa_triton(q, k, v, coords, WIDTH, HEIGHT, sm_scale[, coords_grad]) -> out``, positional.

    ``coords_grad`` is an argument the reference does not have. Left out (or False) coords get no gradient, as in the
    reference (``ops/triton.py:464``); True asks for it, the one the eager operator gets through grid_sample
    (``ops/torch.py:14-15``)."""
    global _apply
    if _apply is None:
        _apply = _native.load_torch().bind(_native.check, globals())
    out = _apply(*args)
    return _fused_deform_sdpa.apply(*args) if out is None else out
