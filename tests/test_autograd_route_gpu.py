"""The operator under the ways PyTorch follows a call other than by requires_grad, and what its backward reads and
raises at the time it runs: where the autograd node is native, nothing of that may be passed by."""
import pytest
import torch
from torch.autograd import forward_ad

from ops import _native
from ops import triton as op

pytestmark = pytest.mark.gpu

B, V, H, HIMG, WIMG, D, P = 1, 2, 2, 3, 4, 32, 3


def inputs(seed=0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, V, H, HIMG * WIMG, D, generator=g).to(dtype).cuda() for _ in range(3))
    return [q, k, v, torch.rand(B, V, HIMG * WIMG, V, P, 2, generator=g).cuda()]


def call(q, k, v, c):
    return op.deform_sdpa_triton(q, k, v, c, WIMG, HIMG, 0.3)


@pytest.mark.parametrize("which", [0, 3])
@pytest.mark.parametrize("requires_grad", [False, True])
@pytest.mark.parametrize("grad_mode", [False, True])
def test_forward_mode_is_refused(which, requires_grad, grad_mode):
    print(f"[case] dual {which} {requires_grad} {grad_mode}", flush=True)
    args = inputs()
    args[0].requires_grad_(requires_grad)
    with forward_ad.dual_level(), torch.set_grad_enabled(grad_mode):
        args[which] = forward_ad.make_dual(args[which], torch.ones_like(args[which]))
        with pytest.raises(NotImplementedError, match="jvp"):
            call(*args)


@pytest.mark.parametrize("grad_mode", [False, True])
def test_scale_in_a_tensor_is_an_input(grad_mode):
    print(f"[case] tensor scale {grad_mode}", flush=True)
    q, k, v, c = inputs()
    want = call(q, k, v, c)
    scale = torch.tensor(0.3, requires_grad=True)
    with torch.set_grad_enabled(grad_mode):
        out = op.deform_sdpa_triton(q, k, v, c, WIMG, HIMG, scale)
    assert torch.equal(out, want) and out.requires_grad == grad_mode
    if grad_mode:
        out.backward(torch.ones_like(out))               # (as in the reference: it gets no gradient)
        assert scale.grad is None
    with forward_ad.dual_level(), torch.set_grad_enabled(grad_mode), pytest.raises(NotImplementedError, match="jvp"):
        op.deform_sdpa_triton(q, k, v, c, WIMG, HIMG, forward_ad.make_dual(scale.detach(), torch.ones(())))


def test_function_transforms_are_refused():
    print("[case] transforms", flush=True)
    q, k, v, c = inputs()
    for f in (lambda x: call(q * x, k, v, c), lambda x: call(q, k, v, c) * x):
        with pytest.raises(RuntimeError, match="functorch"):
            torch.func.vmap(f)(torch.ones(2, device="cuda"))
        with pytest.raises(RuntimeError, match="functorch"):
            torch.func.grad(lambda x: f(x).sum())(torch.ones((), device="cuda"))


@pytest.mark.parametrize("requires_grad", [False, True])
@pytest.mark.parametrize("layout", ["plain", "copied"])
def test_traced_module_follows_its_inputs(requires_grad, layout):
    print(f"[case] trace {requires_grad} {layout}", flush=True)

    def f(q, k, v, c):
        if layout == "copied":
            q, c = q.transpose(3, 4).contiguous().transpose(3, 4), c.double()
        return call(q, k, v, c) * 2.0
    first, second = inputs(0), inputs(1)
    for args in (first, second):
        args[0].requires_grad_(requires_grad)
    traced = torch.jit.trace(f, tuple(first))
    for _ in range(3):                                   # (the executor specialises on the first runs)
        got, want = traced(*second), f(*second)
        assert torch.equal(got, want)
        if requires_grad:
            dout = torch.ones_like(want)
            assert torch.equal(*(torch.autograd.grad(o, second[0], dout)[0] for o in (got, want)))


def test_dispatch_mode_sees_the_buffers():
    print("[case] dispatch mode", flush=True)
    from torch._subclasses import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.n += 1
            return func(*args, **(kwargs or {}))
    args = inputs()
    want = call(*args)
    with Seen() as seen:
        assert torch.equal(call(*args), want)
    assert seen.n > 0
    with FakeTensorMode(allow_non_fake_inputs=True), pytest.raises(RuntimeError):
        call(*args)


@pytest.mark.parametrize("route", ["native", "general"])
def test_dispatch_mode_around_the_backward_sees_its_buffers(route):
    print(f"[case] dispatch mode backward {route}", flush=True)
    from torch._subclasses import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Made(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.n += func is torch.ops.aten.empty.memory_format
            return func(*args, **(kwargs or {}))

    def forward():
        args = inputs()
        args[0].requires_grad_(True)
        f = op.deform_sdpa_triton if route == "native" else op._fused_deform_sdpa.apply
        return args[0], f(*args, WIMG, HIMG, 0.3)
    (q, out), (want, same) = forward(), forward()
    dout = torch.ones_like(out)
    same.backward(dout)
    with Made() as made:
        out.backward(dout)
    assert made.n >= 4 and torch.equal(q.grad, want.grad)        # dq, dk, dv and the workspace
    q, out = forward()
    with FakeTensorMode(allow_non_fake_inputs=True), pytest.raises(RuntimeError):
        out.backward(dout)


@pytest.mark.parametrize("route", ["native", "general"])
def test_backward_raises_the_librarys_error(route):
    print(f"[case] backward error {route}", flush=True)
    args = inputs()
    args[0].requires_grad_(True)
    # saved tensors come back with a head dimension that the library refuses
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t[..., :8].contiguous() if t.shape[-1] == D else t):
        out = call(*args) if route == "native" else op._fused_deform_sdpa.apply(*args, WIMG, HIMG, 0.3)
    with pytest.raises(_native.DsdpaError, match="head dim"):
        out.backward(torch.ones_like(out))


@pytest.mark.parametrize("route", ["native", "general"])
def test_single_stream_is_read_when_the_backward_runs(route, monkeypatch):
    print(f"[case] single stream {route}", flush=True)
    n, p = 64, 8                                         # 4 * 64 * 32^2 * 8 query samples: the least that may fork
    q, k, v = (torch.randn(4, 1, n, 32 * 32, 16, device="cuda") for _ in range(3))
    args = [q.requires_grad_(True), k, v, torch.rand(4, 1, 32 * 32, 1, p, 2, device="cuda")]
    f = op.deform_sdpa_triton if route == "native" else op._fused_deform_sdpa.apply
    out = f(*args, 32, 32, 0.3)

    class Asked:
        times = 0

        def __bool__(self):
            self.times += 1
            return True
    monkeypatch.setattr(op, "SINGLE_STREAM", Asked())
    out.backward(torch.ones_like(out))
    assert op.SINGLE_STREAM.times == 1


@pytest.mark.parametrize("route", ["native", "general"])
def test_profile_carries_the_operators_name(route):
    print(f"[case] profile {route}", flush=True)
    args = inputs()
    args[0].requires_grad_(True)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        out = call(*args) if route == "native" else op._fused_deform_sdpa.apply(*args, WIMG, HIMG, 0.3)
        out.backward(torch.ones_like(out))
    names = {e.key for e in prof.key_averages()}
    assert {"_fused_deform_sdpa", "_fused_deform_sdpaBackward"} <= names
    assert "fused_deform_sdpa" in out.grad_fn.name() and "fused_deform_sdpa" in repr(out)


@pytest.mark.parametrize("route", ["native", "general"])
@pytest.mark.parametrize("which", range(5))
def test_views_at_an_odd_address_are_copied(route, which):
    print(f"[case] odd address {route} {which}", flush=True)
    args = inputs(dtype=torch.bfloat16) + inputs(1, torch.bfloat16)[:1]

    def odd(t):                                          # contiguous, one element after an aligned address
        return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)

    def step(q, k, v, c, dout):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v, c)]
        f = op.deform_sdpa_triton if route == "native" else op._fused_deform_sdpa.apply
        out = f(*leaves, WIMG, HIMG, 0.3, True)
        out.backward(dout)
        return [out.detach()] + [t.grad for t in leaves]
    want = step(*args)
    args[which] = odd(args[which])
    got = step(*args)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    for a, b in zip(got[2:], want[2:]):      # float atomics: sums in another order, one step of bf16 (2^-8) at most
        assert (a.float() - b.float()).abs().max() <= 2.0 ** -7 * b.float().abs().max()


@pytest.mark.parametrize("route", ["native", "general"])
def test_saved_tensors_from_hooks(route):
    print(f"[case] hooks {route}", flush=True)
    f = op.deform_sdpa_triton if route == "native" else op._fused_deform_sdpa.apply

    def dq(unpack):
        args = inputs()
        args[0].requires_grad_(True)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = f(*args, WIMG, HIMG, 0.3)
        out.backward(torch.ones_like(out))
        return args[0].grad
    want = dq(lambda t: t)
    assert torch.equal(dq(lambda t: t.transpose(-1, -2).contiguous().transpose(-1, -2)), want)      # layouts are mended
    for unpack in (torch.Tensor.cpu, torch.Tensor.double, lambda t: t[..., :1, :].contiguous()):
        with pytest.raises(RuntimeError, match="saved for the backward"):
            dq(unpack)
