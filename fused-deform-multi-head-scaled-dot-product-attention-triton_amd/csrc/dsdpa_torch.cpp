// Host side of the PyTorch operator: argument checks, output and workspace allocation, the autograd node and the
// calls of the C ABI (include/dsdpa.h), in C++. The counterpart of the reference's autograd.Function
// (ops/triton.py:377-466) for ordinary calls; ops/triton.py holds the Python entry point and an autograd.Function,
// the general route of every call that is handed back to it here.
//
// Why native: at the small end of the operator's range the GPU finishes long before the host has enqueued the next
// launch. With the checks, torch.empty calls, ctypes conversions and autograd.Function of Python a training step
// took 165 us of host time whatever its size (views x samples 2x2 of the sweep, 18x18, 32 heads: 162 us a step for
// 86 us of kernels).
//
// bind(check, globals) -> apply: check(code) is the Python function that raises for a library error code, globals the
// Python module's, whose SINGLE_STREAM a backward reads when it runs.
// apply(q, k, v, coords, WIDTH, HEIGHT, sm_scale[, coords_grad]) -> out; None when the arguments
// are wrong, or when PyTorch follows the call in a way that goes by an autograd.Function (followed()): nothing has been
// done then, and the call takes the general route, which raises or is followed. No tensor is kept from one call for
// the next.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/accumulate_grad.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/dsdpa.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Node;
using torch::autograd::variable_list;

struct Strides {
    long long st[8];
    bool given = false;                  // false: everything contiguous
    const long long *ptr() const { return given ? st : nullptr; }
};

bool aligned(const Tensor &t, uintptr_t bytes) { return ((uintptr_t)t.data_ptr() & (bytes - 1)) == 0; }

// Contiguous, and at an address that the kernels' vector loads take (a contiguous view may begin at any element).
Tensor packed(const Tensor &t, uintptr_t bytes = 16)
{
    Tensor c = t.contiguous();
    return aligned(c, bytes) ? c : c.clone(at::MemoryFormat::Contiguous);
}

// Whether the kernels can read q, k, v where they lie: head dimension contiguous, k and v laid out alike, rows
// 16-byte aligned, the views and pixels of one (batch, head) within 2^30 elements (the kernels address them in 32
// bits). Fills the `strides` argument of the entry points.
bool readable_in_place(const Tensor &q, const Tensor &k, const Tensor &v, Strides *out)
{
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16)) return false;
    if (q.is_contiguous() && k.is_contiguous() && v.is_contiguous()) return true;
    const int64_t align = 16 / (int64_t)q.element_size(), V = q.size(1), L = q.size(3), D = q.size(4);
    for (const Tensor *t : {&q, &k, &v}) {
        const auto st = t->strides();
        if (st[4] != 1 || st[3] < D) return false;
        for (int i = 0; i < 4; ++i)
            if (st[i] < 0 || st[i] % align) return false;
        if ((V - 1) * st[1] + (L - 1) * st[3] + D > (1ll << 30) || st[1] > (1ll << 30)) return false;
    }
    if (k.strides() != v.strides()) return false;
    for (int i = 0; i < 4; ++i) {
        out->st[i] = q.stride(i);
        out->st[4 + i] = k.stride(i);
    }
    out->given = true;
    return true;
}

// at::detail::empty_cuda: the caching allocator without the dispatcher, and without the fill that at::empty does under
// torch.use_deterministic_algorithms (every element of every tensor handed out is written by the kernels, and nothing of a
// workspace is read that they have not written). A dispatch mode entered around a backward alone sees the buffers.
Tensor fresh(at::IntArrayRef shape, at::ScalarType type, const at::Device &dev)
{
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return at::empty(shape, at::TensorOptions(dev).dtype(type));
    return Tensor(at::detail::empty_cuda(shape, type, dev, std::nullopt));
}

// ... of t's shape and type, contiguous or with t's strides
Tensor fresh_as(const Tensor &t, bool strided)
{
    if (!strided) return fresh(t.sizes(), t.scalar_type(), t.device());
    if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return at::empty_strided(t.sizes(), t.strides(), t.options());
    return Tensor(at::detail::empty_strided_cuda(t.sizes(), t.strides(), t.scalar_type(), t.device()));
}

void *stream_of(const at::Device &dev)
{
    return (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
}

// What bind() was given, as a tuple kept for the process's lifetime (a graph may outlive the bound function).
PyObject *check_of(PyObject *bound) { return PyTuple_GET_ITEM(bound, 0); }

// SINGLE_STREAM now
bool single_stream(PyObject *bound)
{
    pybind11::gil_scoped_acquire gil;
    PyObject *flag = PyDict_GetItemString(PyTuple_GET_ITEM(bound, 1), "SINGLE_STREAM");
    Py_XINCREF(flag);
    const int on = flag ? PyObject_IsTrue(flag) : 0;
    Py_XDECREF(flag);
    if (on < 0) {
        python_error err;
        err.persist();
        throw std::move(err);
    }
    return on == 1;
}

// Raises the library's error in Python, by the bound check(), on the thread whose HIP error it reports. With the lock
// held; a C++ exception that carries the Python one, as autograd expects it from a node.
[[noreturn]] void raise_error(PyObject *check, int rc)
{
    if (PyObject *r = PyObject_CallFunction(check, "i", rc)) {
        Py_DECREF(r);
        PyErr_Format(PyExc_SystemError, "no exception for libdsdpa error %d", rc);
    }
    python_error err;
    err.persist();
    throw std::move(err);
}

int dtype_code(at::ScalarType t)
{
    return t == at::kFloat ? DSDPA_F32 : t == at::kBFloat16 ? DSDPA_BF16 : DSDPA_F16;
}

struct Call {
    int64_t W, H;
    double scale;
    bool coords_grad;
    PyObject *bound;
};

void check(int rc, PyObject *bound)
{
    if (rc == DSDPA_OK) return;
    pybind11::gil_scoped_acquire gil;
    raise_error(check_of(bound), rc);
}

// out and the log-sum-exp of every query row
std::pair<Tensor, Tensor> forward_pass(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &coords, const Call &c)
{
    RECORD_FUNCTION("_fused_deform_sdpa", std::vector<c10::IValue>());
    const at::Device dev = q.device();
    const c10::DeviceGuard on_device(dev);
    Strides st;
    TORCH_CHECK(readable_in_place(q, k, v, &st));
    const int B = (int)q.size(0), V = (int)q.size(1), H = (int)q.size(2), D = (int)q.size(4), P = (int)coords.size(4);
    const int W = (int)c.W, Hi = (int)c.H, code = dtype_code(q.scalar_type());
    Tensor out = fresh(q.sizes(), q.scalar_type(), dev);
    Tensor lse = fresh({q.size(0), q.size(1), q.size(2), q.size(3)}, at::kFloat, dev);
    Tensor ws;                                           // scratch, not kept for the backward
    void *wsp = nullptr;
    if (const size_t bytes = dsdpa_fwd_workspace_bytes(code, B, V, H, Hi, W, D, P)) {
        ws = fresh({(int64_t)bytes}, at::kByte, dev);
        wsp = ws.data_ptr();
    }
    const auto *cp = (const float *)coords.data_ptr();
    auto *lp = (float *)lse.data_ptr();
    void *s = stream_of(dev);
    int rc;
    if (code == DSDPA_F32)
        rc = dsdpa_fwd_f32((const float *)q.data_ptr(), (const float *)k.data_ptr(), (const float *)v.data_ptr(), cp, (float *)out.data_ptr(), lp,
                           wsp, B, V, H, Hi, W, D, P, (float)c.scale, st.ptr(), s);
    else
        rc = (code == DSDPA_BF16 ? dsdpa_fwd_bf16 : dsdpa_fwd_f16)(q.data_ptr(), k.data_ptr(), v.data_ptr(), cp, out.data_ptr(), lp, wsp, B, V,
                                                                   H, Hi, W, D, P, (float)c.scale, st.ptr(), s);
    check(rc, c.bound);
    return {out, lse};
}

// Saved-tensor hooks may bring back other tensors than were saved: q, k, v, coords, out and lse as the kernels read them.
// What does not fit dout's shape and device is refused here: the kernels would read beyond it.
void usable(variable_list &saved, const Tensor &dout, PyObject *bound)
{
    Tensor &q = saved[0], &k = saved[1], &v = saved[2], &coords = saved[3], &out = saved[4], &lse = saved[5];
    const int64_t D = q.dim() == 5 ? q.size(4) : 0;
    if (!(D == 16 || D == 32 || D == 64 || D == 128 || D == 256)) check(DSDPA_ERR_HEAD_DIM, bound);
    bool fits = q.sizes() == dout.sizes() && lse.sizes() == q.sizes().slice(0, 4) && lse.scalar_type() == at::kFloat;
    for (const Tensor *t : {&k, &v, &out}) fits &= t->sizes() == q.sizes() && t->scalar_type() == q.scalar_type();
    for (const Tensor &t : saved) fits &= t.device() == dout.device();
    fits &= coords.dim() == 6 && coords.size(0) == q.size(0) && coords.size(1) == q.size(1) && coords.size(2) == q.size(3) &&
            coords.size(3) == q.size(1) && coords.size(4) >= 1 && coords.size(5) == 2 && coords.scalar_type() == at::kFloat;
    fits &= q.scalar_type() == at::kFloat || q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf;
    TORCH_CHECK(fits, "deform_sdpa_triton: a tensor saved for the backward came back with another shape, type or device");
    Strides st;
    if (!readable_in_place(q, k, v, &st)) q = packed(q), k = packed(k), v = packed(v);
    coords = packed(coords, 8);
    out = packed(out);
    lse = packed(lse);
}

// Whether somebody is shown the gradient that goes into `node`: hooks of the tensor or the node, retain_grad, or a caller
// of torch.autograd.grad that asked for it. (A leaf's node hands it to no hook behind it: those, a data-parallel wrapper's, read .grad.)
bool shown(Node &node)
{
    const auto *exec = torch::autograd::get_current_graph_task_exec_info();
    if (exec && !exec->empty()) {
        const auto at = exec->find(&node);
        if (at != exec->end() && at->second.captures_) return true;
    }
    return !node.pre_hooks().empty() || !node.tensor_pre_hooks().empty() || !node.retains_grad_hooks().empty() ||
           (!node.post_hooks().empty() && !dynamic_cast<torch::autograd::AccumulateGrad *>(&node));
}

// Whether the gradients of those of q, k, v that are not contiguous go straight into the backward of the permutation that made them,
// and neither they nor what comes out of it is shown to anybody. Everyone else gets contiguous gradients, of which views can
// be made, whatever q, k and v look like.
bool only_permuted(const Tensor &q, const Tensor &k)
{
    const std::shared_ptr<Node> self = torch::autograd::get_current_node();
    if (!self || !self->post_hooks().empty()) return false;
    for (uint32_t i = 0; i < 3; ++i) {
        if ((i == 0 ? q : k).is_contiguous()) continue;
        Node *fn = self->next_edge(i).function.get();
        if (!fn) continue;                               // (no gradient asked for)
        const std::string name = fn->name();
        if ((name != "PermuteBackward0" && name != "TransposeBackward0") || shown(*fn)) return false;
        Node *from = fn->next_edge(0).function.get();
        if (from && shown(*from)) return false;
    }
    return true;
}

}  // namespace

// The autograd node. Outside the namespace for a plain name in graphs (torch::autograd::CppNode<fused_deform_sdpa>); the
// ranges in profiles are called as those of the general route's Function are.
struct fused_deform_sdpa : public torch::autograd::Function<fused_deform_sdpa> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &coords, const Call &c)
    {
        auto [out, lse] = forward_pass(q, k, v, coords, c);
        ctx->save_for_backward({q, k, v, coords, out, lse});
        ctx->saved_data["W"] = c.W;
        ctx->saved_data["H"] = c.H;
        ctx->saved_data["scale"] = c.scale;
        ctx->saved_data["bound"] = (int64_t)(intptr_t)c.bound;
        ctx->saved_data["coords_grad"] = c.coords_grad;
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        RECORD_FUNCTION("_fused_deform_sdpaBackward", std::vector<c10::IValue>());
        Tensor dout = grads[0];
        if (!dout.defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
        const at::Device dev = dout.device();
        const c10::DeviceGuard on_device(dev);
        PyObject *bound = (PyObject *)(intptr_t)ctx->saved_data["bound"].toInt();
        variable_list saved = ctx->get_saved_variables();
        usable(saved, dout, bound);
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &coords = saved[3], &out = saved[4], &lse = saved[5];
        if (dout.scalar_type() != q.scalar_type()) dout = dout.to(q.scalar_type());
        dout = packed(dout);
        const bool want_dcoords = ctx->saved_data["coords_grad"].toBool() && ctx->needs_input_grad(3);
        // (asked only where it makes a difference: taking the interpreter's lock costs a small step 2 us)
        const bool may_fork = lse.numel() * q.size(1) * coords.size(4) >= DSDPA_TWO_STREAMS_FROM;
        unsigned flags = may_fork && single_stream(bound) ? DSDPA_FLAG_SINGLE_STREAM : 0;
        if (at::globalContext().deterministicAlgorithms()) {       // the bitwise reproducible backward
            TORCH_CHECK(!want_dcoords, "deform_sdpa_triton: the coordinate gradient has no deterministic implementation "
                                       "(it sums over heads with float atomics); turn one of the two off");
            flags |= DSDPA_FLAG_DETERMINISTIC;
        }
        if (want_dcoords) flags |= DSDPA_FLAG_COORDS_GRAD;
        const int B = (int)q.size(0), V = (int)q.size(1), H = (int)q.size(2), D = (int)q.size(4), P = (int)coords.size(4);
        const int W = (int)ctx->saved_data["W"].toInt(), Hi = (int)ctx->saved_data["H"].toInt(), code = dtype_code(q.scalar_type());
        const float scale = (float)ctx->saved_data["scale"].toDouble();
        Strides st;
        readable_in_place(q, k, v, &st);
        // (of permuted inputs -- a linear layer's output split into heads -- the gradients go back through the permutation as they
        // are: contiguous ones would each be copied there, 10 us apiece of a step of 322 at 4 views of 40x28, 8 heads, D = 64, fp16)
        const bool as_inputs = st.given && q.is_non_overlapping_and_dense() && k.is_non_overlapping_and_dense() && only_permuted(q, k);
        if (as_inputs) flags |= DSDPA_FLAG_GRADS_AS_INPUTS;
        Tensor dq = fresh_as(q, as_inputs), dk = fresh_as(k, as_inputs), dv = fresh_as(v, as_inputs);
        Tensor dcoords = want_dcoords ? fresh(coords.sizes(), at::kFloat, dev) : Tensor();
        Tensor ws = fresh({(int64_t)dsdpa_bwd_workspace_bytes(code, B, V, H, Hi, W, D, P, flags)}, at::kByte, dev);
        const auto *cp = (const float *)coords.data_ptr(), *lp = (const float *)lse.data_ptr();
        float *dcp = want_dcoords ? (float *)dcoords.data_ptr() : nullptr;
        void *s = stream_of(dev);
        int rc;
        if (code == DSDPA_F32)
            rc = dsdpa_bwd_f32((const float *)q.data_ptr(), (const float *)k.data_ptr(), (const float *)v.data_ptr(), cp, (const float *)out.data_ptr(),
                               lp, (const float *)dout.data_ptr(), (float *)dq.data_ptr(), (float *)dk.data_ptr(), (float *)dv.data_ptr(), dcp,
                               ws.data_ptr(), B, V, H, Hi, W, D, P, scale, st.ptr(), flags, s);
        else
            rc = (code == DSDPA_BF16 ? dsdpa_bwd_bf16 : dsdpa_bwd_f16)(q.data_ptr(), k.data_ptr(), v.data_ptr(), cp, out.data_ptr(), lp,
                                                                       dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dcp,
                                                                       ws.data_ptr(), B, V, H, Hi, W, D, P, scale, st.ptr(), flags, s);
        check(rc, bound);
        return {dq, dk, dv, dcoords, Tensor()};
    }
};

namespace {

// Whether the call has to be an autograd.Function's: an input carries a forward-mode tangent, or a torch.func transform
// is active. The kernels read the values alone, and neither shows in requires_grad: from here the tangent would be
// dropped without a word. The Function has no rule for them and raises. Under torch.jit.trace the Function is recorded
// as a node; a call from here would be invisible, and its output a constant of the traced module. And under a dispatch
// mode, or with tensors that are a subclass's, the general route makes its buffers where these see them (fake tensors
// among them, which the kernels cannot read: refused there).
bool followed(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &coords)
{
    if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return true;
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return true;
    for (const Tensor *t : {&q, &k, &v, &coords})
        if (t->_fw_grad(/*level=*/0).defined() || t->unsafeGetTensorImpl()->is_python_dispatch()) return true;
    return false;
}

// The reference's preconditions (ops/triton.py:375,385-388) and this build's own.
bool acceptable(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &coords, const Call &c)
{
    const at::ScalarType t = q.scalar_type();
    if (t != at::kFloat && t != at::kBFloat16 && t != at::kHalf) return false;
    if (q.dim() != 5 || k.sizes() != q.sizes() || v.sizes() != q.sizes() || k.scalar_type() != t || v.scalar_type() != t) return false;
    const int64_t D = q.size(4), L = q.size(3);
    if (!(D == 16 || D == 32 || D == 64 || D == 128 || D == 256) || c.W < 1 || c.H < 1 || c.W > L || c.H > L || c.W * c.H != L) return false;
    if (q.size(0) < 1 || q.size(1) < 1 || q.size(2) < 1 || coords.dim() != 6 || coords.size(4) < 1) return false;
    if (q.size(0) > INT_MAX || q.size(1) > INT_MAX || q.size(2) > INT_MAX || L > INT_MAX) return false;
    if (!coords.is_contiguous() || coords.size(0) != q.size(0) || coords.size(1) != q.size(1) || coords.size(2) != L ||
        coords.size(3) != q.size(1) || coords.size(5) != 2 || coords.size(4) > INT_MAX)
        return false;
    return q.is_cuda() && k.device() == q.device() && v.device() == q.device() && coords.device() == q.device();
}

PyObject *apply(PyObject *bound, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != 7 && n != 8) Py_RETURN_NONE;
    for (int i = 0; i < 4; ++i)
        if (!THPVariable_Check(args[i])) Py_RETURN_NONE;
    // (a scale or size in a tensor may require a gradient or carry a tangent, too: the Function knows it for an input)
    for (Py_ssize_t i = 4; i < n; ++i)
        if (THPVariable_Check(args[i])) Py_RETURN_NONE;
    Tensor q = THPVariable_Unpack(args[0]), k = THPVariable_Unpack(args[1]), v = THPVariable_Unpack(args[2]),
           coords = THPVariable_Unpack(args[3]);
    if (followed(q, k, v, coords)) Py_RETURN_NONE;
    Call c;
    c.bound = bound;
    c.W = PyNumber_AsSsize_t(args[4], PyExc_OverflowError);
    c.H = PyErr_Occurred() ? 0 : PyNumber_AsSsize_t(args[5], PyExc_OverflowError);
    PyObject *scale = PyErr_Occurred() ? nullptr : PyNumber_Float(args[6]);
    const int cg = scale && n == 8 ? PyObject_IsTrue(args[7]) : 0;
    if (scale) {
        c.scale = PyFloat_AS_DOUBLE(scale);
        Py_DECREF(scale);
    }
    if (!scale || cg < 0) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    c.coords_grad = cg == 1;
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        if (acceptable(q, k, v, coords, c)) {
            Strides st;
            if (!readable_in_place(q, k, v, &st)) q = packed(q), k = packed(k), v = packed(v);
            if (coords.scalar_type() != at::kFloat) coords = coords.to(at::kFloat);
            coords = packed(coords, 8);                  // (read as pairs)
            const bool graph = at::GradMode::is_enabled() &&
                               (q.requires_grad() || k.requires_grad() || v.requires_grad() || coords.requires_grad());
            out = graph ? fused_deform_sdpa::apply(q, k, v, coords, c) : forward_pass(q, k, v, coords, c).first;
        }
    }
    if (!out.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef apply_method = {"apply", (PyCFunction)(void (*)(void))apply, METH_FASTCALL,
                            "one call of the operator; None when it has to take the general route"};

PyObject *bind(PyObject *, PyObject *args)
{
    PyObject *check, *globals;
    if (!PyArg_ParseTuple(args, "OO!", &check, &PyDict_Type, &globals)) return nullptr;
    Py_INCREF(args);                     // never given back, see check_of()
    return PyCFunction_New(&apply_method, args);
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "the operator for a module: bind(check, globals) -> apply"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dsdpa_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dsdpa_torch(void) { return PyModule_Create(&module); }
