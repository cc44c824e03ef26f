// causal_conv1d._native: the host path of the prefill, the pool / ring decode step and the backward, from torch tensors
// to the C ABI, without a Python statement per field.  Filled through ctypes the argument block of a prefill took
// 7 of the 18 us such a call needed on the host (CanonLayer, B 1, C 640, L 77: now 10.5 us, of which the kernel is 4).
//
// The functions come in two kinds.  launch_*: the arguments were checked by the caller; the output (a status code where
// the launch failed) is returned, or None where the tensors are not plain.  try_*: the public calls' own arguments; they
// check what the Python functions check and launch, or return None without having done anything when a call is not plain
// (gradients, another device than the current one, tensor subclasses, transforms, types that need a conversion, an
// argument that is wrong): the Python function then goes on as if it had not asked, and raises what there is to raise.
#include <Python.h>
#include <string.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include "canon_conv1d.h"

namespace {

using at::Tensor;

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return CANON_DTYPE_F32;
    case at::kBFloat16: return CANON_DTYPE_BF16;
    case at::kHalf: return CANON_DTYPE_F16;
    default: return -1;
    }
}

int mask_code(at::ScalarType t)
{
    switch (t) {
    case at::kBool:
    case at::kByte: return CANON_MASK_U8;
    case at::kInt: return CANON_MASK_I32;
    case at::kLong: return CANON_MASK_I64;
    case at::kFloat: return CANON_MASK_F32;
    case at::kBFloat16: return CANON_MASK_BF16;
    case at::kHalf: return CANON_MASK_F16;
    default: return -1;
    }
}

// The tensor of an argument: false when it is neither None nor a plain tensor (no subclass, no transform's wrapper).
bool plain(PyObject *o, const Tensor **t)
{
    *t = nullptr;
    if (o == Py_None) return true;
    if (!THPVariable_CheckExact(o)) return false;
    const Tensor &v = THPVariable_Unpack(o);
    if (at::isTensorSubclassLike(v)) return false;
    *t = &v;
    return true;
}

long small_int(PyObject *o) { return PyLong_AsLong(o); }

bool wants_grad(const Tensor *t) { return t && t->requires_grad(); }

// 0, 1, 2 as _RESIDUAL says; -1: something the Python function should look at
int residual_mode(PyObject *o)
{
    if (o == Py_False || o == Py_None) return CANON_RESIDUAL_NONE;
    if (o == Py_True) return CANON_RESIDUAL_MASKED;
    if (!PyUnicode_Check(o)) return -1;
    if (PyUnicode_CompareWithASCIIString(o, "masked") == 0) return CANON_RESIDUAL_MASKED;
    return PyUnicode_CompareWithASCIIString(o, "unmasked") == 0 ? CANON_RESIDUAL_UNMASKED : -1;
}

int activation_flag(PyObject *o)
{
    if (o == Py_None) return CANON_ACT_NONE;
    if (!PyUnicode_Check(o)) return -1;
    return PyUnicode_CompareWithASCIIString(o, "silu") == 0 || PyUnicode_CompareWithASCIIString(o, "swish") == 0 ? CANON_ACT_SILU : -1;
}

int round_mode(PyObject *o)
{
    if (!PyUnicode_Check(o)) return -1;
    if (PyUnicode_CompareWithASCIIString(o, "fused") == 0) return CANON_ROUND_FUSED;
    return PyUnicode_CompareWithASCIIString(o, "eager") == 0 ? CANON_ROUND_EAGER : -1;
}

// The current stream of the tensor's device, which has to be the current device (false without an exception: it is not).
bool stream_of(const Tensor &x, void **stream)
{
    const c10::DeviceIndex dev = (c10::DeviceIndex)x.get_device();
    if (c10::hip::current_device() != dev) return false;
    *stream = (void *)c10::hip::getCurrentHIPStream(dev).stream();
    return true;
}

template <typename F> int without_gil(F &&call)
{
    struct Released {
        PyThreadState *thread = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(thread); }   // (also when an allocation throws)
    } released;
    return call();
}

void *address(const Tensor *t) { return t ? t->data_ptr() : nullptr; }

canon_conv1d_fwd_params fwd_params(const Tensor &x, const Tensor &out, const Tensor &weight, const Tensor *bias, const Tensor *mask,
                                   const Tensor *init, const Tensor *fin, const Tensor *seq, int act, int res, int rnd)
{
    canon_conv1d_fwd_params p;
    memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.x_dtype = dtype_code(x.scalar_type());
    p.w_dtype = dtype_code(weight.scalar_type());
    p.width = (int32_t)weight.size(1);
    p.activation = act; p.residual_mode = res; p.round_mode = rnd;
    p.batch = x.size(0); p.channels = x.size(1); p.seqlen = x.size(2);
    p.x = x.data_ptr();
    p.x_stride_b = x.stride(0); p.x_stride_c = x.stride(1); p.x_stride_l = x.stride(2);
    p.out = out.data_ptr();
    p.out_stride_b = out.stride(0); p.out_stride_c = out.stride(1); p.out_stride_l = out.stride(2);
    p.weight = weight.data_ptr();
    p.w_stride_c = weight.stride(0); p.w_stride_k = weight.stride(1);
    p.bias = address(bias);
    if (mask) {
        p.mask = mask->data_ptr();
        p.mask_dtype = mask_code(mask->scalar_type());
        p.mask_stride_b = mask->stride(0); p.mask_stride_l = mask->stride(1);
    }
    if (init) {
        p.initial_state = init->data_ptr();
        p.init_stride_b = init->stride(0); p.init_stride_c = init->stride(1); p.init_stride_s = init->stride(2);
        p.initial_len = (int32_t)init->size(2);
    }
    if (fin) {
        p.final_state = fin->data_ptr();
        p.final_stride_b = fin->stride(0); p.final_stride_c = fin->stride(1); p.final_stride_s = fin->stride(2);
        p.final_len = (int32_t)fin->size(2);
    }
    if (seq) {
        p.seq_idx = (const int32_t *)seq->data_ptr();
        p.seq_stride_b = seq->stride(0); p.seq_stride_l = seq->stride(1);
    }
    return p;
}

// x (and out): [B, .., C], the token's channels in its last dimension
canon_conv1d_update_params update_params(const Tensor &x, int64_t x_stride_c, const Tensor &out, const Tensor &state,
                                         const Tensor &weight, const Tensor *bias, int act, int res, int rnd)
{
    canon_conv1d_update_params p;
    memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.x_dtype = dtype_code(x.scalar_type());
    p.w_dtype = dtype_code(weight.scalar_type());
    p.width = (int32_t)weight.size(1);
    p.activation = act; p.residual_mode = res; p.round_mode = rnd;
    p.state_len = (int32_t)state.size(2);
    p.batch = x.size(0); p.channels = x.size(-1);
    p.x = x.data_ptr(); p.x_stride_b = x.stride(0); p.x_stride_c = x_stride_c;
    p.out = out.data_ptr(); p.out_stride_b = p.channels; p.out_stride_c = 1;
    p.conv_state = state.data_ptr();
    p.state_stride_b = state.stride(0); p.state_stride_c = state.stride(1); p.state_stride_s = state.stride(2);
    p.weight = weight.data_ptr(); p.w_stride_c = weight.stride(0); p.w_stride_k = weight.stride(1);
    p.bias = address(bias);
    return p;
}

canon_conv1d_part part_of(const Tensor &x, const Tensor &out)
{
    canon_conv1d_part q;
    memset(&q, 0, sizeof(q));
    q.x = x.data_ptr();
    q.x_stride_b = x.stride(0); q.x_stride_c = x.stride(1); q.x_stride_l = x.stride(2);
    q.out = out.data_ptr();
    q.out_stride_b = out.stride(0); q.out_stride_c = out.stride(1); q.out_stride_l = out.stride(2);
    q.channels = x.size(1);
    return q;
}

// What _check_fwd_args accepts without a conversion, on the problem [B, C, L] of x's type and device.
bool fwd_args_ok(const Tensor &x, int64_t B, int64_t C, int64_t L, const Tensor *weight, const Tensor *bias, const Tensor *mask,
                 const Tensor *init, const Tensor *fin)
{
    if (dtype_code(x.scalar_type()) < 0 || !x.is_cuda() || !weight || B * C * L == 0) return false;
    const at::Device dev = x.device();
    if (weight->dim() != 2 || weight->size(0) != C || weight->size(1) < CANON_CONV1D_MIN_WIDTH ||
        weight->size(1) > CANON_CONV1D_MAX_WIDTH || dtype_code(weight->scalar_type()) < 0 || weight->device() != dev)
        return false;
    if (bias && (bias->dim() != 1 || bias->size(0) != C || bias->scalar_type() != weight->scalar_type() ||
                 !bias->is_contiguous() || bias->device() != dev))
        return false;
    if (mask && (mask->dim() != 2 || mask->size(0) != B || mask->size(1) != L || mask_code(mask->scalar_type()) < 0 ||
                 mask->device() != dev))
        return false;
    for (const Tensor *s : {init, fin})
        if (s && (s->dim() != 3 || s->size(0) != B || s->size(1) != C || s->scalar_type() != x.scalar_type() || s->device() != dev))
            return false;
    return true;
}

// The autograd node of a plain call (neither states nor anything a transform adds): forward and backward are one fused
// launch each, nothing but the inputs is saved, and the backward runs in the engine's thread without the interpreter.
// As a Python function, which the engine's thread has to take the interpreter's lock for, a training step that the host
// bounds took 87-95 us (B 16, C 640, L 511, y.detach() and torch.autograd.grad included), with this node 65-67.
int run_bwd(const Tensor &x, Tensor dout, const Tensor &weight, const Tensor *bias, const Tensor *mask, const Tensor &dweight,
            const Tensor *dbias, int act, int res, const Tensor *seq, const Tensor *init, const Tensor *dinit, const Tensor *dfin,
            void *stream, Tensor &dx);
int run_fwd(const Tensor &x, const Tensor &weight, const Tensor *bias, const Tensor *mask, const Tensor *seq, int act, int res, int rnd,
            void *stream, Tensor &out);

[[noreturn]] void refuse(int rc, const char *what)
{
    const std::string message = std::string(what) + ": " + canon_conv1d_last_error();
    if (rc == CANON_ERR_INVALID_ARGUMENT) C10_THROW_ERROR(ValueError, message);
    if (rc == CANON_ERR_UNSUPPORTED) C10_THROW_ERROR(NotImplementedError, message);
    C10_THROW_ERROR(Error, message);
}

// A gradient for a caller that asked for a graph of the backward (create_graph): it depends on `sources`, and a walk from it
// to one of them ends in an error.  (Without a node that says so, a loss made of such a gradient and of something else would
// lose the gradient's share without a word.  As _final in the Python nodes.)
void refuse_second_order(const Tensor &grad, std::initializer_list<Tensor> sources)
{
    torch::autograd::edge_list edges;
    for (const Tensor &t : sources)
        if (t.defined() && t.requires_grad()) edges.push_back(torch::autograd::impl::gradient_edge(t));
    if (!grad.defined() || edges.empty()) return;
    torch::autograd::set_history(grad, std::make_shared<torch::autograd::Error>(
        "causal_conv1d: the backward is a fused kernel without a derivative of its own: its gradients cannot be differentiated",
        std::move(edges)));
}

struct CanonConv : torch::autograd::Function<CanonConv> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &weight, const std::optional<Tensor> &bias,
                          const std::optional<Tensor> &mask, const std::optional<Tensor> &seq, int64_t act, int64_t res, int64_t rnd,
                          void *stream)
    {
        Tensor out;
        const int rc = run_fwd(x, weight, bias ? &*bias : nullptr, mask ? &*mask : nullptr, seq ? &*seq : nullptr, (int)act, (int)res,
                               (int)rnd, stream, out);
        if (rc != CANON_OK) refuse(rc, "causal_conv1d_fn");
        ctx->save_for_backward({x, weight, bias.value_or(Tensor()), mask.value_or(Tensor()), seq.value_or(Tensor())});
        ctx->saved_data["flags"] = act | res << 1;
        ctx->set_materialize_grads(false);
        return out;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, const torch::autograd::variable_list &grads)
    {
        const bool graph_wanted = c10::GradMode::is_enabled();   // (create_graph)
        const at::NoGradGuard no_grad;
        const torch::autograd::variable_list saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &weight = saved[1];
        const auto given = [&](int i) { return saved[i].defined() ? &saved[i] : nullptr; };
        const int64_t flags = ctx->saved_data["flags"].toInt();
        Tensor dout = grads[0].defined() ? grads[0] : at::zeros_like(x);
        if (dout.scalar_type() != x.scalar_type()) dout = dout.to(x.scalar_type());
        const c10::DeviceGuard device(x.device());
        const at::TensorOptions options = weight.options();
        Tensor dx, dweight = at::empty(weight.sizes(), options), dbias;
        if (given(2)) dbias = at::empty({weight.size(0)}, options);
        const int rc = run_bwd(x, std::move(dout), weight, given(2), given(3), dweight, given(2) ? &dbias : nullptr, (int)(flags & 1),
                               (int)(flags >> 1), given(4), nullptr, nullptr, nullptr,
                               (void *)c10::hip::getCurrentHIPStream((c10::DeviceIndex)x.get_device()).stream(), dx);
        if (rc != CANON_OK) refuse(rc, "causal_conv1d_fn backward");
        if (graph_wanted) {
            // (without an activation the backward is linear in each of these)
            const bool act = flags & 1;
            const Tensor none;
            refuse_second_order(dx, {grads[0], weight, act ? x : none, act ? saved[2] : none});
            refuse_second_order(dweight, {grads[0], x, act ? weight : none, act ? saved[2] : none});
            refuse_second_order(dbias, {grads[0], act ? x : none, act ? weight : none, act ? saved[2] : none});
        }
        return {dx, dweight, dbias, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// Whether the node above sees all there is to see: no functorch level, no tracer, no forward-mode tangent (the Python
// function's ways with those, errors included, are what callers know).
bool plain_autograd(std::initializer_list<const Tensor *> inputs)
{
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || torch::jit::tracer::isTracing())
        return false;
    for (const Tensor *t : inputs)
        if (t && t->_fw_grad(0).defined()) return false;
    return true;
}

std::optional<Tensor> optional_of(const Tensor *t) { return t ? std::optional<Tensor>(*t) : std::nullopt; }

// What _narrow_mask does: a wide integer mask of a large call is converted, for this call, to x's type, unless the
// channel-contiguous vector kernels take it (`kept` holds it until the launch is enqueued).
constexpr int64_t kNarrowMinElements = 1 << 24;
const Tensor *narrow(const Tensor *mask, const Tensor &x, int64_t numel, Tensor &kept)
{
    if (!mask || at::isFloatingType(mask->scalar_type()) || mask->element_size() <= x.element_size() || numel < kNarrowMinElements ||
        (x.stride(1) == 1 && x.stride(2) != 1 && x.size(1) * x.element_size() % 8 == 0))
        return mask;
    kept = mask->to(x.scalar_type());
    return &kept;
}

// (a dispatch mode sees the tensor operations of the Python path, not what happens here)
bool no_mode() { return !c10::impl::dispatch_mode_enabled(); }

#define CANON_NONE_UNLESS(cond) do { if (!(cond)) Py_RETURN_NONE; } while (0)

// try_fwd(x, weight, bias, seq_idx, initial_states, final_states, activation, attention_mask, residual, rounding)
//   -> output | status code | None.  final_states: the tensor to fill, or None.
PyObject *try_fwd(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 10 && no_mode());
    const Tensor *x, *weight, *bias, *seq, *init, *fin, *mask;
    CANON_NONE_UNLESS(plain(args[0], &x) && plain(args[1], &weight) && plain(args[2], &bias) && plain(args[3], &seq) &&
                      plain(args[4], &init) && plain(args[5], &fin) && plain(args[7], &mask) && x);
    const int act = activation_flag(args[6]), res = residual_mode(args[8]), rnd = round_mode(args[9]);
    CANON_NONE_UNLESS(act >= 0 && res >= 0 && rnd >= 0 && x->dim() == 3);
    const bool grad = c10::GradMode::is_enabled() && (wants_grad(x) || wants_grad(weight) || wants_grad(bias) || wants_grad(init));
    CANON_NONE_UNLESS(!grad || (!init && !fin && plain_autograd({x, weight, bias})));
    CANON_NONE_UNLESS(fwd_args_ok(*x, x->size(0), x->size(1), x->size(2), weight, bias, mask, init, fin));
    CANON_NONE_UNLESS(!seq || (!init && !fin && seq->dim() == 2 && seq->size(0) == x->size(0) && seq->size(1) == x->size(2) &&
                               seq->scalar_type() == at::kInt && seq->device() == x->device()));
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    Tensor narrowed;
    mask = narrow(mask, *x, x->numel(), narrowed);
    if (grad)
        return THPVariable_Wrap(CanonConv::apply(*x, *weight, optional_of(bias), optional_of(mask), optional_of(seq), (int64_t)act,
                                                 (int64_t)res, (int64_t)rnd, stream));
    Tensor out = at::empty_like(*x);
    const canon_conv1d_fwd_params p = fwd_params(*x, out, *weight, bias, mask, init, fin, seq, act, res, rnd);
    const int rc = without_gil([&] { return canon_conv1d_fwd(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// The block call of CanonLayer (inference), from the layer's own (batch, seqlen, dim) tensors, one or several parts, without
// a view of any of them: try_layer_block(x | (x, ..), taps, bias, history, slots, activation, mask, residual, rounding)
//   -> (output | outputs, new state of that many slots or None) | status code | None
PyObject *try_layer_block(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 9 && no_mode());
    PyObject *const one[1] = {args[0]};
    const bool tuple = PyTuple_CheckExact(args[0]);
    PyObject *const *items = tuple ? &PyTuple_GET_ITEM(args[0], 0) : one;
    const Py_ssize_t np = tuple ? PyTuple_GET_SIZE(args[0]) : 1;
    CANON_NONE_UNLESS(np >= 1 && np <= CANON_CONV1D_MAX_PARTS);
    const Tensor *xs[CANON_CONV1D_MAX_PARTS], *weight, *bias, *init, *mask;
    int64_t dim = 0;
    bool grad = false;
    for (Py_ssize_t i = 0; i < np; ++i) {
        // (dense: the output then has x's strides, whichever way round its last two dimensions are named)
        CANON_NONE_UNLESS(plain(items[i], &xs[i]) && xs[i] && xs[i]->dim() == 3 && xs[i]->is_non_overlapping_and_dense());
        CANON_NONE_UNLESS(xs[i]->scalar_type() == xs[0]->scalar_type() && xs[i]->device() == xs[0]->device() &&
                          xs[i]->size(0) == xs[0]->size(0) && xs[i]->size(1) == xs[0]->size(1));
        dim += xs[i]->size(2);
        grad |= xs[i]->requires_grad();
    }
    CANON_NONE_UNLESS(plain(args[1], &weight) && plain(args[2], &bias) && plain(args[3], &init) && plain(args[6], &mask));
    const int act = activation_flag(args[5]), res = residual_mode(args[7]), rnd = round_mode(args[8]);
    const long slots = PyLong_AsLong(args[4]);
    CANON_NONE_UNLESS(act >= 0 && res >= 0 && rnd >= 0 && slots >= 0);
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() || !(grad || wants_grad(weight) || wants_grad(bias) || wants_grad(init)));
    const Tensor &x0 = *xs[0];
    const int64_t B = x0.size(0), L = x0.size(1);
    CANON_NONE_UNLESS(fwd_args_ok(x0, B, dim, L, weight, bias, mask, init, nullptr));
    void *stream;
    CANON_NONE_UNLESS(stream_of(x0, &stream));
    const Tensor view = x0.transpose(1, 2);
    Tensor narrowed, state, outs[CANON_CONV1D_MAX_PARTS];
    mask = narrow(mask, view, B * dim * L, narrowed);
    if (slots > 0) state = at::empty({B, dim, slots}, x0.options());
    canon_conv1d_part parts[CANON_CONV1D_MAX_PARTS];
    for (Py_ssize_t i = 0; i < np; ++i) {
        outs[i] = at::empty_like(*xs[i]);
        parts[i] = part_of(*xs[i], outs[i]);
        std::swap(parts[i].x_stride_c, parts[i].x_stride_l);
        std::swap(parts[i].out_stride_c, parts[i].out_stride_l);
        parts[i].channels = xs[i]->size(2);
    }
    canon_conv1d_fwd_params p = fwd_params(view, outs[0], *weight, bias, mask, init, slots > 0 ? &state : nullptr, nullptr, act, res, rnd);
    p.channels = dim;
    if (np == 1) {
        p.out_stride_c = parts[0].out_stride_c;
        p.out_stride_l = parts[0].out_stride_l;
    } else {
        p.x = p.out = nullptr;
    }
    const int rc = without_gil([&] { return np == 1 ? canon_conv1d_fwd(&p, stream) : canon_conv1d_fwd_parts(&p, parts, (int32_t)np, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    PyObject *out;
    if (tuple) {
        out = PyTuple_New(np);
        if (!out) return nullptr;
        for (Py_ssize_t i = 0; i < np; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(outs[i])));
    } else {
        out = THPVariable_Wrap(std::move(outs[0]));
    }
    PyObject *result = PyTuple_New(2);
    if (!result) return nullptr;
    PyTuple_SET_ITEM(result, 0, out);
    if (slots > 0) {
        PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(std::move(state)));
    } else {
        Py_INCREF(Py_None);
        PyTuple_SET_ITEM(result, 1, Py_None);
    }
    return result;
    END_HANDLE_TH_ERRORS
}

// try_fwd_parts((x, ..), weight, bias, initial_states, final_states, activation, attention_mask, residual, rounding)
//   -> tuple of outputs | status code | None
PyObject *try_fwd_parts(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 9 && no_mode() && (PyTuple_CheckExact(args[0]) || PyList_CheckExact(args[0])));
    const Py_ssize_t np = PySequence_Fast_GET_SIZE(args[0]);
    CANON_NONE_UNLESS(np >= 1 && np <= CANON_CONV1D_MAX_PARTS);
    const Tensor *xs[CANON_CONV1D_MAX_PARTS], *weight, *bias, *init, *fin, *mask;
    int64_t dim = 0;
    bool grad = false;
    for (Py_ssize_t i = 0; i < np; ++i) {
        CANON_NONE_UNLESS(plain(PySequence_Fast_GET_ITEM(args[0], i), &xs[i]) && xs[i] && xs[i]->dim() == 3);
        CANON_NONE_UNLESS(xs[i]->scalar_type() == xs[0]->scalar_type() && xs[i]->device() == xs[0]->device() &&
                          xs[i]->size(0) == xs[0]->size(0) && xs[i]->size(2) == xs[0]->size(2));
        dim += xs[i]->size(1);
        grad |= xs[i]->requires_grad();
    }
    CANON_NONE_UNLESS(plain(args[1], &weight) && plain(args[2], &bias) && plain(args[3], &init) && plain(args[4], &fin) &&
                      plain(args[6], &mask));
    const int act = activation_flag(args[5]), res = residual_mode(args[7]), rnd = round_mode(args[8]);
    CANON_NONE_UNLESS(act >= 0 && res >= 0 && rnd >= 0);
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() || !(grad || wants_grad(weight) || wants_grad(bias) || wants_grad(init)));
    CANON_NONE_UNLESS(fwd_args_ok(*xs[0], xs[0]->size(0), dim, xs[0]->size(2), weight, bias, mask, init, fin));
    void *stream;
    CANON_NONE_UNLESS(stream_of(*xs[0], &stream));
    Tensor outs[CANON_CONV1D_MAX_PARTS];
    canon_conv1d_part parts[CANON_CONV1D_MAX_PARTS];
    for (Py_ssize_t i = 0; i < np; ++i) {
        outs[i] = at::empty_like(*xs[i]);
        parts[i] = part_of(*xs[i], outs[i]);
    }
    Tensor narrowed;
    mask = narrow(mask, *xs[0], xs[0]->size(0) * dim * xs[0]->size(2), narrowed);
    canon_conv1d_fwd_params p = fwd_params(*xs[0], outs[0], *weight, bias, mask, init, fin, nullptr, act, res, rnd);
    p.channels = dim;
    p.x = p.out = nullptr;
    const int rc = without_gil([&] { return canon_conv1d_fwd_parts(&p, parts, (int32_t)np, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    PyObject *result = PyTuple_New(np);
    if (!result) return nullptr;
    for (Py_ssize_t i = 0; i < np; ++i) PyTuple_SET_ITEM(result, i, THPVariable_Wrap(std::move(outs[i])));
    return result;
    END_HANDLE_TH_ERRORS
}

// The plain decode step of a signature that has been through every check before (see causal_conv1d_update): `known` maps
// signatures to argument blocks in which only the addresses are missing (with the signature a tuple of Python's sizes and
// strides and the launch through ctypes, B 256, C 3456: 10.4 us a call, here 6.5).  try_known_update(x, conv_state, weight, bias,
// activation, token_mask, residual, rounding, known) -> output | status code | the signature, which the table does not hold
// (nothing was done) | None
PyObject *try_known_update(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 9 && no_mode());
    const Tensor *x, *state, *weight, *bias, *mask;
    CANON_NONE_UNLESS(plain(args[0], &x) && plain(args[1], &state) && plain(args[2], &weight) && plain(args[3], &bias) &&
                      plain(args[5], &mask) && x && state && weight && PyDict_CheckExact(args[8]));
    const int act = activation_flag(args[4]), res = residual_mode(args[6]), rnd = round_mode(args[7]);
    CANON_NONE_UNLESS(act >= 0 && res >= 0 && rnd >= 0 && x->dim() == 2 && state->dim() == 3 && weight->dim() == 2 && x->is_cuda());
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() ||
                      !(wants_grad(x) || wants_grad(state) || wants_grad(weight) || wants_grad(bias) || wants_grad(mask)));
    CANON_NONE_UNLESS((!bias || bias->dim() == 1) && (!mask || mask->dim() == 1));
    // two entries, then a type and a size and stride per dimension: x 2, state 3, weight 2, bias 1, mask 1 (checked above)
    int64_t key[2 + 5 + 2 * (2 + 3 + 2 + 1 + 1)] = {act | res << 4 | rnd << 8, x->get_device()};
    int at = 2;
    for (const Tensor *t : {x, state, weight, bias, mask}) {
        if (!t) {
            key[at++] = -1;
            continue;
        }
        CANON_NONE_UNLESS(t->device() == x->device());
        key[at++] = (int64_t)t->scalar_type() | t->dim() << 8;
        for (int64_t i = 0; i < t->dim(); ++i) {
            key[at++] = t->size(i);
            key[at++] = t->stride(i);
        }
    }
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    PyObject *signature = PyBytes_FromStringAndSize((const char *)key, at * sizeof(key[0]));
    if (!signature) return nullptr;
    PyObject *block = PyDict_GetItemWithError(args[8], signature);   // (borrowed)
    if (!block) {
        if (!PyErr_Occurred()) return signature;
        Py_DECREF(signature);
        return nullptr;
    }
    Py_DECREF(signature);
    CANON_NONE_UNLESS(PyBytes_CheckExact(block) && PyBytes_GET_SIZE(block) == sizeof(canon_conv1d_update_params));
    canon_conv1d_update_params p;
    memcpy(&p, PyBytes_AS_STRING(block), sizeof(p));
    Tensor out = at::empty(x->sizes(), x->options());
    p.x = x->data_ptr();
    p.out = out.data_ptr();
    p.conv_state = state->data_ptr();
    p.weight = weight->data_ptr();
    p.bias = address(bias);
    p.token_mask = address(mask);
    const int rc = without_gil([&] { return canon_conv1d_update(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// try_update_modes(x, conv_state, weight, bias, activation, cache_seqlens, conv_state_indices, token_mask, residual,
//   rounding) -> output | status code | None: the decode step over a ring buffer or a state pool, x (batch, dim)
PyObject *try_update_modes(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 10 && no_mode());
    const Tensor *x, *state, *weight, *bias, *seqlens, *indices, *mask;
    CANON_NONE_UNLESS(plain(args[0], &x) && plain(args[1], &state) && plain(args[2], &weight) && plain(args[3], &bias) &&
                      plain(args[5], &seqlens) && plain(args[6], &indices) && plain(args[7], &mask) && x && state);
    const int act = activation_flag(args[4]), res = residual_mode(args[8]), rnd = round_mode(args[9]);
    CANON_NONE_UNLESS(act >= 0 && res >= 0 && rnd >= 0 && x->dim() == 2 && state->dim() == 3);
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() ||
                      !(wants_grad(x) || wants_grad(state) || wants_grad(weight) || wants_grad(bias) || wants_grad(mask)));
    const int64_t B = x->size(0), C = x->size(1);
    CANON_NONE_UNLESS(fwd_args_ok(*x, B, C, 1, weight, bias, nullptr, nullptr, nullptr));
    CANON_NONE_UNLESS(state->size(1) == C && (indices || state->size(0) == B) && state->scalar_type() == x->scalar_type() &&
                      state->device() == x->device() && state->size(2) >= weight->size(1) - 1);
    for (const Tensor *t : {seqlens, indices})
        CANON_NONE_UNLESS(!t || (t->dim() == 1 && t->size(0) == B && t->scalar_type() == at::kInt && t->device() == x->device() &&
                                 t->is_contiguous()));
    CANON_NONE_UNLESS(!mask || (mask->dim() == 1 && mask->size(0) == B && mask_code(mask->scalar_type()) >= 0 &&
                                mask->device() == x->device()));
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    Tensor out = at::empty({B, C}, x->options());
    canon_conv1d_update_params p = update_params(*x, x->stride(1), out, *state, *weight, bias, act, res, rnd);
    if (mask) {
        p.token_mask = mask->data_ptr();
        p.mask_dtype = mask_code(mask->scalar_type());
        p.mask_stride_b = mask->stride(0);
    }
    p.cache_seqlens = (const int32_t *)address(seqlens);
    if (indices) {
        p.conv_state_indices = (const int32_t *)indices->data_ptr();
        p.state_rows = (int32_t)state->size(0);
    }
    const int rc = without_gil([&] { return canon_conv1d_update_zero_skipped(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// try_decode_step(x, conv_state, weight, bias, attention_mask, activation, rounding) -> output | status code | None: the
// single-token call of CanonLayer, x (batch, 1, dim), the whole-history mask whose last column scales the token, the
// residual the unmasked token
PyObject *try_decode_step(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 7 && no_mode());
    const Tensor *x, *state, *weight, *bias, *mask;
    CANON_NONE_UNLESS(plain(args[0], &x) && plain(args[1], &state) && plain(args[2], &weight) && plain(args[3], &bias) &&
                      plain(args[4], &mask) && x && state);
    const int act = activation_flag(args[5]), rnd = round_mode(args[6]);
    CANON_NONE_UNLESS(act >= 0 && rnd >= 0 && x->dim() == 3 && x->size(1) == 1 && state->dim() == 3);
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() || !(wants_grad(x) || wants_grad(state) || wants_grad(weight) || wants_grad(bias)));
    const int64_t B = x->size(0), C = x->size(2);
    CANON_NONE_UNLESS(fwd_args_ok(*x, B, C, 1, weight, bias, nullptr, nullptr, state) && state->size(2) >= weight->size(1) - 1);
    CANON_NONE_UNLESS(!mask || (mask->dim() == 2 && mask->size(0) == B && mask->size(1) > 0 &&
                                mask_code(mask->scalar_type()) >= 0 && mask->device() == x->device()));
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    Tensor out = at::empty({B, 1, C}, x->options());
    canon_conv1d_update_params p = update_params(*x, x->stride(2), out, *state, *weight, bias, act, CANON_RESIDUAL_UNMASKED, rnd);
    if (mask) {
        p.token_mask = (const char *)mask->data_ptr() + (mask->size(1) - 1) * mask->stride(1) * (int64_t)mask->element_size();
        p.mask_dtype = mask_code(mask->scalar_type());
        p.mask_stride_b = mask->stride(0);
    }
    const int rc = without_gil([&] { return canon_conv1d_update(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// launch_fwd(x, weight, bias, mask, initial_states, final_states, act, res, rnd, seq_idx) -> output | status code, of
// checked arguments; None when x's device is not the current one or a tensor is not plain
PyObject *launch_fwd(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 10 && no_mode());
    const Tensor *x, *weight, *bias, *mask, *init, *fin, *seq;
    CANON_NONE_UNLESS(plain(args[0], &x) && plain(args[1], &weight) && plain(args[2], &bias) && plain(args[3], &mask) &&
                      plain(args[4], &init) && plain(args[5], &fin) && plain(args[9], &seq) && x && weight);
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    Tensor out = at::empty_like(*x);
    const canon_conv1d_fwd_params p = fwd_params(*x, out, *weight, bias, mask, init, fin, seq, (int)small_int(args[6]),
                                                 (int)small_int(args[7]), (int)small_int(args[8]));
    const int rc = without_gil([&] { return canon_conv1d_fwd(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// launch_bwd(x, dout, weight, bias, mask, dweight, dbias, act, res, seq_idx, initial_states, dinit, dfinal)
//   -> dx | status code, of checked arguments (dout and dfinal of x's type); None when x's device is not the current one
//   or a tensor is not plain
PyObject *launch_bwd(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    CANON_NONE_UNLESS(n == 13 && no_mode());
    const Tensor *xp, *gp, *wp, *dwp, *bias, *mask, *dbias, *seq, *init, *dinit, *dfin;
    CANON_NONE_UNLESS(plain(args[0], &xp) && plain(args[1], &gp) && plain(args[2], &wp) && plain(args[3], &bias) &&
                      plain(args[4], &mask) && plain(args[5], &dwp) && plain(args[6], &dbias) && plain(args[9], &seq) &&
                      plain(args[10], &init) && plain(args[11], &dinit) && plain(args[12], &dfin) && xp && gp && wp && dwp);
    const long act = small_int(args[7]), res = small_int(args[8]);
    void *stream;
    CANON_NONE_UNLESS(stream_of(*xp, &stream));
    Tensor dx;
    const int rc = without_gil([&] {
        return run_bwd(*xp, *gp, *wp, bias, mask, *dwp, dbias, (int)act, (int)res, seq, init, dinit, dfin, stream, dx);
    });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(dx));
    END_HANDLE_TH_ERRORS
}

int run_fwd(const Tensor &x, const Tensor &weight, const Tensor *bias, const Tensor *mask, const Tensor *seq, int act, int res, int rnd,
            void *stream, Tensor &out)
{
    out = at::empty_like(x);
    const canon_conv1d_fwd_params p = fwd_params(x, out, weight, bias, mask, nullptr, nullptr, seq, act, res, rnd);
    return without_gil([&] { return canon_conv1d_fwd(&p, stream); });
}

// The backward launch of checked arguments (dout and dfin of x's type) into dweight / dbias and a dx in x's layout, with a
// scratch of this call alone.  Callable without the interpreter's lock.
int run_bwd(const Tensor &x, Tensor dout, const Tensor &weight, const Tensor *bias, const Tensor *mask, const Tensor &dweight,
            const Tensor *dbias, int act, int res, const Tensor *seq, const Tensor *init, const Tensor *dinit, const Tensor *dfin,
            void *stream, Tensor &dx)
{
    dx = at::empty_like(x);
    if (dout.strides() != x.strides()) {
        // x's own layout keeps the vector kernels (empty_like: x's strides where x is dense)
        Tensor copy = at::empty_like(x);
        copy.copy_(dout);
        dout = std::move(copy);
    }
    canon_conv1d_bwd_params p;
    memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.x_dtype = dtype_code(x.scalar_type());
    p.w_dtype = dtype_code(weight.scalar_type());
    p.grad_dtype = dtype_code(dweight.scalar_type());
    p.width = (int32_t)weight.size(1);
    p.activation = act; p.residual_mode = res;
    p.batch = x.size(0); p.channels = x.size(1); p.seqlen = x.size(2);
    p.x = x.data_ptr();
    p.x_stride_b = x.stride(0); p.x_stride_c = x.stride(1); p.x_stride_l = x.stride(2);
    p.dout = dout.data_ptr();
    p.dout_stride_b = dout.stride(0); p.dout_stride_c = dout.stride(1); p.dout_stride_l = dout.stride(2);
    p.dx = dx.data_ptr();
    p.dx_stride_b = dx.stride(0); p.dx_stride_c = dx.stride(1); p.dx_stride_l = dx.stride(2);
    p.weight = weight.data_ptr();
    p.w_stride_c = weight.stride(0); p.w_stride_k = weight.stride(1);
    p.bias = address(bias);
    if (mask) {
        p.mask = mask->data_ptr();
        p.mask_dtype = mask_code(mask->scalar_type());
        p.mask_stride_b = mask->stride(0); p.mask_stride_l = mask->stride(1);
    }
    if (seq) {
        p.seq_idx = (const int32_t *)seq->data_ptr();
        p.seq_stride_b = seq->stride(0); p.seq_stride_l = seq->stride(1);
    }
    if (init) {
        p.initial_state = init->data_ptr();
        p.init_stride_b = init->stride(0); p.init_stride_c = init->stride(1); p.init_stride_s = init->stride(2);
        p.initial_len = (int32_t)init->size(2);
        if (dinit) {
            p.dinitial_state = dinit->data_ptr();
            p.dinit_stride_b = dinit->stride(0); p.dinit_stride_c = dinit->stride(1); p.dinit_stride_s = dinit->stride(2);
        }
    }
    if (dfin) {
        p.dfinal_state = dfin->data_ptr();
        p.dfinal_stride_b = dfin->stride(0); p.dfinal_stride_c = dfin->stride(1); p.dfinal_stride_s = dfin->stride(2);
        p.final_len = (int32_t)dfin->size(2);
    }
    p.dweight = dweight.data_ptr();
    p.dbias = address(dbias);
    const int64_t bytes = canon_conv1d_bwd_workspace_bytes(&p);
    if (bytes < 0) return CANON_ERR_INVALID_ARGUMENT;
    Tensor workspace = at::empty({bytes > 16 ? bytes : 16}, x.options().dtype(at::kByte));
    p.workspace = workspace.data_ptr();
    p.workspace_bytes = workspace.numel();
    return canon_conv1d_bwd(&p, stream);
}

#define CANON_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CANON_METHOD(try_fwd), CANON_METHOD(try_fwd_parts), CANON_METHOD(try_layer_block), CANON_METHOD(try_known_update),
                         CANON_METHOD(try_update_modes), CANON_METHOD(try_decode_step), CANON_METHOD(launch_fwd), CANON_METHOD(launch_bwd),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native()
{
    // (torch's C++ interface is another one in every release: the loader compares this before it calls anything)
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
