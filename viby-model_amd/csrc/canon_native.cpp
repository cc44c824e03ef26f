// causal_conv1d._native: the host path of the prefill, the pool / ring decode step and the backward, from torch tensors
// to the C ABI, without a Python statement per field.  Filled through ctypes the argument block of a prefill took
// 7 of the 18 us such a call needed on the host (CanonLayer, B 1, C 640, L 77: now 12 us, of which the kernel is 4).
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
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "canon_conv1d.h"

namespace {

using at::Tensor;

PyObject *g_raw_stream = nullptr;   // torch._C._cuda_getCurrentRawStream
PyObject *g_get_device = nullptr;   // torch._C._cuda_getDevice

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
    const int dev = x.get_device();
    PyObject *current = PyObject_CallNoArgs(g_get_device);
    if (!current) throw python_error();
    const long now = PyLong_AsLong(current);
    Py_DECREF(current);
    if (now != dev) return false;
    PyObject *index = PyLong_FromLong(dev);
    PyObject *raw = PyObject_CallOneArg(g_raw_stream, index);
    Py_DECREF(index);
    if (!raw) throw python_error();
    *stream = PyLong_AsVoidPtr(raw);
    Py_DECREF(raw);
    return true;
}

template <typename F> int without_gil(F &&call)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call();
    Py_END_ALLOW_THREADS
    return rc;
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
    CANON_NONE_UNLESS(!c10::GradMode::is_enabled() || !(wants_grad(x) || wants_grad(weight) || wants_grad(bias) || wants_grad(init)));
    CANON_NONE_UNLESS(fwd_args_ok(*x, x->size(0), x->size(1), x->size(2), weight, bias, mask, init, fin));
    CANON_NONE_UNLESS(!seq || (!init && !fin && seq->dim() == 2 && seq->size(0) == x->size(0) && seq->size(1) == x->size(2) &&
                               seq->scalar_type() == at::kInt && seq->device() == x->device()));
    void *stream;
    CANON_NONE_UNLESS(stream_of(*x, &stream));
    Tensor out = at::empty_like(*x), narrowed;
    mask = narrow(mask, *x, x->numel(), narrowed);
    const canon_conv1d_fwd_params p = fwd_params(*x, out, *weight, bias, mask, init, fin, seq, act, res, rnd);
    const int rc = without_gil([&] { return canon_conv1d_fwd(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
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
    const Tensor &x = *xp, &weight = *wp, &dweight = *dwp;
    void *stream;
    CANON_NONE_UNLESS(stream_of(x, &stream));
    Tensor dx = at::empty_like(x);
    Tensor dout = *gp;
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
    p.activation = (int32_t)small_int(args[7]); p.residual_mode = (int32_t)small_int(args[8]);
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
    if (bytes < 0) return PyLong_FromLong(CANON_ERR_INVALID_ARGUMENT);
    Tensor workspace = at::empty({bytes > 16 ? bytes : 16}, x.options().dtype(at::kByte));
    p.workspace = workspace.data_ptr();
    p.workspace_bytes = workspace.numel();
    const int rc = without_gil([&] { return canon_conv1d_bwd(&p, stream); });
    if (rc != CANON_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(dx));
    END_HANDLE_TH_ERRORS
}

#define CANON_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CANON_METHOD(try_fwd), CANON_METHOD(try_fwd_parts), CANON_METHOD(try_update_modes), CANON_METHOD(try_decode_step),
                         CANON_METHOD(launch_fwd), CANON_METHOD(launch_bwd), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native()
{
    PyObject *torch_c = PyImport_ImportModule("torch._C");
    if (!torch_c) return nullptr;
    g_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
    g_get_device = PyObject_GetAttrString(torch_c, "_cuda_getDevice");
    Py_DECREF(torch_c);
    if (!g_raw_stream || !g_get_device) return nullptr;
    // (torch's C++ interface is another one in every release: the loader compares this before it calls anything)
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
