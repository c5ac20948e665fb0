// Python calls -> C ABI, natively: the extension module behind binarybrain_amd/ops.py.
//
// A small layer's pass is bound by what the host does per call, not by the device: a launch costs 2.6 us of host time here, while a call through
// ctypes, with torch.empty, torch.cuda.current_stream and the checks in Python, cost 9 (one launch) to 19 us (three launches) — 142 us for the
// eight calls of a classifier step whose kernels take 75 us.  Here arguments are read from the vector call without a parser, outputs come from
// at::empty, the stream from torch's current stream, hints are set by the function that makes the call, and every tensor argument is
// checked (device, contiguous) as it is converted.  The entry points of include/bbhip.h that need nothing else are exported as they are, by a
// template that derives the conversion from the signature.
//
// The interpreter lock is released around each entry, as ctypes does.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <stdexcept>
#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/bbhip.h"

namespace {

PyObject *g_error = nullptr;                    // BbhipError of capi.py (set_error_type)

struct Failed : std::runtime_error { using std::runtime_error::runtime_error; };
struct PythonError {};                          // the interpreter's error is set

using T = at::Tensor const &;

// ---- arguments -----------------------------------------------------------------------------------------------------------------
at::Tensor const &tensor_arg(PyObject *o)
{
    if (!THPVariable_Check(o)) { PyErr_Format(PyExc_TypeError, "expected a torch tensor, got %s", Py_TYPE(o)->tp_name); throw PythonError(); }
    at::Tensor const &t = THPVariable_Unpack(o);
    if (!t.is_cuda())       { throw Failed("bbhip ops need device tensors"); }
    if (!t.is_contiguous()) { throw Failed("bbhip ops need contiguous tensors"); }
    return t;
}

struct OptTensor { at::Tensor const *t; explicit operator bool() const { return t != nullptr; } at::Tensor const &operator*() const { return *t; } };
struct Clamp     { bool on; float lo, hi; };    // None or (lo, hi)
struct Stream    { void *p; };

template <class A> struct FromPy;
template <> struct FromPy<T>         { static T get(PyObject *o) { return tensor_arg(o); } };
template <> struct FromPy<OptTensor> { static OptTensor get(PyObject *o) { return OptTensor{o == Py_None ? nullptr : &tensor_arg(o)}; } };
template <> struct FromPy<int> {
    static int get(PyObject *o)
    {
        long const v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred()) { throw PythonError(); }
        if (v < -2147483648L || v > 4294967295L) { PyErr_SetString(PyExc_OverflowError, "integer argument does not fit 32 bits"); throw PythonError(); }
        return (int)v;
    }
};
template <> struct FromPy<unsigned> { static unsigned get(PyObject *o) { return (unsigned)FromPy<int>::get(o); } };
template <> struct FromPy<bool> {
    static bool get(PyObject *o)
    {
        int const v = (o == Py_True) ? 1 : (o == Py_False) ? 0 : PyObject_IsTrue(o);
        if (v < 0) { throw PythonError(); }
        return v != 0;
    }
};
template <> struct FromPy<double> {
    static double get(PyObject *o)
    {
        double const v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) { throw PythonError(); }
        return v;
    }
};
template <> struct FromPy<float> { static float get(PyObject *o) { return (float)FromPy<double>::get(o); } };
template <> struct FromPy<Clamp> {
    static Clamp get(PyObject *o)
    {
        if (o == Py_None) { return Clamp{false, 0.0f, 0.0f}; }
        PyObject *lo = PySequence_GetItem(o, 0), *hi = lo ? PySequence_GetItem(o, 1) : nullptr;
        if (!hi) { Py_XDECREF(lo); throw PythonError(); }
        double const l = PyFloat_AsDouble(lo), h = PyFloat_AsDouble(hi);
        Py_DECREF(lo); Py_DECREF(hi);
        if (PyErr_Occurred()) { throw PythonError(); }
        return Clamp{true, (float)l, (float)h};
    }
};
// a device buffer of a plain entry point: a tensor or None.  A buffer that the entry may write to is asked for as such: torch then gives a tensor
// that shares its storage with a lazy clone storage of its own.
template <class E> struct FromPy<E *> {
    static E *get(PyObject *o)
    {
        if (o == Py_None) { return nullptr; }
        at::Tensor const &t = tensor_arg(o);
        if constexpr (std::is_const_v<E>) { return static_cast<E *>(t.const_data_ptr()); }
        else                              { return static_cast<E *>(t.mutable_data_ptr()); }
    }
};

// ---- results -------------------------------------------------------------------------------------------------------------------
PyObject *to_py(double v) { return PyFloat_FromDouble(v); }
PyObject *to_py(at::Tensor const &t) { if (!t.defined()) { Py_RETURN_NONE; } return THPVariable_Wrap(t); }
template <class... A, size_t... I>
PyObject *tuple_to_py(std::tuple<A...> const &v, std::index_sequence<I...>)
{
    PyObject *out = PyTuple_New(sizeof...(A));
    if (!out) { throw PythonError(); }
    bool ok = true;
    (void)std::initializer_list<int>{(PyTuple_SET_ITEM(out, I, to_py(std::get<I>(v))), ok = ok && PyTuple_GET_ITEM(out, I) != nullptr, 0)...};
    if (!ok) { Py_DECREF(out); throw PythonError(); }
    return out;
}
template <class... A> PyObject *to_py(std::tuple<A...> const &v) { return tuple_to_py(v, std::index_sequence_for<A...>()); }

void *current_stream(void) { return at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

void clear_hints(void)
{
    bbhip_HintInputNodeSize(0); bbhip_HintPackedInput(nullptr, 0, 0, 0); bbhip_HintPackedOutput(nullptr, 0, 0);
    bbhip_HintTableGradientOverwrite(0); bbhip_HintPreparedTables(nullptr, 0, 0); bbhip_HintZeroOutputPadding(0);
}

// One entry point with the interpreter lock released; a failure becomes a BbhipError with the library's message.
template <class... P, class... A>
void call(int (*entry)(P...), A... args)
{
    PyThreadState *const state = PyEval_SaveThread();
    int const rc = entry(args...);
    PyEval_RestoreThread(state);
    if (rc != 0) { throw Failed(bbhip_GetLastErrorString()); }
}

// ---- the vector-call wrapper of a function ---------------------------------------------------------------------------------------
template <class F> struct Caller;
template <class R, class... A> struct Caller<R (*)(A...)> {
    static constexpr size_t kArgs = sizeof...(A);
    template <size_t... I> static PyObject *go(R (*f)(A...), PyObject *const *args, std::index_sequence<I...>)
    {
        if constexpr (std::is_void_v<R>) { f(FromPy<A>::get(args[I])...); Py_RETURN_NONE; }
        else { return to_py(f(FromPy<A>::get(args[I])...)); }
    }
    static PyObject *run(R (*f)(A...), PyObject *const *args) { return go(f, args, std::index_sequence_for<A...>()); }
};
// an entry point of the C ABI: its last parameter is the stream
template <class F> struct EntryCaller;
template <class... P> struct EntryCaller<int (*)(P...)> {
    static constexpr size_t kArgs = sizeof...(P) - 1;
    template <size_t I> using Param = std::tuple_element_t<I, std::tuple<P...>>;
    static_assert(std::is_same_v<Param<kArgs>, void *>, "the stream comes last");
    template <size_t... I> static PyObject *go(int (*f)(P...), PyObject *const *args, std::index_sequence<I...>)
    {
        std::tuple<Param<I>...> v{FromPy<Param<I>>::get(args[I])...};
        call(f, std::get<I>(v)..., current_stream());
        Py_RETURN_NONE;
    }
    static PyObject *run(int (*f)(P...), PyObject *const *args) { return go(f, args, std::make_index_sequence<kArgs>()); }
};

template <template <class> class C, auto F>
PyObject *wrapped(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    using W = C<decltype(F)>;
    if ((size_t)n != W::kArgs) { PyErr_Format(PyExc_TypeError, "expected %zu arguments, got %zd", W::kArgs, n); return nullptr; }
    try { return W::run(F, args); }
    catch (PythonError const &) {}
    catch (Failed const &e) { PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, e.what()); }
    catch (std::exception const &e) { PyErr_SetString(PyExc_RuntimeError, e.what()); }
    clear_hints();              // none is left behind for another call
    return nullptr;
}

// ---- buffers -------------------------------------------------------------------------------------------------------------------
// (what at::empty comes to for device tensors, without the dispatcher's passes.  Every output has storage of its own, 0.6 us of host time each: one that a
// program keeps must not keep the others of its call, be saved with them, or grow into them.)
at::Tensor new_tensor(T like, at::IntArrayRef sizes, at::ScalarType type) { return at::Tensor(at::detail::empty_cuda(sizes, type, like.device(), std::nullopt)); }
at::Tensor rows_f32(T like, int64_t rows, int64_t stride) { return new_tensor(like, {rows, stride}, at::kFloat); }
at::Tensor rows_i32(T like, int64_t rows, int64_t words)  { return new_tensor(like, {rows, words}, at::kInt); }
at::Tensor zeros_i32(T like, int64_t rows, int64_t words) { return at::zeros({rows, words}, like.options().dtype(at::kInt)); }
at::Tensor line_f32(T like, int64_t n) { return new_tensor(like, {n}, at::kFloat); }

template <class E> E *data(T t) { return static_cast<E *>(t.data_ptr()); }
template <class E> E *data(OptTensor t) { return t ? static_cast<E *>((*t).data_ptr()) : nullptr; }

int rows_of(T t)   { return (int)t.size(0); }
int stride_of(T t) { return (int)t.size(1); }

// packed output rows: the caller's, or new ones whose padding the next call zeroes (the library is told, no fill launch)
at::Tensor packed_output(OptTensor out, T like, int64_t rows, int64_t words)
{
    if (out) { return *out; }
    bbhip_HintZeroOutputPadding(1);
    return rows_i32(like, rows, words);
}

void require(bool ok, char const *what) { if (!ok) { throw Failed(what); } }

// ---- hints of the next LUT call --------------------------------------------------------------------------------------------------
void hint_input(T x, OptTensor packed, bool holds, bool forward)
{
    if (packed) {
        require((*packed).scalar_type() == at::kInt && (*packed).size(0) == x.size(0), "packed: int32 rows, one per row of x");
        bbhip_HintPackedInput(data<int>(packed), rows_of(x), stride_of(*packed), holds);
    }
    else if (forward) { bbhip_HintInputNodeSize(rows_of(x)); }      // the forward signatures do not carry the row count of x
}

void hint_tables(OptTensor tables, bool holds)
{
    if (!tables) { return; }
    require((*tables).scalar_type() == at::kFloat, "tables: float32");
    bbhip_HintPreparedTables(data<float>(tables), (size_t)(*tables).numel() * 4, holds);
}

void hint_output(OptTensor packed_out, int rows)
{
    if (!packed_out) { return; }
    require((*packed_out).scalar_type() == at::kInt && (*packed_out).size(0) == rows, "packed_out: int32 rows, one per output node");
    bbhip_HintPackedOutput(data<int>(packed_out), rows, stride_of(*packed_out));
}

// ---- LUT layers ------------------------------------------------------------------------------------------------------------------
// `hints`: false leaves out every bbhip_Hint* (what a caller of the plain signatures gets)
at::Tensor stochastic_lut_forward(int n, T x, T idx, T W, int frames, bool input_binary, bool lut_binarize, float bias, OptTensor out, Clamp clamp,
                                  OptTensor packed, bool holds, bool hints)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = out ? *out : rows_f32(x, O, S);
    if (hints) { hint_input(x, packed, holds, true); }
    if (clamp.on) {
        call(bbhip_fp32_StochasticLut_ForwardClampW, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float>(W), O, frames, S,
             (int)input_binary, (int)lut_binarize, bias, clamp.lo, clamp.hi, current_stream());
    }
    else {
        call(bbhip_fp32_StochasticLut_Forward, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float const>(W), O, frames, S,
             (int)input_binary, (int)lut_binarize, bias, current_stream());
    }
    return y;
}

// frames per dx_tmp pass, as the reference sizes its scratch (include/bb/StochasticLutN.h:584-587)
int64_t tmp_frames(int64_t nodes, int64_t n, int64_t frames, int64_t max_bytes)
{
    int64_t t = max_bytes / (4 * nodes * n);
    t = ((t < 32 ? 32 : t) + 31) & ~(int64_t)31;
    return t < frames ? t : frames;
}

struct DxTmp { at::Tensor t; float *p = nullptr; int frames = 0, stride = 0; };
DxTmp dx_tmp_of(T like, int nodes, int n, int frames, int64_t max_bytes)
{
    DxTmp d;
    if (bbhip_GetDxMode() == 2) {
        d.frames = (int)tmp_frames(nodes, n, frames, max_bytes);
        d.stride = (d.frames + 63) / 64 * 64;
        d.t = rows_f32(like, (int64_t)nodes * n, d.stride);
        d.p = data<float>(d.t);
    }
    return d;
}

// dx_tmp given: described to the library in every mode (mode 2 needs it, mode 0 may fall back to it); tmp_frame_size < 0: as many as fit
at::Tensor stochastic_lut_backward(int n, T x, T dy, T idx, T W, T dW, int frames, OptTensor rev, bool input_binary, bool lut_binarize, float bias,
                                   OptTensor dx_tmp, int tmp_frame_size, double max_tmp_bytes, OptTensor out, OptTensor packed, bool overwrite, bool hints)
{
    int const I = rows_of(x), O = rows_of(idx), S = stride_of(dy);
    at::Tensor dx = out ? *out : rows_f32(x, I, S);
    DxTmp tmp;
    if (dx_tmp) {
        tmp.p = data<float>(dx_tmp); tmp.stride = stride_of(*dx_tmp);
        tmp.frames = tmp_frame_size >= 0 ? tmp_frame_size : (tmp.stride < frames ? tmp.stride : frames);
    }
    else { tmp = dx_tmp_of(x, O, n, frames, (int64_t)max_tmp_bytes); }
    if (hints) { hint_input(x, packed, true, false); }
    if (overwrite) { bbhip_HintTableGradientOverwrite(1); }
    call(bbhip_fp32_StochasticLut_Backward, n, data<float const>(x), data<float const>(dy), data<float>(dx), tmp.p, data<int const>(idx),
         data<int const>(rev), data<float const>(W), data<float>(dW), rev ? stride_of(*rev) : 0, I, O, frames, S, tmp.frames, tmp.stride,
         (int)input_binary, (int)lut_binarize, bias, current_stream());
    return dx;
}

at::Tensor bit_stochastic_lut_backward(int n, T x, T dy, T idx, T W, T dW, int frames, OptTensor rev, bool lut_binarize, float bias, double max_tmp_bytes)
{
    int const I = rows_of(x), O = rows_of(idx), S = stride_of(dy);
    at::Tensor dx = rows_f32(dy, I, S);
    DxTmp const tmp = dx_tmp_of(dy, O, n, frames, (int64_t)max_tmp_bytes);
    call(bbhip_bit_fp32_StochasticLut_Backward, n, data<int const>(x), data<float const>(dy), data<float>(dx), tmp.p, data<int const>(idx),
         data<int const>(rev), data<float const>(W), data<float>(dW), rev ? stride_of(*rev) : 0, I, O, frames, S, stride_of(x), tmp.frames, tmp.stride,
         (int)lut_binarize, bias, current_stream());
    return dx;
}

std::tuple<at::Tensor, at::Tensor, at::Tensor>
differentiable_lut_forward_training(int n, T x, T idx, T W, int frames, T running_mean, T running_var, float gamma, float beta, float momentum, float bias,
                                    bool lut_binarize, bool binary_mode, Clamp clamp, OptTensor packed, OptTensor tables, bool holds, OptTensor packed_out,
                                    bool hints)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = rows_f32(x, O, S);
    at::Tensor mean = line_f32(x, O), rstd = line_f32(x, O);
    if (hints) {
        hint_input(x, packed, holds, true);
        hint_tables(tables, false);
        if (binary_mode) { hint_output(packed_out, O); }
    }
    if (clamp.on) {
        call(bbhip_fp32_DifferentiableLutN_ForwardTrainingClampW, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float>(W),
             data<float>(mean), data<float>(rstd), data<float>(running_mean), data<float>(running_var), gamma, beta, momentum, bias, O, frames, S,
             (int)lut_binarize, (int)binary_mode, clamp.lo, clamp.hi, current_stream());
    }
    else {
        call(bbhip_fp32_DifferentiableLutN_ForwardTraining, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float const>(W),
             data<float>(mean), data<float>(rstd), data<float>(running_mean), data<float>(running_var), gamma, beta, momentum, bias, O, frames, S,
             (int)lut_binarize, (int)binary_mode, current_stream());
    }
    return {std::move(y), std::move(mean), std::move(rstd)};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor>
bit_differentiable_lut_forward_training(int n, T x, T idx, T W, int frames, T running_mean, T running_var, float gamma, float beta, float momentum,
                                        float bias, bool lut_binarize, Clamp clamp, OptTensor tables, OptTensor out, bool hints)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = packed_output(out, x, O, S);
    at::Tensor mean = line_f32(x, O), rstd = line_f32(x, O);
    if (hints) { hint_tables(tables, false); }
    if (clamp.on) {
        call(bbhip_bit_fp32_DifferentiableLutN_ForwardTrainingClampW, n, data<int const>(x), data<int>(y), data<int const>(idx), data<float>(W),
             data<float>(mean), data<float>(rstd), data<float>(running_mean), data<float>(running_var), gamma, beta, momentum, bias, O, frames, S,
             (int)lut_binarize, clamp.lo, clamp.hi, current_stream());
    }
    else {
        call(bbhip_bit_fp32_DifferentiableLutN_ForwardTraining, n, data<int const>(x), data<int>(y), data<int const>(idx), data<float const>(W),
             data<float>(mean), data<float>(rstd), data<float>(running_mean), data<float>(running_var), gamma, beta, momentum, bias, O, frames, S,
             (int)lut_binarize, current_stream());
    }
    return {std::move(y), std::move(mean), std::move(rstd)};
}

at::Tensor differentiable_lut_forward_inference(int n, T x, T idx, T W, int frames, T running_mean, T running_var, float gamma, float beta, float bias,
                                                bool lut_binarize, bool binary_mode, OptTensor packed, bool holds, OptTensor packed_out, bool hints)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = rows_f32(x, O, S);
    if (hints) {
        hint_input(x, packed, holds, true);
        if (binary_mode) { hint_output(packed_out, O); }
    }
    call(bbhip_fp32_DifferentiableLutN_ForwardInference, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float const>(W),
         data<float const>(running_mean), data<float const>(running_var), gamma, beta, bias, O, frames, S, (int)lut_binarize, (int)binary_mode,
         current_stream());
    return y;
}

at::Tensor bit_differentiable_lut_forward_inference(int n, T x, T idx, T W, int frames, T running_mean, T running_var, float gamma, float beta, float bias,
                                                    bool lut_binarize)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = packed_output(OptTensor{nullptr}, x, O, S);
    call(bbhip_bit_fp32_DifferentiableLutN_ForwardInference, n, data<int const>(x), data<int>(y), data<int const>(idx), data<float const>(W),
         data<float const>(running_mean), data<float const>(running_var), gamma, beta, bias, O, frames, S, (int)lut_binarize, current_stream());
    return y;
}

at::Tensor differentiable_lut_forward_nobn(int n, T x, T idx, T W, int frames, float bias, bool lut_binarize, bool binary_mode, OptTensor packed, bool holds,
                                           OptTensor packed_out, bool hints)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = rows_f32(x, O, S);
    if (hints) {
        hint_input(x, packed, holds, true);
        if (binary_mode) { hint_output(packed_out, O); }
    }
    call(bbhip_fp32_DifferentiableLutN_ForwardNoBn, n, data<float const>(x), data<float>(y), data<int const>(idx), data<float const>(W), bias, O, frames, S,
         (int)lut_binarize, (int)binary_mode, current_stream());
    return y;
}

at::Tensor differentiable_lut_backward(int n, T x, T dy, T idx, T W, T dW, int frames, T mean, T rstd, OptTensor rev, float gamma, float beta, float bias,
                                       bool lut_binarize, bool binary_mode, double max_tmp_bytes, OptTensor packed, OptTensor tables, bool overwrite,
                                       bool hints)
{
    int const I = rows_of(x), O = rows_of(idx), S = stride_of(dy);
    at::Tensor dx = rows_f32(x, I, S);
    float *const unused = data<float>(dx);          // dmean and dvar: any address that is not null (include/bbhip.h)
    DxTmp const tmp = dx_tmp_of(x, O, n, frames, (int64_t)max_tmp_bytes);
    if (hints) {
        hint_input(x, packed, true, false);
        hint_tables(tables, true);
    }
    if (overwrite) { bbhip_HintTableGradientOverwrite(1); }
    call(bbhip_fp32_DifferentiableLutN_Backward, n, data<float const>(x), data<float const>(dy), data<float>(dx), tmp.p, data<int const>(idx),
         data<int const>(rev), data<float const>(W), data<float>(dW), data<float const>(mean), data<float const>(rstd), unused, unused,
         gamma, beta, bias, rev ? stride_of(*rev) : 0, I, O, frames, S, tmp.frames, tmp.stride, (int)lut_binarize, (int)binary_mode,
         current_stream());
    return dx;
}

at::Tensor bit_differentiable_lut_backward(int n, T x, T dy, T idx, T W, T dW, int frames, T mean, T rstd, OptTensor rev, float gamma, float beta, float bias,
                                           bool lut_binarize, double max_tmp_bytes, OptTensor tables, bool hints)
{
    int const I = rows_of(x), O = rows_of(idx), S = stride_of(dy);
    at::Tensor dx = rows_f32(dy, I, S);
    float *const unused = data<float>(dx);          // dmean and dvar, as above
    DxTmp const tmp = dx_tmp_of(dy, O, n, frames, (int64_t)max_tmp_bytes);
    if (hints) { hint_tables(tables, true); }
    call(bbhip_bit_fp32_DifferentiableLutN_Backward, n, data<int const>(x), data<float const>(dy), data<float>(dx), tmp.p, data<int const>(idx),
         data<int const>(rev), data<float const>(W), data<float>(dW), data<float const>(mean), data<float const>(rstd), unused, unused,
         gamma, beta, bias, rev ? stride_of(*rev) : 0, I, O, frames, S, stride_of(x), tmp.frames, tmp.stride, (int)lut_binarize,
         current_stream());
    return dx;
}

at::Tensor binary_lut_forward(int n, T x, T idx, T table, int frames, OptTensor out)
{
    int const O = rows_of(idx), S = stride_of(x);
    at::Tensor y = packed_output(out, x, O, S);
    call(bbhip_bit_BinaryLutN_Forward, n, data<int const>(x), data<int>(y), data<int const>(idx), data<int const>(table), O, frames, S, current_stream());
    return y;
}

// ---- the classifier's tail ---------------------------------------------------------------------------------------------------------
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor>
classifier_tail(T x, T idx, T t, int frames, float t_sum, bool input_binary, bool mean, bool want_y, bool want_dy, bool want_accuracy)
{
    int const ch = rows_of(idx), n = stride_of(idx), S = stride_of(x), I = rows_of(x);
    require(t.size(1) == S, "classifier_tail: t must have the row pitch of x");
    require(frames >= 0, "classifier_tail: frames");
    at::Tensor y, dy, accuracy, category, dx = rows_f32(x, I, S), loss = new_tensor(x, {frames}, at::kDouble);
    if (want_y)  { y = rows_f32(x, ch, S); }
    if (want_dy) { dy = rows_f32(x, ch, S); }
    if (want_accuracy) { accuracy = new_tensor(x, {frames}, at::kInt); category = new_tensor(x, {frames}, at::kInt); }
    auto const f = [](at::Tensor const &a) { return a.defined() ? data<float>(a) : nullptr; };
    auto const i = [](at::Tensor const &a) { return a.defined() ? data<int>(a) : nullptr; };
    call(bbhip_fp32_ClassifierTail_ForwardBackward, data<float const>(x), f(y), data<float>(dx), data<int const>(idx), data<float const>(t), f(dy),
         data<double>(loss), i(accuracy), i(category), t_sum, n, I, ch, frames, S, (int)input_binary, (int)!mean, current_stream());
    return {std::move(y), std::move(dx), std::move(loss), std::move(accuracy), std::move(category), std::move(dy)};
}

// ---- Adam ------------------------------------------------------------------------------------------------------------------------
// the bias-corrected rate (AdamState.lr_t), every operation rounded to float: 0.1 us where numpy's scalars take 1.0
double adam_rate(float lr, float b1, float b2)
{
    float const root = std::sqrt(1.0f - b2), rate = lr * root;
    return (double)(rate / (1.0f - b1));
}

// ---- buffers for the wrappers that stay in Python ------------------------------------------------------------------------------------
at::Tensor new_rows(T like, int rows, int stride)  { return rows_f32(like, rows, stride); }
at::Tensor new_bits(T like, int rows, int words)   { return rows_i32(like, rows, words); }
at::Tensor new_padded_bits(T like, int rows, int words) { return packed_output(OptTensor{nullptr}, like, rows, words); }     // for the next call's output
at::Tensor new_zero_bits(T like, int rows, int words) { return zeros_i32(like, rows, words); }
at::Tensor new_line(T like, int n)                 { return line_f32(like, n); }

PyObject *set_error_type(PyObject *, PyObject *type) { Py_XINCREF(type); Py_XSETREF(g_error, type); Py_RETURN_NONE; }

#define BBHIP_FUNCTION(name) {#name, (PyCFunction)(void (*)(void))wrapped<Caller, &name>, METH_FASTCALL, nullptr}
#define BBHIP_ENTRY(name)    {#name, (PyCFunction)(void (*)(void))wrapped<EntryCaller, &bbhip_##name>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"set_error_type", set_error_type, METH_O, nullptr},
    BBHIP_FUNCTION(stochastic_lut_forward), BBHIP_FUNCTION(stochastic_lut_backward), BBHIP_FUNCTION(bit_stochastic_lut_backward),
    BBHIP_FUNCTION(differentiable_lut_forward_training), BBHIP_FUNCTION(bit_differentiable_lut_forward_training),
    BBHIP_FUNCTION(differentiable_lut_forward_inference), BBHIP_FUNCTION(bit_differentiable_lut_forward_inference),
    BBHIP_FUNCTION(differentiable_lut_forward_nobn), BBHIP_FUNCTION(differentiable_lut_backward), BBHIP_FUNCTION(bit_differentiable_lut_backward),
    BBHIP_FUNCTION(binary_lut_forward), BBHIP_FUNCTION(classifier_tail), BBHIP_FUNCTION(adam_rate),
    BBHIP_FUNCTION(new_rows), BBHIP_FUNCTION(new_bits), BBHIP_FUNCTION(new_padded_bits), BBHIP_FUNCTION(new_zero_bits), BBHIP_FUNCTION(new_line),
    BBHIP_ENTRY(fp32_Vector_set), BBHIP_ENTRY(fp32_Vector_clamp), BBHIP_ENTRY(fp32_Vector_add_ex), BBHIP_ENTRY(fp32_Vector_mul_ex),
    BBHIP_ENTRY(fp32_Vector_div_ex), BBHIP_ENTRY(fp32_Vector_sqrt), BBHIP_ENTRY(fp32_Vector_exp), BBHIP_ENTRY(fp32_Vector_min),
    BBHIP_ENTRY(fp32_Vector_min_v), BBHIP_ENTRY(fp32_Vector_max), BBHIP_ENTRY(fp32_Vector_max_v),
    BBHIP_ENTRY(fp32_OptimizerAdam), BBHIP_ENTRY(fp32_OptimizerAdam_Update),
    BBHIP_ENTRY(fp32_ConvBitToReal), BBHIP_ENTRY(fp32_Im2Col_Forward), BBHIP_ENTRY(bit_Im2Col_Forward), BBHIP_ENTRY(fp32_Im2Col_Backward),
    BBHIP_ENTRY(fp32_Col2Im_Forward), BBHIP_ENTRY(bit_Col2Im_Forward), BBHIP_ENTRY(fp32_Col2Im_Backward),
    BBHIP_ENTRY(fp32_StochasticMaxPooling2x2_Forward), BBHIP_ENTRY(fp32_StochasticMaxPooling2x2_Backward),
    BBHIP_ENTRY(fp32_StochasticBatchNormalization_ForwardTraining), BBHIP_ENTRY(fp32_StochasticBatchNormalization_ReForward),
    BBHIP_ENTRY(fp32_StochasticBatchNormalization_ForwardInference), BBHIP_ENTRY(fp32_StochasticBatchNormalization_Backward),
    BBHIP_ENTRY(fp32_AverageLut_Forward), BBHIP_ENTRY(fp32_AverageLut_ForwardSum), BBHIP_ENTRY(bit_AverageLut_Forward),
    BBHIP_ENTRY(fp32_AverageLut_Backward), BBHIP_ENTRY(fp32_MaxLut_Forward), BBHIP_ENTRY(bit_MaxLut_Forward), BBHIP_ENTRY(fp32_MaxLut_Backward),
    BBHIP_ENTRY(bit_fp32_MaxLut_Backward), BBHIP_ENTRY(fp32_Reduce_Forward), BBHIP_ENTRY(bit_fp32_Reduce_Forward), BBHIP_ENTRY(fp32_Reduce_Backward),
    BBHIP_ENTRY(fp32_LossMeanSquaredError), BBHIP_ENTRY(fp32_MetricsMeanSquaredError), BBHIP_ENTRY(fp32_LossSoftmaxCrossEntropy),
    BBHIP_ENTRY(fp32_MetricsCategoricalAccuracy), BBHIP_ENTRY(fp32_RealToBinary_Forward), BBHIP_ENTRY(fp32_bit_RealToBinary_Forward),
    BBHIP_ENTRY(fp32_BinaryToReal_Forward), BBHIP_ENTRY(bit_fp32_BinaryToReal_Forward), BBHIP_ENTRY(fp32_BinaryToReal_Backward),
    BBHIP_ENTRY(fp32_Binarize_Forward), BBHIP_ENTRY(fp32_bit_Binarize_Forward), BBHIP_ENTRY(fp32_HardTanh_Forward), BBHIP_ENTRY(fp32_HardTanh_Backward),
    BBHIP_ENTRY(fp32_MaxPooling_Forward), BBHIP_ENTRY(bit_MaxPooling_Forward), BBHIP_ENTRY(fp32_MaxPooling_Backward),
    BBHIP_ENTRY(bit_fp32_MaxPooling_Backward), BBHIP_ENTRY(fp32_UpSampling_Forward), BBHIP_ENTRY(bit_UpSampling_Forward),
    BBHIP_ENTRY(fp32_UpSampling_Backward), BBHIP_ENTRY(Shuffle_Forward), BBHIP_ENTRY(Shuffle_Backward),
    BBHIP_ENTRY(bit_fp32_StochasticLut_Forward), BBHIP_ENTRY(bit_bit_fp32_StochasticLut_Forward),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bbops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bbops(void) { return PyModule_Create(&module); }
