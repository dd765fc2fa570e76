// The call path of the Python binding for tensors that need no explanation.
//
// A decode-sized call (one token through one projection) takes the GPU 3.6 us.  Through ctypes the same call costs the
// host about 13 us: attribute look-ups and checks in Python, fifteen boxed arguments, two or three allocations through
// torch.empty and a stream object, each a microsecond or so.  These functions do the same checks on the tensors
// themselves, allocate the result, call the C ABI and return; what is left of the host's time is the launch.
//
// Every function answers None where anything at all is unusual (another type, device, layout or shape than the plain
// call takes, a status other than OK): the caller then runs its Python path, which makes the same call with every check
// spelled out and reports the error.  Nothing is computed here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Stream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>

#include "../../../include/bitnet_hip.h"

namespace {

PyObject *raw_stream_of = nullptr;   // torch._C._cuda_getCurrentRawStream
PyObject *name_cuda_stream = nullptr, *name_key = nullptr;

// The layer's (handle, in_features, out_features), which the binding keeps as the attribute `_key`.
struct Layer {
    bitnet_hip_bitlinear *handle = nullptr;
    int64_t in = 0, out = 0;
};
bool read_layer(PyObject *key, Layer &l)
{
    if (!PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key) != 3) return false;
    l.handle = static_cast<bitnet_hip_bitlinear *>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(key, 0)));
    l.in = PyLong_AsLongLong(PyTuple_GET_ITEM(key, 1));
    l.out = PyLong_AsLongLong(PyTuple_GET_ITEM(key, 2));
    return !PyErr_Occurred() && l.handle && l.in > 0 && l.out > 0;
}

// A dense f32 tensor on the current device, or null.
const at::Tensor *plain_f32(PyObject *obj, c10::Device &device)
{
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(obj);
    if (!t.is_cuda() || t.scalar_type() != at::kFloat || !t.is_contiguous()) return nullptr;
    if (device.index() < 0) {
        device = t.device();
        if (c10::impl::getDeviceGuardImpl(at::kCUDA)->getDevice() != device) return nullptr;
    } else if (t.device() != device) {
        return nullptr;
    }
    return &t;
}

// An optional operand of exactly `count` elements: true with *ptr set (null if absent), false if it is not plain.
bool optional_f32(PyObject *obj, int64_t count, c10::Device &device, const float **ptr)
{
    *ptr = nullptr;
    if (obj == Py_None) return true;
    const at::Tensor *t = plain_f32(obj, device);
    if (!t || t->numel() != count) return false;
    *ptr = t->const_data_ptr<float>();
    return true;
}

// The stream a call is made on.  `other` is set where the caller names one that is not the current stream.
struct CallStream {
    void *handle = nullptr;
    std::optional<c10::Stream> other;
};
bool call_stream(PyObject *obj, const c10::Device &device, CallStream &s)
{
    PyObject *v;
    if (obj == Py_None) {
        PyObject *index = PyLong_FromLong(device.index());
        if (!index) return false;
        v = PyObject_CallOneArg(raw_stream_of, index);
        Py_DECREF(index);
    } else {
        if (!THPStream_Check(obj)) return false;
        const THPStream *given = reinterpret_cast<const THPStream *>(obj);
        const c10::Stream stream = c10::Stream::unpack3(given->stream_id, static_cast<c10::DeviceIndex>(given->device_index),
                                                        static_cast<c10::DeviceType>(given->device_type));
        if (stream.device() != device) return false;
        if (c10::impl::getDeviceGuardImpl(at::kCUDA)->getStream(device) != stream) s.other = stream;
        v = PyObject_GetAttr(obj, name_cuda_stream);
    }
    if (!v) return false;
    s.handle = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !PyErr_Occurred();
}

PyObject *unusual()
{
    PyErr_Clear();
    Py_RETURN_NONE;
}

// What torch's dispatcher ends in for an empty tensor on a device, called directly unless a dispatch mode of Python's wants to see it.  With
// launch_kernel (csrc/common.hpp) calls of one to eight tokens 4.4 -> 4.05 us, ones that bring scratch 5.8 -> 5.1.
at::Tensor fresh(at::IntArrayRef shape, const at::TensorOptions &options)
{
    if (c10::impl::dispatch_mode_enabled()) {
        at::AutoDispatchBelowADInplaceOrView below;
        return at::empty(shape, options);
    }
    return at::detail::empty_cuda(shape, c10::typeMetaToScalarType(options.dtype()), options.device(), std::nullopt);
}

// Memory that the call's kernels use.  The allocator hands a block out, and takes it back, in the order of one stream, so the
// block is asked for on the stream the call runs on: what is freed there before its kernels have run (scratch, a result the
// caller drops) goes to later work of that stream only.  The caller may use a result on the current stream as well and drop it
// there, which the allocator is told.
at::Tensor new_on(const CallStream &s, at::IntArrayRef shape, const at::TensorOptions &options)
{
    if (!s.other) return fresh(shape, options);
    const c10::impl::DeviceGuardImplInterface *impl = c10::impl::getDeviceGuardImpl(at::kCUDA);
    const c10::Stream current = impl->exchangeStream(*s.other);
    struct Back {
        const c10::impl::DeviceGuardImplInterface *impl;
        c10::Stream current;
        ~Back() { impl->exchangeStream(current); }
    };
    at::Tensor t;
    {
        const Back back{impl, current};
        t = fresh(shape, options);
    }
    impl->recordDataPtrOnStream(t.storage().data_ptr(), current);
    return t;
}

// forward(key, x, gamma, residual, out, eps, sum_order, stream)
PyObject *forward(PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 8) return unusual();
    Layer l;
    c10::Device device(at::kCUDA, -1);
    if (!read_layer(args[0], l)) return unusual();
    const at::Tensor *x = plain_f32(args[1], device);
    if (!x) return unusual();
    const int64_t rank = x->dim();
    if ((rank != 2 && rank != 3) || x->size(rank - 1) != l.in) return unusual();
    const int64_t m = rank == 2 ? x->size(0) : x->size(0) * x->size(1);
    const float *gamma, *residual;
    if (m == 0 || !optional_f32(args[2], l.in, device, &gamma) || !optional_f32(args[3], m * l.out, device, &residual))
        return unusual();
    const double eps = PyFloat_AsDouble(args[5]);
    const long order = PyLong_AsLong(args[6]);
    CallStream stream;
    if (PyErr_Occurred() || !call_stream(args[7], device, stream)) return unusual();
    size_t dims[3] = {(size_t)x->size(0), (size_t)x->size(1), rank == 3 ? (size_t)x->size(2) : 0};
    at::Tensor made;
    const at::Tensor *y;
    if (args[4] == Py_None) {
        const int64_t shape[3] = {x->size(0), rank == 3 ? x->size(1) : l.out, l.out};
        made = new_on(stream, at::IntArrayRef(shape, rank), x->options());
        y = &made;
    } else {
        y = plain_f32(args[4], device);
        if (!y || y->dim() != rank || y->size(rank - 1) != l.out || y->numel() != m * l.out || y->size(0) != x->size(0))
            return unusual();
    }
    // scratch only where the call runs the stand-alone quantiser
    const float *xp = x->const_data_ptr<float>();
    size_t ws_bytes = bitnet_hip_bitlinear_forward_scratch_on(&l.handle, 1, xp, (size_t)m, gamma, (int)order, stream.handle);
    float *yp = y->data_ptr<float>();
    // a result over the input takes two launches, and scratch, whatever the size
    if (!ws_bytes && yp < xp + m * l.in && xp < yp + m * l.out) ws_bytes = bitnet_hip_bitlinear_workspace_size(l.handle, (size_t)m);
    at::Tensor ws;
    if (ws_bytes) ws = new_on(stream, {(int64_t)((ws_bytes + 3) / 4)}, x->options());
    void *wp = ws_bytes ? ws.data_ptr() : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bitnet_hip_bitlinear_forward(l.handle, xp, dims, (int)rank, gamma, (float)eps, (int)order, residual, yp, wp, ws_bytes,
                                      nullptr, nullptr, nullptr, stream.handle);
    Py_END_ALLOW_THREADS
    if (rc != BITNET_HIP_OK) return unusual();
    if (args[4] != Py_None) {
        Py_INCREF(args[4]);
        return args[4];
    }
    return THPVariable_Wrap(made);
}

// forward_multi(layers, x, gamma, eps, sum_order, stream)
PyObject *forward_multi(PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 6) return unusual();
    constexpr Py_ssize_t MOST = 16;
    PyObject *seq = args[0];
    const bool list = PyList_CheckExact(seq);
    if (!list && !PyTuple_CheckExact(seq)) return unusual();
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
    if (count < 1 || count > MOST) return unusual();
    bitnet_hip_bitlinear *handles[MOST];
    int64_t widths[MOST];
    c10::Device device(at::kCUDA, -1);
    const at::Tensor *x = plain_f32(args[1], device);
    if (!x || x->dim() != 2) return unusual();
    const int64_t m = x->size(0), k = x->size(1);
    for (Py_ssize_t j = 0; j < count; ++j) {
        PyObject *key = PyObject_GetAttr(PySequence_Fast_GET_ITEM(seq, j), name_key);
        Layer l;
        const bool ok = key && read_layer(key, l) && l.in == k;
        Py_XDECREF(key);
        if (!ok) return unusual();
        handles[j] = l.handle;
        widths[j] = l.out;
    }
    const float *gamma;
    if (m == 0 || !optional_f32(args[2], k, device, &gamma)) return unusual();
    const double eps = PyFloat_AsDouble(args[3]);
    const long order = PyLong_AsLong(args[4]);
    CallStream stream;
    if (PyErr_Occurred() || !call_stream(args[5], device, stream)) return unusual();
    at::Tensor outs[MOST];
    float *ptrs[MOST];
    for (Py_ssize_t j = 0; j < count; ++j) {
        outs[j] = new_on(stream, {m, widths[j]}, x->options());
        ptrs[j] = outs[j].data_ptr<float>();
    }
    const float *xp = x->const_data_ptr<float>();
    const size_t ws_bytes = bitnet_hip_bitlinear_forward_scratch_on(handles, (size_t)count, xp, (size_t)m, gamma, (int)order, stream.handle);
    at::Tensor ws;
    if (ws_bytes) ws = new_on(stream, {(int64_t)((ws_bytes + 3) / 4)}, x->options());
    void *wp = ws_bytes ? ws.data_ptr() : nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bitnet_hip_bitlinear_forward_multi(handles, (size_t)count, xp, (size_t)m, gamma, (float)eps, (int)order, ptrs, wp,
                                            ws_bytes, stream.handle);
    Py_END_ALLOW_THREADS
    if (rc != BITNET_HIP_OK) return unusual();
    PyObject *res = PyList_New(count);
    if (!res) return nullptr;
    for (Py_ssize_t j = 0; j < count; ++j) {
        PyObject *t = THPVariable_Wrap(outs[j]);
        if (!t) {
            Py_DECREF(res);
            return nullptr;
        }
        PyList_SET_ITEM(res, j, t);
    }
    return res;
}

// decode(decoder, hidden, begin, end, x, out, stream)
PyObject *decode(PyObject *const *args, Py_ssize_t nargs)
{
    if (nargs != 7) return unusual();
    auto *dec = static_cast<bitnet_hip_decoder *>(PyLong_AsVoidPtr(args[0]));
    const int64_t hidden = PyLong_AsLongLong(args[1]), begin = PyLong_AsLongLong(args[2]), end = PyLong_AsLongLong(args[3]);
    c10::Device device(at::kCUDA, -1);
    if (PyErr_Occurred() || !dec || begin < 0 || end < begin) return unusual();
    const at::Tensor *x = plain_f32(args[4], device);
    if (!x || x->dim() != 2 || x->size(1) != hidden) return unusual();
    CallStream stream;
    if (!call_stream(args[6], device, stream)) return unusual();
    at::Tensor made;
    const at::Tensor *y;
    if (args[5] == Py_None) {
        made = new_on(stream, x->sizes(), x->options());
        y = &made;
    } else {
        y = plain_f32(args[5], device);
        if (!y || y->sizes() != x->sizes()) return unusual();
    }
    const float *xp = x->const_data_ptr<float>();
    float *yp = y->data_ptr<float>();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bitnet_hip_decoder_decode_layers(dec, (size_t)begin, (size_t)end, xp, (size_t)x->size(0), yp, nullptr, nullptr, stream.handle);
    Py_END_ALLOW_THREADS
    if (rc != BITNET_HIP_OK) return unusual();
    if (args[5] != Py_None) {
        Py_INCREF(args[5]);
        return args[5];
    }
    return THPVariable_Wrap(made);
}

// abs_max(x, stream): the float, or None
PyObject *abs_max(PyObject *const *args, Py_ssize_t nargs)
{
    c10::Device device(at::kCUDA, -1);
    if (nargs != 2) return unusual();
    const at::Tensor *x = plain_f32(args[0], device);
    CallStream stream;
    if (!x || !call_stream(args[1], device, stream)) return unusual();
    const float *xp = x->const_data_ptr<float>();
    const size_t count = (size_t)x->numel();
    float v = 0.0f;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bitnet_hip_abs_max(xp, count, &v, stream.handle);
    Py_END_ALLOW_THREADS
    return rc == BITNET_HIP_OK ? PyFloat_FromDouble(v) : unusual();
}

// quantize_scaled(x, precision, scale, reference_u8, stream): (int8 values, scale tensor [1])
PyObject *quantize_scaled(PyObject *const *args, Py_ssize_t nargs)
{
    c10::Device device(at::kCUDA, -1);
    if (nargs != 5) return unusual();
    const at::Tensor *x = plain_f32(args[0], device);
    const long precision = PyLong_AsLong(args[1]);
    const double scale = PyFloat_AsDouble(args[2]);
    const int u8 = PyObject_IsTrue(args[3]);
    CallStream stream;
    if (!x || PyErr_Occurred() || u8 < 0 || !call_stream(args[4], device, stream)) return unusual();
    const at::Tensor values = new_on(stream, x->sizes(), x->options().dtype(at::kChar)), scales = new_on(stream, {1}, x->options());
    if (bitnet_hip_quantize_activations_scaled_keep(x->const_data_ptr<float>(), (size_t)x->numel(), (int)precision, (float)scale, u8,
                                                    values.data_ptr<int8_t>(), scales.data_ptr<float>(), stream.handle) != BITNET_HIP_OK)
        return unusual();
    PyObject *v = THPVariable_Wrap(values), *sc = THPVariable_Wrap(scales);
    PyObject *pair = v && sc ? PyTuple_Pack(2, v, sc) : nullptr;
    Py_XDECREF(v);
    Py_XDECREF(sc);
    return pair;
}

// quantize_dynamic(x, precision, average or None, decay, reference_u8, stream): (int8 values, scale tensor [1], max |x|)
PyObject *quantize_dynamic(PyObject *const *args, Py_ssize_t nargs)
{
    c10::Device device(at::kCUDA, -1);
    if (nargs != 6) return unusual();
    const at::Tensor *x = plain_f32(args[0], device);
    const long precision = PyLong_AsLong(args[1]);
    const bool averaged = args[2] != Py_None;
    const float average = averaged ? (float)PyFloat_AsDouble(args[2]) : 0.0f, decay = (float)PyFloat_AsDouble(args[3]);
    const int u8 = PyObject_IsTrue(args[4]);
    CallStream stream;
    if (!x || x->numel() == 0 || PyErr_Occurred() || u8 < 0 || !call_stream(args[5], device, stream)) return unusual();
    const at::Tensor values = new_on(stream, x->sizes(), x->options().dtype(at::kChar)), scales = new_on(stream, {1}, x->options()),
                     scratch = new_on(stream, {256}, x->options());
    const float *xp = x->const_data_ptr<float>();
    const size_t count = (size_t)x->numel();
    int8_t *vp = values.data_ptr<int8_t>();
    float *sp = scales.data_ptr<float>(), *tp = scratch.data_ptr<float>(), abs_max = 0.0f;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = bitnet_hip_quantize_activations_dynamic(xp, count, (int)precision, averaged ? &average : nullptr, decay, u8, vp, sp, &abs_max, tp, stream.handle);
    Py_END_ALLOW_THREADS
    if (rc != BITNET_HIP_OK) return unusual();
    PyObject *v = THPVariable_Wrap(values), *sc = THPVariable_Wrap(scales), *am = PyFloat_FromDouble(abs_max);
    PyObject *res = v && sc && am ? PyTuple_Pack(3, v, sc, am) : nullptr;
    Py_XDECREF(v);
    Py_XDECREF(sc);
    Py_XDECREF(am);
    return res;
}

// What Python calls: a C++ exception (a tensor without storage or strides refuses the question, an allocation fails) must not pass
// into the interpreter, where it would end the process.
template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    try {
        return F(args, nargs);
    } catch (...) {
        return unusual();
    }
}

template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
PyMethodDef method(const char *name)
{
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<F>)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {
    method<quantize_dynamic>("quantize_dynamic"),
    method<abs_max>("abs_max"),
    method<quantize_scaled>("quantize_scaled"),
    method<forward>("forward"),
    method<forward_multi>("forward_multi"),
    method<decode>("decode"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call()
{
    PyObject *torch_c = PyImport_ImportModule("torch._C");
    if (!torch_c) return nullptr;
    raw_stream_of = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
    Py_DECREF(torch_c);
    name_cuda_stream = PyUnicode_InternFromString("cuda_stream");
    name_key = PyUnicode_InternFromString("_key");
    if (!raw_stream_of || !name_cuda_stream || !name_key) return nullptr;
    return PyModule_Create(&module);
}
