// Native face of ops.py: tensors to descriptors, result allocation and the call into libchx_hip.so without ctypes.
// Filling two descriptors attribute by attribute, allocating and converting the arguments took 12 us of Python per op,
// more than most launches of this path run for; here it is about 2 (and the launch itself 2.4).
//
// The functions take exactly the positional arguments listed above each; ops.py has the signatures, the defaults and the
// attribute rules that need the reference's text (auto_pad).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <string>

#include <chx_hip.h>

#include "../runtime/chxvm_capi.h"

namespace {

PyObject* g_error = nullptr;  // capi.ChxHipError(code, message)

struct PythonError {};  // a Python exception is set

[[noreturn]] void fail(PyObject* type, const char* message) {
    PyErr_SetString(type, message);
    throw PythonError();
}

int32_t dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kBool: return CHX_HIP_BOOL;
        case at::kChar: return CHX_HIP_INT8;
        case at::kShort: return CHX_HIP_INT16;
        case at::kInt: return CHX_HIP_INT32;
        case at::kLong: return CHX_HIP_INT64;
        case at::kByte: return CHX_HIP_UINT8;
        case at::kHalf: return CHX_HIP_FLOAT16;
        case at::kFloat: return CHX_HIP_FLOAT32;
        case at::kDouble: return CHX_HIP_FLOAT64;
        default: fail(PyExc_KeyError, "tensor of a type the library does not have");
    }
}

int64_t element_size(int32_t code) {
    switch (code) {
        case CHX_HIP_INT16: case CHX_HIP_FLOAT16: return 2;
        case CHX_HIP_INT32: case CHX_HIP_FLOAT32: return 4;
        case CHX_HIP_INT64: case CHX_HIP_FLOAT64: return 8;
        default: return 1;
    }
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) fail(PyExc_TypeError, "a torch tensor is expected");
    return THPVariable_Unpack(o);
}

void describe(const at::Tensor& t, chx_hip_tensor* d) {
    const int64_t nd = t.dim(), es = t.element_size();
    if (nd > CHX_HIP_MAX_NDIM) fail(PyExc_IndexError, "tensor with more axes than the library has");
    memset(d, 0, sizeof(*d));
    d->data = t.data_ptr();
    d->dtype = dtype_code(t.scalar_type());
    d->ndim = static_cast<int32_t>(nd);
    for (int64_t i = 0; i < nd; ++i) {
        d->shape[i] = t.size(i);
        d->strides[i] = t.stride(i) * es;
    }
}

// A tensor argument that may be None.
struct Operand {
    chx_hip_tensor desc;
    chx_hip_tensor* ptr = nullptr;
    explicit Operand(PyObject* o) {
        if (o == Py_None) return;
        describe(tensor(o), &desc);
        ptr = &desc;
    }
    explicit Operand(const at::Tensor& t) {
        describe(t, &desc);
        ptr = &desc;
    }
};

double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PythonError();
    return v;
}

long long integer(PyObject* o) {
    if (PyLong_CheckExact(o)) {
        const long long v = PyLong_AsLongLong(o);
        if (v == -1 && PyErr_Occurred()) throw PythonError();
        return v;
    }
    PyObject* n = PyNumber_Long(o);
    if (!n) throw PythonError();
    const long long v = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v == -1 && PyErr_Occurred()) throw PythonError();
    return v;
}

at::ScalarType scalar_type(PyObject* o) {
    if (!THPDtype_Check(o)) fail(PyExc_TypeError, "a torch dtype is expected");
    return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

void* current_stream() {
    return c10::hip::getCurrentHIPStream().stream();
}

// Runs `call` without the interpreter lock (some entry points wait for the device) and raises on an error code.
template <class F>
void checked(F call) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call();
    Py_END_ALLOW_THREADS
    if (rc == 0) return;
    PyObject* args = Py_BuildValue("(iN)", rc, PyUnicode_DecodeUTF8(chx_hip_last_error(), static_cast<Py_ssize_t>(strlen(chx_hip_last_error())), "replace"));
    if (args) {
        PyObject* e = PyObject_CallObject(g_error, args);
        Py_DECREF(args);
        if (e) {
            PyErr_SetObject(g_error, e);
            Py_DECREF(e);
        }
    }
    throw PythonError();
}

template <class F>
PyObject* guarded(F body) {
    try {
        return body();
    } catch (const PythonError&) {
        return nullptr;
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
        return nullptr;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

void need(Py_ssize_t given, Py_ssize_t wanted) {
    if (given != wanted) fail(PyExc_TypeError, "wrong number of arguments");
}

// Channels-last memory that is not C-contiguous as well (what ops.py asks with permute(0, 2, 3, 1).is_contiguous()).
bool channels_last(const at::Tensor& x) {
    if (x.dim() != 4 || x.is_contiguous()) return false;
    int64_t expect = 1;
    for (int ax : {1, 3, 2, 0}) {
        if (x.size(ax) != 1 && x.stride(ax) != expect) return false;
        expect *= x.size(ax);
    }
    return true;
}

at::Tensor empty_nhwc(at::IntArrayRef nchw, const at::TensorOptions& options) {
    const int64_t c = nchw[1], h = nchw[2], w = nchw[3];
    return at::empty_strided(nchw, {h * w * c, 1, w * c, c}, options);
}

at::Tensor result_like(const at::Tensor& x, at::IntArrayRef shape, at::ScalarType type) {
    const at::TensorOptions options = x.options().dtype(type);
    return channels_last(x) ? empty_nhwc(shape, options) : at::empty(shape, options);
}

PyObject* wrapped(PyObject* out, const at::Tensor& made) {
    if (out != Py_None) {
        Py_INCREF(out);
        return out;
    }
    return THPVariable_Wrap(made);
}

// (stride_h, stride_w, pad_h_begin, pad_w_begin, pad_h_end, pad_w_end, group)
chx_hip_conv_params conv_params(PyObject* o) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 7) fail(PyExc_TypeError, "a tuple of seven numbers describes a convolution");
    int32_t v[7];
    for (int i = 0; i < 7; ++i) v[i] = static_cast<int32_t>(integer(PyTuple_GET_ITEM(o, i)));
    return chx_hip_conv_params{v[0], v[1], v[2], v[3], v[4], v[5], v[6]};
}

at::Tensor conv_result(const at::Tensor& x, int64_t oc, int64_t kh, int64_t kw, const chx_hip_conv_params& p, at::ScalarType type) {
    auto out = [](int64_t in, int64_t begin, int64_t end, int64_t k, int64_t stride) {
        // (a window that does not fit gives an extent of 0 or less, which the library or the allocation refuses)
        if (stride == 0) fail(PyExc_ZeroDivisionError, "a stride of 0");
        const int64_t room = in + begin + end - k, q = room / stride;
        return (room % stride != 0 && (room < 0) != (stride < 0) ? q - 1 : q) + 1;
    };
    return result_like(x, {x.size(0), oc, out(x.size(2), p.pad_h_begin, p.pad_h_end, kh, p.stride_h), out(x.size(3), p.pad_w_begin, p.pad_w_end, kw, p.stride_w)}, type);
}

at::Tensor matmul_result(const at::Tensor& a, const at::Tensor& b, at::ScalarType type) {
    if (a.dim() < 1 || b.dim() < 1) fail(PyExc_IndexError, "a matrix product of 0-d tensors");
    c10::SmallVector<int64_t, 8> shape(a.sizes().begin(), a.sizes().end());
    shape.back() = b.size(-1);
    return at::empty(shape, a.options().dtype(type));
}

// init(ChxHipError)
PyObject* init(PyObject*, PyObject* error) {
    Py_INCREF(error);
    Py_XDECREF(g_error);
    g_error = error;
    Py_RETURN_NONE;
}

// quantize_linear(x, y_scale, y_zero_point, dtype, flags, out or None)
PyObject* quantize_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 6);
        const at::Tensor& x = tensor(a[0]);
        const float scale = static_cast<float>(number(a[1]));
        const int32_t zp = static_cast<int32_t>(integer(a[2]));
        const uint32_t flags = static_cast<uint32_t>(integer(a[4]));
        at::Tensor made;
        if (a[5] == Py_None) made = at::empty_like(x, x.options().dtype(scalar_type(a[3])));
        Operand xd(x), yd(a[5] == Py_None ? made : tensor(a[5]));
        void* s = current_stream();
        checked([&] { return chx_hip_quantize_linear(xd.ptr, scale, zp, flags, yd.ptr, s); });
        return wrapped(a[5], made);
    });
}

// dequantize_linear(x, x_scale, x_zero_point, out or None)
PyObject* dequantize_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 4);
        const at::Tensor& x = tensor(a[0]);
        const float scale = static_cast<float>(number(a[1]));
        const int32_t zp = static_cast<int32_t>(integer(a[2]));
        at::Tensor made;
        if (a[3] == Py_None) made = at::empty_like(x, x.options().dtype(at::kFloat));
        Operand xd(x), yd(a[3] == Py_None ? made : tensor(a[3]));
        void* s = current_stream();
        checked([&] { return chx_hip_dequantize_linear(xd.ptr, scale, zp, yd.ptr, s); });
        return wrapped(a[3], made);
    });
}

// elementwise(inputs, code bytes, fusion id, tuple of result dtypes, outs or None) -> list of results
PyObject* elementwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 5);
        constexpr Py_ssize_t kMost = 64;
        PyObject* ins = PySequence_Fast(a[0], "a sequence of inputs is expected");
        if (!ins) throw PythonError();
        struct Release {
            PyObject* o;
            ~Release() { Py_XDECREF(o); }
        } release_ins{ins};
        const Py_ssize_t nin = PySequence_Fast_GET_SIZE(ins), nout = PyTuple_Check(a[3]) ? PyTuple_GET_SIZE(a[3]) : -1;
        if (nin < 1 || nin > kMost || nout < 0 || nout > kMost) fail(PyExc_ValueError, "a fusion group has 1 to 64 inputs and results");
        const char* code = PyBytes_AsString(a[1]);
        if (!code) throw PythonError();
        const int32_t id = static_cast<int32_t>(integer(a[2]));
        chx_hip_tensor desc[2 * kMost];
        const chx_hip_tensor* in[kMost];
        chx_hip_tensor* out[kMost];
        int64_t shape[CHX_HIP_MAX_NDIM];
        int nd = 0;
        for (Py_ssize_t i = 0; i < nin; ++i) {
            describe(tensor(PySequence_Fast_GET_ITEM(ins, i)), &desc[i]);
            in[i] = &desc[i];
            nd = std::max(nd, static_cast<int>(desc[i].ndim));
        }
        PyObject* results = nullptr;
        if (a[4] == Py_None) {
            for (int ax = 0; ax < nd; ++ax) shape[ax] = 1;
            for (Py_ssize_t i = 0; i < nin; ++i)
                for (int ax = 0; ax < desc[i].ndim; ++ax) {
                    int64_t& to = shape[nd - desc[i].ndim + ax];
                    if (desc[i].shape[ax] == 1) continue;
                    if (to != 1 && to != desc[i].shape[ax]) fail(PyExc_RuntimeError, "the shapes of the inputs do not broadcast");
                    to = desc[i].shape[ax];
                }
            const at::IntArrayRef sizes(shape, static_cast<size_t>(nd));
            // channels-last when every operand of the full shape is, so that chains between convolutions never transpose
            bool any = false, all = nd == 4;
            for (Py_ssize_t i = 0; i < nin && all; ++i) {
                const at::Tensor& t = tensor(PySequence_Fast_GET_ITEM(ins, i));
                if (t.sizes() != sizes) continue;
                any = true;
                all = channels_last(t);
            }
            const at::TensorOptions base = tensor(PySequence_Fast_GET_ITEM(ins, 0)).options();
            results = PyList_New(nout);
            if (!results) throw PythonError();
            Release guard{results};
            for (Py_ssize_t i = 0; i < nout; ++i) {
                const at::TensorOptions o = base.dtype(scalar_type(PyTuple_GET_ITEM(a[3], i)));
                at::Tensor t = any && all ? empty_nhwc(sizes, o) : at::empty(sizes, o);
                describe(t, &desc[nin + i]);
                PyObject* w = THPVariable_Wrap(std::move(t));
                if (!w) throw PythonError();
                PyList_SET_ITEM(results, i, w);
            }
            guard.o = nullptr;
        } else {
            results = a[4];
            Py_INCREF(results);
            Release guard{results};
            PyObject* outs = PySequence_Fast(results, "a sequence of results is expected");
            if (!outs) throw PythonError();
            Release release_outs{outs};
            if (PySequence_Fast_GET_SIZE(outs) != nout) fail(PyExc_ValueError, "as many results as the program has outputs are expected");
            for (Py_ssize_t i = 0; i < nout; ++i) describe(tensor(PySequence_Fast_GET_ITEM(outs, i)), &desc[nin + i]);
            guard.o = nullptr;
        }
        Release guard{results};
        for (Py_ssize_t i = 0; i < nout; ++i) out[i] = &desc[nin + i];
        void* s = current_stream();
        checked([&] { return chx_hip_elementwise(code, id, in, static_cast<int32_t>(nin), out, static_cast<int32_t>(nout), s); });
        guard.o = nullptr;
        return results;
    });
}

// qlinear_conv(x, x_scale, x_zero_point, w, w_scale, w_zero_point, y_scale, y_zero_point, b or None, geometry, dtype, flags, out or None)
PyObject* qlinear_conv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 13);
        const at::Tensor &x = tensor(a[0]), &w = tensor(a[3]);
        const float xs = static_cast<float>(number(a[1])), ys = static_cast<float>(number(a[6]));
        const int32_t xz = static_cast<int32_t>(integer(a[2])), yz = static_cast<int32_t>(integer(a[7]));
        const chx_hip_conv_params p = conv_params(a[9]);
        const uint32_t flags = static_cast<uint32_t>(integer(a[11]));
        at::Tensor made;
        if (a[12] == Py_None) made = conv_result(x, w.size(0), w.size(2), w.size(3), p, scalar_type(a[10]));
        Operand xd(x), wd(w), sd(a[4]), zd(a[5]), bd(a[8]), yd(a[12] == Py_None ? made : tensor(a[12]));
        void* s = current_stream();
        checked([&] { return chx_hip_qlinear_conv(xd.ptr, xs, xz, wd.ptr, sd.ptr, zd.ptr, ys, yz, bd.ptr, &p, flags, yd.ptr, s); });
        return wrapped(a[12], made);
    });
}

// conv_integer(x, w, x_zero_point, w_zero_point or None, geometry, out or None)
PyObject* conv_integer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 6);
        const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
        const int32_t xz = static_cast<int32_t>(integer(a[2]));
        const chx_hip_conv_params p = conv_params(a[4]);
        at::Tensor made;
        if (a[5] == Py_None) made = conv_result(x, w.size(0), w.size(2), w.size(3), p, at::kInt);
        Operand xd(x), wd(w), zd(a[3]), yd(a[5] == Py_None ? made : tensor(a[5]));
        void* s = current_stream();
        checked([&] { return chx_hip_conv_integer(xd.ptr, wd.ptr, xz, zd.ptr, &p, yd.ptr, s); });
        return wrapped(a[5], made);
    });
}

// matmul_integer(a, b, a_zero_point or None, b_zero_point or None, out or None)
PyObject* matmul_integer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 5);
        at::Tensor made;
        if (a[4] == Py_None) made = matmul_result(tensor(a[0]), tensor(a[1]), at::kInt);
        Operand ad(a[0]), bd(a[1]), az(a[2]), bz(a[3]), yd(a[4] == Py_None ? made : tensor(a[4]));
        void* s = current_stream();
        checked([&] { return chx_hip_matmul_integer(ad.ptr, bd.ptr, az.ptr, bz.ptr, yd.ptr, s); });
        return wrapped(a[4], made);
    });
}

// qlinear_matmul(a, a_scale, a_zero_point, b, b_scale, b_zero_point, y_scale, y_zero_point, bias or None, dtype, flags, out or None)
PyObject* qlinear_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 12);
        const float as = static_cast<float>(number(a[1])), bs = static_cast<float>(number(a[4])), ys = static_cast<float>(number(a[6]));
        const int32_t az = static_cast<int32_t>(integer(a[2])), bz = static_cast<int32_t>(integer(a[5])), yz = static_cast<int32_t>(integer(a[7]));
        const uint32_t flags = static_cast<uint32_t>(integer(a[10]));
        at::Tensor made;
        if (a[11] == Py_None) made = matmul_result(tensor(a[0]), tensor(a[3]), scalar_type(a[9]));
        Operand ad(a[0]), bd(a[3]), bias(a[8]), yd(a[11] == Py_None ? made : tensor(a[11]));
        void* s = current_stream();
        checked([&] { return chx_hip_qlinear_matmul(ad.ptr, as, az, bd.ptr, bs, bz, ys, yz, bias.ptr, flags, yd.ptr, s); });
        return wrapped(a[11], made);
    });
}

// plan_run(plan, x, (oc, kh, kw), geometry, x_scale, x_zero_point, y_scale, y_zero_point, dtype, flags, out or None)
PyObject* plan_run(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 11);
        const chx_hip_qconv_plan* plan = reinterpret_cast<const chx_hip_qconv_plan*>(integer(a[0]));
        const at::Tensor& x = tensor(a[1]);
        if (x.dim() != 4) fail(PyExc_ValueError, "a convolution plan takes a tensor of four axes");
        const float xs = static_cast<float>(number(a[4])), ys = static_cast<float>(number(a[6]));
        const int32_t xz = static_cast<int32_t>(integer(a[5])), yz = static_cast<int32_t>(integer(a[7]));
        const uint32_t flags = static_cast<uint32_t>(integer(a[9]));
        at::Tensor made;
        if (a[10] == Py_None) {
            if (!PyTuple_Check(a[2]) || PyTuple_GET_SIZE(a[2]) != 3) fail(PyExc_TypeError, "(oc, kh, kw) is expected");
            made = conv_result(x, integer(PyTuple_GET_ITEM(a[2], 0)), integer(PyTuple_GET_ITEM(a[2], 1)), integer(PyTuple_GET_ITEM(a[2], 2)), conv_params(a[3]),
                               scalar_type(a[8]));
        }
        Operand xd(x), yd(a[10] == Py_None ? made : tensor(a[10]));
        void* s = current_stream();
        checked([&] { return chx_hip_qconv_plan_run(plan, xd.ptr, xs, xz, ys, yz, flags, yd.ptr, s); });
        return wrapped(a[10], made);
    });
}

// ---- runs of the virtual machine (chxvm.py); its library is loaded by the caller, who hands the entry points over ----
struct Machine {
    decltype(&chxvm_program_run_to_host) run;
    decltype(&chxvm_outputs_count) count;
    decltype(&chxvm_outputs_name) name;
    decltype(&chxvm_outputs_layout) layout;
    decltype(&chxvm_outputs_host) host;
    decltype(&chxvm_outputs_destroy) destroy;
} g_machine;

// vm_init(address of each, in the order above)
PyObject* vm_init(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 6);
        void* at[6];
        for (int i = 0; i < 6; ++i) at[i] = reinterpret_cast<void*>(integer(a[i]));
        static_assert(sizeof(g_machine) == sizeof(at), "six addresses");
        memcpy(&g_machine, at, sizeof(at));
        Py_RETURN_NONE;
    });
}

// [(name, dtype code, shape, bytearray with the dense elements)], or null, with no exception set, when the runtime has
// no host copy of one of them
PyObject* host_copies(const chxvm_outputs* out) {
    const int32_t n = g_machine.count(out);
    PyObject* list = PyList_New(n);
    if (!list) throw PythonError();
    for (int32_t i = 0; i < n; ++i) {
        chx_hip_tensor d;
        const void* p = nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = g_machine.layout(out, i, &d);
        if (rc == 0) p = g_machine.host(out, i);
        Py_END_ALLOW_THREADS
        if (!p) {
            Py_DECREF(list);
            return nullptr;
        }
        int64_t bytes = element_size(d.dtype);
        PyObject* shape = PyTuple_New(d.ndim);
        for (int32_t k = 0; shape && k < d.ndim; ++k) {
            bytes *= d.shape[k];
            PyTuple_SET_ITEM(shape, k, PyLong_FromLongLong(d.shape[k]));
        }
        PyObject* item = shape ? Py_BuildValue("(siNN)", g_machine.name(out, i), static_cast<int>(d.dtype), shape,
                                               PyByteArray_FromStringAndSize(static_cast<const char*>(p), static_cast<Py_ssize_t>(bytes)))
                               : nullptr;
        if (!item) {
            Py_DECREF(list);
            throw PythonError();
        }
        PyList_SET_ITEM(list, i, item);
    }
    return list;
}

// vm_outputs(outputs) -> the list above or None
PyObject* vm_outputs(PyObject*, PyObject* o) {
    return guarded([&]() -> PyObject* {
        PyObject* list = host_copies(reinterpret_cast<const chxvm_outputs*>(integer(o)));
        if (!list) Py_RETURN_NONE;
        return list;
    });
}

// vm_run(program, {name: tensor}, trace level) -> (code of the runtime, address of the outputs or 0, the list above or
// None); with a list the outputs are gone already
PyObject* vm_run(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need(n, 3);
        chxvm_program* program = reinterpret_cast<chxvm_program*>(integer(a[0]));
        if (!PyDict_Check(a[1])) fail(PyExc_TypeError, "a dict of tensors is expected");
        const int32_t trace = static_cast<int32_t>(integer(a[2]));
        c10::SmallVector<std::string, 4> keys;
        c10::SmallVector<const char*, 4> names;
        c10::SmallVector<chx_hip_tensor, 4> descs;
        Py_ssize_t at = 0;
        PyObject *key, *value;
        while (PyDict_Next(a[1], &at, &key, &value)) {
            const char* name = PyUnicode_AsUTF8(key);
            if (!name) throw PythonError();
            keys.emplace_back(name);
            descs.emplace_back();
            describe(tensor(value), &descs.back());
        }
        for (const std::string& k : keys) names.push_back(k.c_str());
        chxvm_outputs* out = nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = g_machine.run(program, names.data(), descs.data(), static_cast<int32_t>(names.size()), trace, &out);
        Py_END_ALLOW_THREADS
        if (rc != 0) return Py_BuildValue("(iiO)", rc, 0, Py_None);
        PyObject* list = host_copies(out);
        if (!list) return Py_BuildValue("(iLO)", 0, static_cast<long long>(reinterpret_cast<intptr_t>(out)), Py_None);
        Py_BEGIN_ALLOW_THREADS
        g_machine.destroy(out);
        Py_END_ALLOW_THREADS
        return Py_BuildValue("(iiN)", 0, 0, list);
    });
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
        {"init", init, METH_O, nullptr},
        {"quantize_linear", fast(quantize_linear), METH_FASTCALL, nullptr},
        {"dequantize_linear", fast(dequantize_linear), METH_FASTCALL, nullptr},
        {"elementwise", fast(elementwise), METH_FASTCALL, nullptr},
        {"qlinear_conv", fast(qlinear_conv), METH_FASTCALL, nullptr},
        {"conv_integer", fast(conv_integer), METH_FASTCALL, nullptr},
        {"matmul_integer", fast(matmul_integer), METH_FASTCALL, nullptr},
        {"qlinear_matmul", fast(qlinear_matmul), METH_FASTCALL, nullptr},
        {"plan_run", fast(plan_run), METH_FASTCALL, nullptr},
        {"vm_init", fast(vm_init), METH_FASTCALL, nullptr},
        {"vm_run", fast(vm_run), METH_FASTCALL, nullptr},
        {"vm_outputs", vm_outputs, METH_O, nullptr},
        {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_chx_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__chx_torch_ops(void) {
    return PyModule_Create(&module);
}
