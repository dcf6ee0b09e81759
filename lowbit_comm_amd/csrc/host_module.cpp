// Host side of the codec's entry points as a Python extension module (lowbit_comm_amd._host): what a call costs before
// its kernel starts.
//
// A 64 KiB tensor's quantize kernel runs 2 us and a launch costs the host another 2 to 3 us, so for small buckets the
// Python around a launch is most of the time: validating tensors, marshalling sixteen arguments, allocating the payload.
// Here that is one C call.  Two things live in this module:
//
//   Launch       one call of the C ABI (include/lbc.h) with its arguments converted once; calling it looks up torch's
//                current stream and enqueues the kernel, 1.4 us less than the same call through ctypes (four 1 MiB bf16
//                buckets through the pipelined hook 74.6 -> 66.6 us; a ring of fourteen hops gains less than its runs differ)
//   functions    the codec facade's allocating calls, from tensors to the launch (quantize and decode of a 10,007-element tensor
//                38.1 -> 11.2 us together, of 25 MiB fp32 23.2 -> 15.3, which is what the two kernels take)
//
// A function returns what the Python entry point returns (a tensor, or False for a valid request without a kernel), and
// None when the operands are not what its one combined test expects: the caller then takes the validating Python path,
// which names what is wrong.  Nothing is kept from one call to the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/core/Generator.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <memory>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/lbc.h"

namespace {

// ---- Launch: a call of the C ABI with its arguments bound -----------------------------------------------------------
struct Call {
    virtual int run(void *stream) = 0;
    virtual ~Call() = default;
    std::vector<std::vector<char>> held;   // arrays the arguments point to
};

bool convert(PyObject *o, Call &, int64_t &v) { v = PyLong_AsLongLong(o); return !PyErr_Occurred(); }
bool convert(PyObject *o, Call &, uint64_t &v) { v = PyLong_AsUnsignedLongLongMask(o); return !PyErr_Occurred(); }
bool convert(PyObject *o, Call &, float &v) { v = static_cast<float>(PyFloat_AsDouble(o)); return !PyErr_Occurred(); }
bool convert(PyObject *o, Call &, int &v) {
    const long long wide = PyLong_AsLongLong(o);
    v = static_cast<int>(wide);
    return !PyErr_Occurred();
}
// An address or None for null; for an array of addresses also an object that exports it as a buffer (a ctypes array), of
// which the launch keeps a copy.
template <typename P> bool convert(PyObject *o, Call &call, P *&v) {
    if (o == Py_None) {
        v = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        v = reinterpret_cast<P *>(PyLong_AsVoidPtr(o));
        return !PyErr_Occurred();
    }
    if (!std::is_pointer<P>::value) {
        PyErr_Format(PyExc_TypeError, "an address or None is wanted, not %s", Py_TYPE(o)->tp_name);
        return false;
    }
    Py_buffer view;
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return false;
    const char *bytes = static_cast<const char *>(view.buf);
    call.held.emplace_back(bytes, bytes + view.len);
    PyBuffer_Release(&view);
    v = reinterpret_cast<P *>(call.held.back().data());
    return true;
}

template <typename Fn> struct Bound;
template <typename... A> struct Bound<int (*)(A...)> : Call {
    using Fn = int (*)(A...);
    static constexpr size_t kGiven = sizeof...(A) - 1;   // all but the stream, which comes with the call
    Fn fn;
    std::tuple<A...> values;

    explicit Bound(Fn f) : fn(f) {}
    template <size_t... I> bool fill(PyObject *args, std::index_sequence<I...>) {
        return (convert(PyTuple_GET_ITEM(args, I), *this, std::get<I>(values)) && ...);
    }
    int run(void *stream) override {
        auto now = values;
        std::get<kGiven>(now) = stream;
        return std::apply(fn, now);
    }
    static std::unique_ptr<Call> make(Fn f, PyObject *args) {
        if (PyTuple_GET_SIZE(args) != static_cast<Py_ssize_t>(kGiven)) {
            PyErr_Format(PyExc_TypeError, "expected %zu arguments, got %zd", kGiven, PyTuple_GET_SIZE(args));
            return nullptr;
        }
        auto bound = std::make_unique<Bound>(f);
        if (!bound->fill(args, std::make_index_sequence<kGiven>{})) return nullptr;
        return bound;
    }
};

template <auto Fn> std::unique_ptr<Call> make_call(PyObject *args) { return Bound<decltype(Fn)>::make(Fn, args); }

struct Entry {
    const char *name;
    std::unique_ptr<Call> (*make)(PyObject *args);
};
constexpr Entry kEntries[] = {
    {"lbc_quant_pack", make_call<&lbc_quant_pack>},
    {"lbc_quant_pack_chunks", make_call<&lbc_quant_pack_chunks>},
    {"lbc_dequant", make_call<&lbc_dequant>},
    {"lbc_dequant_chunks", make_call<&lbc_dequant_chunks>},
    {"lbc_dequant_reduce", make_call<&lbc_dequant_reduce>},
    {"lbc_quant_pack_chunks_and_dequant_reduce", make_call<&lbc_quant_pack_chunks_and_dequant_reduce>},
    {"lbc_dequant_reduce_quant", make_call<&lbc_dequant_reduce_quant>},
    {"lbc_bucket_pipeline_step", make_call<&lbc_bucket_pipeline_step>},
    {"lbc_bucket_pipeline_step_any", make_call<&lbc_bucket_pipeline_step_any>},
    {"lbc_ring_step", make_call<&lbc_ring_step>},
    {"lbc_ring_relay", make_call<&lbc_ring_relay>},
    {"lbc_ef_update", make_call<&lbc_ef_update>},
    {"lbc_wire_quant_pack", make_call<&lbc_wire_quant_pack>},
    {"lbc_wire_compensate_quant_pack", make_call<&lbc_wire_compensate_quant_pack>},
    {"lbc_wire_quant_pack_chunks", make_call<&lbc_wire_quant_pack_chunks>},
    {"lbc_wire_dequant", make_call<&lbc_wire_dequant>},
    {"lbc_wire_dequant_chunks", make_call<&lbc_wire_dequant_chunks>},
    {"lbc_wire_dequant_reduce", make_call<&lbc_wire_dequant_reduce>},
    {"lbc_wire_ring_step", make_call<&lbc_wire_ring_step>},
    {"lbc_wire_quant_general", make_call<&lbc_wire_quant_general>},
    {"lbc_wire_dequant_general", make_call<&lbc_wire_dequant_general>},
};

// LBC_OK -> True, LBC_UNSUPPORTED -> False, anything else raises with the library's text.
PyObject *answer(int rc) {
    if (rc == LBC_OK) Py_RETURN_TRUE;
    if (rc == LBC_UNSUPPORTED) Py_RETURN_FALSE;
    const char *text = lbc_last_error();
    if (text != nullptr && *text != '\0') PyErr_SetString(PyExc_RuntimeError, text);
    else PyErr_Format(PyExc_RuntimeError, "lbc call failed with code %d", rc);
    return nullptr;
}

// Runs `call(stream)` on torch's current stream of `device`, with that device current and the interpreter released (a
// launch waits when the device's queue is full).
template <typename F> int enqueue(c10::DeviceIndex device, F &&call) {
    c10::OptionalDeviceGuard guard;
    if (device != c10::hip::current_device()) guard.reset_device(c10::Device(c10::DeviceType::CUDA, device));
    void *stream = c10::hip::getCurrentHIPStream(device).stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call(stream);
    Py_END_ALLOW_THREADS
    return rc;
}

struct Launch {
    PyObject_HEAD
    Call *call;
    int device;
};

int launch_init(PyObject *self, PyObject *args, PyObject *) {
    const char *name;
    PyObject *values;
    int device;
    if (!PyArg_ParseTuple(args, "sO!i", &name, &PyTuple_Type, &values, &device)) return -1;
    for (const Entry &entry : kEntries) {
        if (std::strcmp(entry.name, name) != 0) continue;
        std::unique_ptr<Call> call = entry.make(values);
        if (!call) return -1;
        Launch *launch = reinterpret_cast<Launch *>(self);
        delete launch->call;
        launch->call = call.release();
        launch->device = device;
        return 0;
    }
    PyErr_Format(PyExc_ValueError, "no entry point named %s", name);
    return -1;
}

PyObject *launch_call(PyObject *self, PyObject *args, PyObject *kwargs) {
    HANDLE_TH_ERRORS
    Launch *launch = reinterpret_cast<Launch *>(self);
    PyObject *given = nullptr;
    if (kwargs == nullptr && PyTuple_GET_SIZE(args) == 1) {   // the usual calls: a stream, or nothing
        given = PyTuple_GET_ITEM(args, 0);
    } else if (kwargs != nullptr || PyTuple_GET_SIZE(args) != 0) {
        static const char *const kNames[] = {"stream", nullptr};
        if (!PyArg_ParseTupleAndKeywords(args, kwargs, "|O:Launch", const_cast<char **>(kNames), &given)) return nullptr;
    }
    if (launch->call == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "the launch was not bound");
        return nullptr;
    }
    if (given == nullptr || given == Py_None)
        return answer(enqueue(static_cast<c10::DeviceIndex>(launch->device), [&](void *stream) { return launch->call->run(stream); }));
    if (!PyLong_Check(given)) {
        PyErr_Format(PyExc_TypeError, "stream must be a stream handle or None, not %s", Py_TYPE(given)->tp_name);
        return nullptr;
    }
    void *stream = PyLong_AsVoidPtr(given);
    if (PyErr_Occurred()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = launch->call->run(stream);
    Py_END_ALLOW_THREADS
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

void launch_dealloc(PyObject *self) {
    delete reinterpret_cast<Launch *>(self)->call;
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject LaunchType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- tensors ----------------------------------------------------------------------------------------------------
int code_of(at::ScalarType type) {
    switch (type) {
        case at::kFloat: return LBC_F32;
        case at::kHalf: return LBC_F16;
        case at::kBFloat16: return LBC_BF16;
        default: return LBC_NONE;
    }
}
at::ScalarType type_of(long code) { return code == LBC_F32 ? at::kFloat : (code == LBC_F16 ? at::kHalf : at::kBFloat16); }

// The tensor behind `o` when it is a contiguous GPU tensor that holds its values as they are (no lazy negation), else null.
const at::Tensor *gpu_tensor(PyObject *o) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous() && !t.is_neg() ? &t : nullptr;
}
const at::Tensor *payload_tensor(PyObject *o) {
    const at::Tensor *t = gpu_tensor(o);
    return t != nullptr && t->scalar_type() == at::kByte ? t : nullptr;
}
// Does autograd follow what is computed from `t`, backward or forward?
bool watched(const at::Tensor &t) { return t.requires_grad() || t._fw_grad(/*level=*/0).defined(); }
bool with(const at::Tensor &t, const at::Tensor &like) { return t.get_device() == like.get_device(); }

at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor &like) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

struct Policy {
    long group, topk, stochastic, bit, quant_type;
};
bool integer(PyObject *o, long &v) {
    v = PyLong_Check(o) ? PyLong_AsLong(o) : (o == Py_True ? 1 : (o == Py_False ? 0 : -1000));
    return v != -1000 && !(v == -1 && PyErr_Occurred());
}
bool valid_group(long g) { return g == 16 || g == 32 || g == 64; }
// what the portable format serves: linear 8-bit codes, no outliers, no noise
bool portable(const Policy &p) { return valid_group(p.group) && p.topk == 0 && p.stochastic == 0 && p.bit == 8 && p.quant_type == LBC_QUANT_LINEAR; }
int64_t groups_of(int64_t numel, long g) { return (numel + g - 1) / g; }

// An operand that the combined test does not expect, or a Python error set by a conversion.
PyObject *elsewhere() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

// The calls below stand for public methods of a codec module, which a subclass, a patched class or an instance may have
// replaced.  Their first two arguments are the module and a table (name, attribute, name, attribute, ...) of the methods
// that the call by-passes: it is made only when the module's class has exactly these attributes and the module itself holds
// none of them.  (Here, because the same test in Python costs a small call 0.1 us.)
bool owns(PyObject *module, PyObject *table) {
    if (!PyTuple_Check(table)) return false;
    PyObject **held = _PyObject_GetDictPtr(module);
    for (Py_ssize_t i = 0; i + 1 < PyTuple_GET_SIZE(table); i += 2) {
        PyObject *name = PyTuple_GET_ITEM(table, i);
        if (_PyType_Lookup(Py_TYPE(module), name) != PyTuple_GET_ITEM(table, i + 1)) return false;
        if (held != nullptr && *held != nullptr && PyDict_GetItemWithError(*held, name) != nullptr) return false;
    }
    return !PyErr_Occurred();
}

// ---- the portable format ---------------------------------------------------------------------------------------
// quantize(module, table, input, group_size, topk, stochastic, bit, quant_type, access) -> payload
PyObject *quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p;
    long access;
    if (n != 7 || !integer(a[1], p.group) || !integer(a[2], p.topk) || !integer(a[3], p.stochastic) || !integer(a[4], p.bit) ||
        !integer(a[5], p.quant_type) || !integer(a[6], access))
        return elsewhere();
    const at::Tensor *x = gpu_tensor(a[0]);
    if (x == nullptr || x->numel() == 0 || !portable(p)) return elsewhere();
    const int type = code_of(x->scalar_type());
    if (type == LBC_NONE) return elsewhere();
    const int64_t numel = x->numel(), groups = groups_of(numel, p.group), code_bytes = groups * p.group;
    at::Tensor payload = fresh({code_bytes + 4 * groups}, at::kByte, *x);
    uint8_t *base = static_cast<uint8_t *>(payload.data_ptr());
    const void *data = x->data_ptr();
    const int rc = enqueue(x->get_device(), [&](void *stream) {
        return lbc_quant_pack(data, type, nullptr, LBC_NONE, numel, static_cast<int>(p.group), reinterpret_cast<int8_t *>(base),
                              reinterpret_cast<float *>(base + code_bytes), nullptr, LBC_NONE, nullptr, LBC_F32, nullptr, LBC_NONE,
                              static_cast<int>(access), stream);
    });
    if (rc == LBC_OK) return THPVariable_Wrap(std::move(payload));
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// _host.FLAT: the shape of everything that a payload holds, in one dimension.  An object of its own, because None and the
// like are shapes that a caller may get wrong.
PyObject *flat = nullptr;

// The sizes of the tensor to make: `o` is a tuple of them, or FLAT for one dimension of `all` elements.  False: neither.
bool sizes_of(PyObject *o, int64_t all, c10::SmallVector<int64_t, 5> &sizes, int64_t &numel) {
    numel = 1;
    if (o == flat) {
        sizes.push_back(all);
        numel = all;
        return true;
    }
    if (!PyTuple_Check(o)) return false;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(o); ++i) {
        long v;
        if (PyBool_Check(PyTuple_GET_ITEM(o, i)) || !integer(PyTuple_GET_ITEM(o, i), v) || v < 0) return false;
        sizes.push_back(v);
        if (__builtin_mul_overflow(numel, v, &numel)) return false;
    }
    return true;
}

// dequantize(module, table, payload, shape, dtype, group_size, topk, bit, reduce_op, quant_type, access) -> tensor of that
// shape (FLAT: every element the payload holds)
PyObject *dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p{};
    long dtype, op, access;
    if (n != 9 || !integer(a[2], dtype) || !integer(a[3], p.group) || !integer(a[4], p.topk) || !integer(a[5], p.bit) ||
        !integer(a[6], op) || !integer(a[7], p.quant_type) || !integer(a[8], access))
        return elsewhere();
    const at::Tensor *payload = payload_tensor(a[0]);
    if (payload == nullptr || !portable(p) || op != LBC_REDUCE_NONE || dtype < LBC_F32 || dtype > LBC_BF16) return elsewhere();
    const int64_t nbytes = payload->numel(), per_group = p.group + 4, padded = nbytes / per_group * p.group;
    c10::SmallVector<int64_t, 5> sizes;
    int64_t numel;
    if (nbytes % per_group != 0 || !sizes_of(a[1], padded, sizes, numel) || numel == 0 ||
        groups_of(numel, p.group) * p.group != padded)
        return elsewhere();
    at::Tensor out = fresh(sizes, type_of(dtype), *payload);
    const uint8_t *base = static_cast<const uint8_t *>(payload->data_ptr());
    void *data = out.data_ptr();
    const int rc = enqueue(payload->get_device(), [&](void *stream) {
        return lbc_dequant(reinterpret_cast<const int8_t *>(base), reinterpret_cast<const float *>(base + padded), numel,
                           static_cast<int>(p.group), data, static_cast<int>(dtype), LBC_REDUCE_NONE, static_cast<int>(access), stream);
    });
    if (rc == LBC_OK) return THPVariable_Wrap(std::move(out));
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// The payload tensors of a list or tuple, each of `nbytes` bytes (-1: as many as the first) on one device; 0 when it is
// anything else.
int payloads_of(PyObject *list, int64_t &nbytes, const uint8_t **pointers, const at::Tensor *&first) {
    PyObject **items;
    Py_ssize_t count;
    if (PyList_Check(list)) {
        items = reinterpret_cast<PyListObject *>(list)->ob_item;
        count = PyList_GET_SIZE(list);
    } else if (PyTuple_Check(list)) {
        items = reinterpret_cast<PyTupleObject *>(list)->ob_item;
        count = PyTuple_GET_SIZE(list);
    } else {
        return 0;
    }
    if (count < 1 || count > LBC_MAX_PAYLOADS) return 0;
    for (Py_ssize_t i = 0; i < count; ++i) {
        const at::Tensor *t = payload_tensor(items[i]);
        if (t == nullptr) return 0;
        if (i == 0) {
            first = t;
            if (nbytes < 0) nbytes = t->numel();
        }
        if (t->numel() != nbytes || !with(*t, *first)) return 0;
        pointers[i] = static_cast<const uint8_t *>(t->data_ptr());
    }
    return static_cast<int>(count);
}

// dequantize_reduce(module, table, payloads, shape, dtype, group_size, topk, bit, quant_type, divisor, access) -> tensor, as dequantize
PyObject *dequantize_reduce(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p{};
    long dtype, access;
    if (n != 9 || !integer(a[2], dtype) || !integer(a[3], p.group) || !integer(a[4], p.topk) || !integer(a[5], p.bit) ||
        !integer(a[6], p.quant_type) || !integer(a[8], access))
        return elsewhere();
    const double divisor = PyFloat_AsDouble(a[7]);
    if (!portable(p) || dtype < LBC_F32 || dtype > LBC_BF16 || !(divisor > 0.0)) return elsewhere();
    int64_t nbytes = -1, numel;
    const uint8_t *bases[LBC_MAX_PAYLOADS];
    const at::Tensor *first = nullptr;
    const int world = payloads_of(a[0], nbytes, bases, first);
    const int64_t per_group = p.group + 4;
    if (world == 0 || nbytes % per_group != 0) return elsewhere();
    const int64_t padded = nbytes / per_group * p.group;
    c10::SmallVector<int64_t, 5> sizes;
    if (!sizes_of(a[1], padded, sizes, numel) || numel == 0 || groups_of(numel, p.group) * p.group != padded) return elsewhere();
    const int8_t *codes[LBC_MAX_PAYLOADS];
    const float *scales[LBC_MAX_PAYLOADS];
    for (int r = 0; r < world; ++r) {
        codes[r] = reinterpret_cast<const int8_t *>(bases[r]);
        scales[r] = reinterpret_cast<const float *>(bases[r] + padded);
    }
    at::Tensor out = fresh(sizes, type_of(dtype), *first);
    void *data = out.data_ptr();
    const int rc = enqueue(first->get_device(), [&](void *stream) {
        return lbc_dequant_reduce(codes, scales, world, numel, static_cast<int>(p.group), static_cast<float>(divisor), data,
                                  static_cast<int>(dtype), nullptr, nullptr, static_cast<int>(access), stream);
    });
    if (rc == LBC_OK) return THPVariable_Wrap(std::move(out));
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// ---- the CUDA extension's format ---------------------------------------------------------------------------------
bool cuda_policy(const Policy &p) {
    return valid_group(p.group) && p.topk >= 0 && p.topk <= 2 && (p.bit == 8 || p.bit == 4) && p.quant_type >= LBC_QUANT_LINEAR &&
           p.quant_type <= LBC_QUANT_E2M1 && (p.quant_type == LBC_QUANT_LINEAR || p.bit == 4);
}
bool plain(const Policy &p) { return p.topk == 0 && p.stochastic == 0 && p.quant_type == LBC_QUANT_LINEAR; }
// bytes of a group: codes, the scale in the tensor's type, with outliers the index word and the outliers themselves
int64_t cuda_group_bytes(const Policy &p, int type) {
    return p.group * p.bit / 8 + (type == LBC_F32 ? 4 : 2) * (p.topk == 0 ? 1 : p.topk + 2);
}

// (seed, offset) of the device's default generator, advanced past `increment` draws rounded up to a multiple of four, as
// HipCudaWireModule.philox_engine_inputs does it.
std::pair<uint64_t, uint64_t> philox_inputs(const at::Tensor &x, uint64_t increment) {
    at::Generator generator = at::globalContext().defaultGenerator(x.device());
    std::lock_guard<std::mutex> lock(generator.mutex());
    const uint64_t offset = generator.get_offset();
    generator.set_offset(offset + (increment + 3) / 4 * 4);
    return {generator.current_seed(), offset};
}

// wire_quantize(module, table, input, output or None, group_size, topk, stochastic, bit, quant_type, compact, access) -> payload
PyObject *wire_quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p;
    long compact, access;
    if (n != 9 || !integer(a[2], p.group) || !integer(a[3], p.topk) || !integer(a[4], p.stochastic) || !integer(a[5], p.bit) ||
        !integer(a[6], p.quant_type) || !integer(a[7], compact) || !integer(a[8], access))
        return elsewhere();
    const at::Tensor *x = gpu_tensor(a[0]);
    if (x == nullptr || x->numel() == 0 || !cuda_policy(p)) return elsewhere();
    const int type = code_of(x->scalar_type());
    const int64_t numel = x->numel();
    if (type == LBC_NONE || (!plain(p) && numel % p.group != 0)) return elsewhere();
    const int64_t nbytes = groups_of(numel, p.group) * cuda_group_bytes(p, type);
    at::Tensor payload;
    if (a[1] == Py_None) {
        payload = fresh({nbytes}, at::kByte, *x);
    } else {
        const at::Tensor *given = payload_tensor(a[1]);
        if (given == nullptr || given->numel() != nbytes || !with(*given, *x)) return elsewhere();
        payload = *given;
    }
    uint8_t *base = static_cast<uint8_t *>(payload.data_ptr());
    const void *data = x->data_ptr();
    const int g = static_cast<int>(p.group), bit = static_cast<int>(p.bit), inside = compact != 0;
    std::pair<uint64_t, uint64_t> stream_position{0, 0};
    if (p.stochastic) stream_position = philox_inputs(*x, static_cast<uint64_t>(numel));
    const int rc = enqueue(x->get_device(), [&](void *stream) {
        if (plain(p)) return lbc_wire_quant_pack(data, nullptr, type, numel, g, bit, inside, base, static_cast<int>(access), stream);
        return lbc_wire_quant_general(data, type, numel, g, bit, static_cast<int>(p.quant_type), static_cast<int>(p.topk), p.stochastic != 0,
                                      stream_position.first, stream_position.second, inside, base, stream);
    });
    if (rc == LBC_OK) return THPVariable_Wrap(std::move(payload));
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// wire_compensate_quantize(module, table, x, residual, group_size, topk, stochastic, bit, quant_type, compact, access) -> (x + residual, its
// payload), both from one launch.  Plain codes; operands of one type, one shape and one device that autograd does not watch.
PyObject *wire_compensate_quantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p;
    long compact, access;
    if (n != 9 || !integer(a[2], p.group) || !integer(a[3], p.topk) || !integer(a[4], p.stochastic) || !integer(a[5], p.bit) ||
        !integer(a[6], p.quant_type) || !integer(a[7], compact) || !integer(a[8], access))
        return elsewhere();
    if (!THPVariable_CheckExact(a[0]) || !THPVariable_CheckExact(a[1])) return elsewhere();
    const at::Tensor *x = gpu_tensor(a[0]), *r = gpu_tensor(a[1]);
    if (x == nullptr || r == nullptr || x->numel() == 0 || !cuda_policy(p) || !plain(p)) return elsewhere();
    const int type = code_of(x->scalar_type());
    if (type == LBC_NONE || r->scalar_type() != x->scalar_type() || !x->sizes().equals(r->sizes()) || !with(*r, *x) ||
        watched(*x) || watched(*r))
        return elsewhere();
    const int64_t numel = x->numel();
    at::Tensor prepared = fresh(x->sizes(), x->scalar_type(), *x);
    at::Tensor payload = fresh({groups_of(numel, p.group) * cuda_group_bytes(p, type)}, at::kByte, *x);
    const void *data = x->data_ptr(), *residual = r->data_ptr();
    void *sum = prepared.data_ptr();
    uint8_t *base = static_cast<uint8_t *>(payload.data_ptr());
    const int rc = enqueue(x->get_device(), [&](void *stream) {
        return lbc_wire_compensate_quant_pack(data, residual, sum, type, numel, static_cast<int>(p.group), static_cast<int>(p.bit),
                                              compact != 0, base, static_cast<int>(access), stream);
    });
    if (rc != LBC_OK) return answer(rc);
    PyObject *pair = PyTuple_New(2);
    if (pair == nullptr) return nullptr;
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(prepared)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(payload)));
    return pair;
    END_HANDLE_TH_ERRORS
}

// wire_dequantize(module, table, payload, shape, dtype, group_size, topk, bit, reduce_op, quant_type, compact, access) -> tensor of that
// shape (FLAT: every element the payload holds)
PyObject *wire_dequantize(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 2 || !owns(a[0], a[1])) return elsewhere();
    a += 2;
    n -= 2;
    Policy p{};
    long dtype, op, compact, access;
    if (n != 10 || !integer(a[2], dtype) || !integer(a[3], p.group) || !integer(a[4], p.topk) || !integer(a[5], p.bit) ||
        !integer(a[6], op) || !integer(a[7], p.quant_type) || !integer(a[8], compact) || !integer(a[9], access))
        return elsewhere();
    const at::Tensor *payload = payload_tensor(a[0]);
    if (payload == nullptr || !cuda_policy(p) || op != LBC_REDUCE_NONE || dtype < LBC_F32 || dtype > LBC_BF16) return elsewhere();
    const int type = static_cast<int>(dtype);
    const int64_t nbytes = payload->numel(), per_group = cuda_group_bytes(p, type), padded = nbytes / per_group * p.group;
    c10::SmallVector<int64_t, 5> sizes;
    int64_t numel;
    if (nbytes % per_group != 0 || !sizes_of(a[1], padded, sizes, numel) || numel == 0 ||
        groups_of(numel, p.group) * p.group != padded || (!plain(p) && numel % p.group != 0))
        return elsewhere();
    at::Tensor out = fresh(sizes, type_of(dtype), *payload);
    const uint8_t *base = static_cast<const uint8_t *>(payload->data_ptr());
    void *data = out.data_ptr();
    const int g = static_cast<int>(p.group), bit = static_cast<int>(p.bit), inside = compact != 0;
    const int rc = enqueue(payload->get_device(), [&](void *stream) {
        if (plain(p)) return lbc_wire_dequant(base, numel, g, bit, inside, data, type, LBC_REDUCE_NONE, static_cast<int>(access), stream);
        return lbc_wire_dequant_general(base, numel, g, bit, static_cast<int>(p.quant_type), static_cast<int>(p.topk), inside, data, type,
                                        LBC_REDUCE_NONE, stream);
    });
    if (rc == LBC_OK) return THPVariable_Wrap(std::move(out));
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// wire_reduce(payloads, out, prepared or None, residual or None, group_size, topk, bit, quant_type, compact, divisor,
// fused multiply-add, access) -> True: out = sum or mean, and with prepared the residual update.  What the extension's
// fused reduce takes: group 64, plain 8-bit codes, whole groups of outputs.
PyObject *wire_reduce(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Policy p{};
    long compact, fma, access;
    if (n != 12 || !integer(a[4], p.group) || !integer(a[5], p.topk) || !integer(a[6], p.bit) || !integer(a[7], p.quant_type) ||
        !integer(a[8], compact) || !integer(a[10], fma) || !integer(a[11], access))
        return elsewhere();
    const double divisor = PyFloat_AsDouble(a[9]);   // the library refuses one whose reciprocal is not positive
    if (divisor == -1.0 && PyErr_Occurred()) return nullptr;
    const at::Tensor *out = gpu_tensor(a[1]);
    if (out == nullptr || !plain(p) || p.group != 64 || p.bit != 8) return elsewhere();
    const int type = code_of(out->scalar_type());
    if (type == LBC_NONE || out->numel() == 0 || out->numel() % 64 != 0) return elsewhere();
    int64_t nbytes = out->numel() / 64 * cuda_group_bytes(p, type), numel = out->numel();
    const uint8_t *bases[LBC_MAX_PAYLOADS];
    const at::Tensor *first = nullptr;
    const int world = payloads_of(a[0], nbytes, bases, first);
    if (world == 0 || !with(*first, *out) || (a[2] == Py_None) != (a[3] == Py_None)) return elsewhere();
    const void *prepared = nullptr;
    void *residual = nullptr;
    if (a[2] != Py_None) {
        const at::Tensor *before = gpu_tensor(a[2]), *after = gpu_tensor(a[3]);
        if (before == nullptr || after == nullptr || before->scalar_type() != out->scalar_type() ||
            after->scalar_type() != out->scalar_type() || !with(*before, *out) || !with(*after, *out) ||
            before->numel() != after->numel() || groups_of(before->numel(), 64) * 64 != out->numel())
            return elsewhere();
        prepared = before->data_ptr();
        residual = after->data_ptr();
        numel = before->numel();
    }
    void *data = out->data_ptr();
    const float inverse = 1.0f / static_cast<float>(divisor);
    return answer(enqueue(out->get_device(), [&](void *stream) {
        return lbc_wire_dequant_reduce(bases, world, numel, 64, compact != 0, inverse, fma != 0, data, type, prepared, residual,
                                       static_cast<int>(access), stream);
    }));
    END_HANDLE_TH_ERRORS
}

// specs(objects...) -> (address, type, elements, ...) of every tensor, flattened, None as 0 and a list or tuple as its
// tensors behind their count; None when one of them is not a contiguous GPU tensor.  What a bound launch depends on.
bool append_spec(PyObject *o, std::vector<int64_t> &out, bool nested) {
    if (o == Py_None) {
        out.push_back(0);
        return true;
    }
    if (const at::Tensor *t = gpu_tensor(o)) {
        out.push_back(static_cast<int64_t>(reinterpret_cast<intptr_t>(t->data_ptr())));
        out.push_back(static_cast<int64_t>(t->scalar_type()));
        out.push_back(t->numel());
        return true;
    }
    if (nested || !(PyList_Check(o) || PyTuple_Check(o))) return false;
    PyObject *fast = PySequence_Fast(o, "");
    if (fast == nullptr) return false;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(fast);
    bool fine = count >= 1 && count <= LBC_MAX_PAYLOADS;
    out.push_back(count);
    for (Py_ssize_t i = 0; fine && i < count; ++i) fine = append_spec(PySequence_Fast_GET_ITEM(fast, i), out, true) && out.back() != 0;
    Py_DECREF(fast);
    return fine;
}
PyObject *specs(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    std::vector<int64_t> values;
    values.reserve(40);
    for (Py_ssize_t i = 0; i < n; ++i)
        if (!append_spec(a[i], values, false)) return elsewhere();
    PyObject *tuple = PyTuple_New(static_cast<Py_ssize_t>(values.size()));
    if (tuple == nullptr) return nullptr;
    for (size_t i = 0; i < values.size(); ++i) {
        PyObject *v = PyLong_FromLongLong(values[i]);
        if (v == nullptr) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, static_cast<Py_ssize_t>(i), v);
    }
    return tuple;
    END_HANDLE_TH_ERRORS
}

// ---- the stages of the pipelined reduce-scatter ------------------------------------------------------------------
// What one step of the bucket pipeline launches, from the plans of its buckets: the arguments of the three stages come out of
// a plan's buffers and the step's tensors here, where binding them per tensor address and looking the bound launches and
// their merged launch up again took the interpreter 5 us a step (four 1 MiB bf16 buckets through the hook 66 -> 48 us).
struct Stages {   // a plan's buffers, as the stages address them
    PyObject_HEAD
    at::Tensor *rows;   // send, received, gathered; null until initialised
    int64_t numel, shard, stride, code_bytes;
    int world, rank, group, dtype;
};

int stages_init(PyObject *self, PyObject *args, PyObject *) {
    long long numel;
    int world, rank, group, dtype;
    PyObject *tensors[3];
    if (!PyArg_ParseTuple(args, "LiiiiOOO", &numel, &world, &rank, &group, &dtype, &tensors[0], &tensors[1], &tensors[2])) return -1;
    const bool sane = numel > 0 && world >= 1 && world <= LBC_MAX_PAYLOADS && rank >= 0 && rank < world && valid_group(group) &&
                      dtype >= LBC_F32 && dtype <= LBC_BF16;
    const int64_t shard = sane ? (numel + world - 1) / world : 0, groups = sane ? groups_of(shard, group) : 0;
    const at::Tensor *rows[3];
    bool fit = sane;
    for (int i = 0; fit && i < 3; ++i) {
        rows[i] = payload_tensor(tensors[i]);
        fit = rows[i] != nullptr && rows[i]->dim() == 2 && rows[i]->size(0) == world && rows[i]->size(1) >= groups * (group + 4) &&
              rows[i]->size(1) == rows[0]->size(1) && with(*rows[i], *rows[0]);
    }
    if (!fit) {
        PyErr_SetString(PyExc_ValueError, "the buffers do not belong to such a plan");
        return -1;
    }
    Stages *s = reinterpret_cast<Stages *>(self);
    delete[] s->rows;
    s->rows = new at::Tensor[3]{*rows[0], *rows[1], *rows[2]};
    s->numel = numel;
    s->shard = shard;
    s->stride = rows[0]->size(1);
    s->code_bytes = groups * group;
    s->world = world;
    s->rank = rank;
    s->group = group;
    s->dtype = dtype;
    return 0;
}

void stages_dealloc(PyObject *self) {
    delete[] reinterpret_cast<Stages *>(self)->rows;
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject StagesType = {PyVarObject_HEAD_INIT(nullptr, 0)};

const Stages *stages_of(PyObject *o) {
    const Stages *s = Py_TYPE(o) == &StagesType ? reinterpret_cast<const Stages *>(o) : nullptr;
    return s != nullptr && s->rows != nullptr ? s : nullptr;
}
uint8_t *row_of(const Stages &s, int which, int64_t row) { return static_cast<uint8_t *>(s.rows[which].data_ptr()) + row * s.stride; }

// pipeline_step(table, plan, stages, tensor, residual, plan, stages, mean, plan, stages, out, access, stream): quantize of `tensor`
// (with `residual`, updated in place, or None), reduce + requantize, decode into `out`; a stage whose plan is None is absent.
// `table` names the plan methods the call stands for.  One launch: True; no grid for this combination: False, nothing was launched.
PyObject *pipeline_step(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    long access;
    if (n != 13 || !integer(a[11], access)) return elsewhere();
    PyObject *const table = a[0];
    lbc_quant_chunks_stage quant{};
    lbc_reduce_quant_stage reduce{};
    lbc_dequant_chunks_stage decode{};
    const int8_t *codes[LBC_MAX_PAYLOADS];
    const float *scales[LBC_MAX_PAYLOADS];
    const Stages *first = nullptr;
    auto belongs = [&](PyObject *plan, const Stages *s) {
        if (s == nullptr || !owns(plan, table)) return false;
        if (first == nullptr) first = s;
        return s->group == first->group && s->dtype == first->dtype && with(s->rows[0], first->rows[0]);
    };
    const bool has_quant = a[1] != Py_None, has_reduce = a[5] != Py_None, has_decode = a[8] != Py_None;
    if (has_quant) {
        const Stages *s = stages_of(a[2]);
        const at::Tensor *x = gpu_tensor(a[3]);
        if (!belongs(a[1], s) || x == nullptr || x->numel() != s->numel || code_of(x->scalar_type()) != s->dtype || !with(*x, s->rows[0]))
            return elsewhere();
        quant = {x->data_ptr(), nullptr, row_of(*s, 0, 0), nullptr, s->numel, s->stride, s->dtype, LBC_NONE, LBC_NONE, s->world};
        if (a[4] != Py_None) {
            const at::Tensor *residual = gpu_tensor(a[4]);
            if (residual == nullptr || residual->numel() != s->numel || residual->scalar_type() != at::kFloat || !with(*residual, *x))
                return elsewhere();
            quant.residual = quant.new_residual = residual->data_ptr();
            quant.residual_dtype = quant.new_residual_dtype = LBC_F32;
        }
    }
    if (has_reduce) {
        const Stages *s = stages_of(a[6]);
        if (!belongs(a[5], s) || !PyBool_Check(a[7])) return elsewhere();
        for (int r = 0; r < s->world; ++r) {
            const uint8_t *row = row_of(*s, 1, r);
            codes[r] = reinterpret_cast<const int8_t *>(row);
            scales[r] = reinterpret_cast<const float *>(row + s->code_bytes);
        }
        uint8_t *mine = row_of(*s, 2, s->rank);
        reduce = {codes, scales, reinterpret_cast<int8_t *>(mine), reinterpret_cast<float *>(mine + s->code_bytes), s->shard,
                  a[7] == Py_True ? static_cast<float>(s->world) : 1.0f, s->world, s->dtype};
    }
    if (has_decode) {
        const Stages *s = stages_of(a[9]);
        const at::Tensor *out = gpu_tensor(a[10]);
        if (!belongs(a[8], s) || out == nullptr || out->numel() != s->numel || code_of(out->scalar_type()) != s->dtype ||
            !with(*out, s->rows[0]))
            return elsewhere();
        decode = {row_of(*s, 2, 0), out->data_ptr(), s->stride, s->shard, s->numel, s->world, s->dtype};
    }
    if (first == nullptr) return elsewhere();
    auto call = [&](void *stream) {
        return lbc_bucket_pipeline_step_any(has_quant ? &quant : nullptr, has_reduce ? &reduce : nullptr, has_decode ? &decode : nullptr,
                                            first->group, static_cast<int>(access), stream);
    };
    if (a[12] == Py_None) return answer(enqueue(first->rows[0].get_device(), call));
    if (!PyLong_Check(a[12])) return elsewhere();
    void *stream = PyLong_AsVoidPtr(a[12]);
    if (PyErr_Occurred()) return elsewhere();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call(stream);
    Py_END_ALLOW_THREADS
    return answer(rc);
    END_HANDLE_TH_ERRORS
}

// own(object, table) -> whether a native call may stand for the object's methods in the table.
PyObject *own(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n == 2 && owns(a[0], a[1])) Py_RETURN_TRUE;
    PyErr_Clear();
    Py_RETURN_FALSE;
}

PyObject *abi_version(PyObject *, PyObject *) { return PyLong_FromLong(lbc_abi_version() == LBC_ABI_VERSION ? LBC_ABI_VERSION : -1); }

PyMethodDef kMethods[] = {
    {"abi_version", abi_version, METH_NOARGS, "ABI version of include/lbc.h this module was built with, -1 when the library has another."},
    {"quantize", reinterpret_cast<PyCFunction>(quantize), METH_FASTCALL, "Quantize into a fresh portable payload."},
    {"dequantize", reinterpret_cast<PyCFunction>(dequantize), METH_FASTCALL, "Decode a portable payload into a fresh tensor."},
    {"dequantize_reduce", reinterpret_cast<PyCFunction>(dequantize_reduce), METH_FASTCALL, "Decode and reduce portable payloads into a fresh tensor."},
    {"wire_compensate_quantize", reinterpret_cast<PyCFunction>(wire_compensate_quantize), METH_FASTCALL, "x + residual and its payload in the CUDA extension's format."},
    {"wire_quantize", reinterpret_cast<PyCFunction>(wire_quantize), METH_FASTCALL, "Quantize into a payload of the CUDA extension's format."},
    {"wire_dequantize", reinterpret_cast<PyCFunction>(wire_dequantize), METH_FASTCALL, "Decode a payload of that format into a fresh tensor."},
    {"wire_reduce", reinterpret_cast<PyCFunction>(wire_reduce), METH_FASTCALL, "Fused reduce of payloads of that format, optionally with the residual update."},
    {"pipeline_step", reinterpret_cast<PyCFunction>(pipeline_step), METH_FASTCALL, "One launch for the ready stages of a bucket pipeline."},
    {"own", reinterpret_cast<PyCFunction>(own), METH_FASTCALL, "Are the methods in a table the module's own?"},
    {"specs", reinterpret_cast<PyCFunction>(specs), METH_FASTCALL, "Addresses, types and element counts of contiguous GPU tensors."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Native host side of the gfx950 codec's entry points.", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    LaunchType.tp_name = "lowbit_comm_amd._host.Launch";
    LaunchType.tp_basicsize = sizeof(Launch);
    LaunchType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
    LaunchType.tp_doc = "Launch(entry point, arguments, device index): one call of the C ABI; calling it enqueues the kernel.";
    LaunchType.tp_new = PyType_GenericNew;
    LaunchType.tp_init = launch_init;
    LaunchType.tp_call = launch_call;
    LaunchType.tp_dealloc = launch_dealloc;
    if (PyType_Ready(&LaunchType) < 0) return nullptr;
    StagesType.tp_name = "lowbit_comm_amd._host.Stages";
    StagesType.tp_basicsize = sizeof(Stages);
    StagesType.tp_flags = Py_TPFLAGS_DEFAULT;
    StagesType.tp_doc = "Stages(numel, world, rank, group, dtype code, send, received, gathered): a plan's buffers for pipeline_step.";
    StagesType.tp_new = PyType_GenericNew;
    StagesType.tp_init = stages_init;
    StagesType.tp_dealloc = stages_dealloc;
    if (PyType_Ready(&StagesType) < 0) return nullptr;
    PyObject *module = PyModule_Create(&kModule);
    if (module == nullptr) return nullptr;
    if (flat == nullptr) flat = PyUnicode_FromString("FLAT");
    Py_XINCREF(flat);
    if (flat == nullptr || PyModule_AddObject(module, "FLAT", flat) < 0) {
        Py_XDECREF(flat);
        Py_DECREF(module);
        return nullptr;
    }
    for (auto [name, type] : {std::make_pair("Launch", &LaunchType), std::make_pair("Stages", &StagesType)}) {
        Py_INCREF(type);
        if (PyModule_AddObject(module, name, reinterpret_cast<PyObject *>(type)) < 0) {
            Py_DECREF(type);
            Py_DECREF(module);
            return nullptr;
        }
    }
    return module;
}
