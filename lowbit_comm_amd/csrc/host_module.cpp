// Host side of the codec's entry points as a Python extension module (lowbit_comm_amd._host): what a call costs before
// its kernel starts.
//
// A 64 KiB tensor's quantize kernel runs 2 us and a launch costs the host another 2 to 3 us, so for small buckets the
// Python around a launch is most of the time.  Launch is one call of the C ABI (include/lbc.h) with its arguments
// converted once: calling it looks up torch's current stream and enqueues the kernel, 1.4 us less than the same call
// through ctypes, whose sixteen argument conversions were paid for at every launch (four 1 MiB bf16 buckets through the
// pipelined hook 74.6 -> 66.6 us, a ring of fourteen hops 142 -> 134 us).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>

#include <cstring>
#include <memory>
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
    {"lbc_ring_step", make_call<&lbc_ring_step>},
    {"lbc_ef_update", make_call<&lbc_ef_update>},
    {"lbc_wire_quant_pack", make_call<&lbc_wire_quant_pack>},
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
    PyObject *given = PyTuple_GET_SIZE(args) > 0 ? PyTuple_GET_ITEM(args, 0) : nullptr;
    if (given == nullptr && kwargs != nullptr) given = PyDict_GetItemString(kwargs, "stream");
    if (launch->call == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "the launch was not bound");
        return nullptr;
    }
    if (given == nullptr || given == Py_None)
        return answer(enqueue(static_cast<c10::DeviceIndex>(launch->device), [&](void *stream) { return launch->call->run(stream); }));
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

PyObject *abi_version(PyObject *, PyObject *) { return PyLong_FromLong(lbc_abi_version() == LBC_ABI_VERSION ? LBC_ABI_VERSION : -1); }

PyMethodDef kMethods[] = {
    {"abi_version", abi_version, METH_NOARGS, "ABI version of include/lbc.h this module was built with, -1 when the library has another."},
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
    PyObject *module = PyModule_Create(&kModule);
    if (module == nullptr) return nullptr;
    Py_INCREF(&LaunchType);
    if (PyModule_AddObject(module, "Launch", reinterpret_cast<PyObject *>(&LaunchType)) < 0) {
        Py_DECREF(&LaunchType);
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
