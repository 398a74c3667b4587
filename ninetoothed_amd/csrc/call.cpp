// The way of a repeated call from Python into the library.  A program whose kernels take a few microseconds is bound by
// its host: of the 5.9 us that a 512^3 product costs its caller, reading shapes, strides, types and devices through Python
// attributes took 2.3, converting the arguments for a C call 1.3.  Here a call's signature is read from the tensors
// themselves into a string of bytes, the dictionary that the kernel keeps gives what its first call has prepared -- entry
// point, layouts, constants -- and only the addresses and scalars of this call are filled in.
//
// Every call whose arguments are not ordinary strided tensors, numbers of the built-in types and integer keywords takes
// the way through Python (None is returned), and so does the first call of a signature and a linear program's whose operands that
// entry point does not take.  Any other result of the library is raised here: what it may have launched is not launched again.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "../../include/ninetoothed_hip.h"

namespace {

enum Kind { kMatmul, kAddmm, kLinear, kSoftmax, kAttention, kConv2d, kConv2dStrided, kMap };
const char *const kKinds[] = {"matmul", "addmm", "linear", "softmax", "attention", "conv2d", "conv2d_strided", "map"};

// An argument of the entry point: a tensor (the address of a call's argument plus an offset), a scalar that lies behind a
// pointer, or nothing (position -1).
struct Slot {
    enum What { kNull, kTensor, kFloat, kTruth } what = kNull;
    Py_ssize_t position = -1;
    int64_t offset = 0;
    std::vector<uint64_t> shape;
    std::vector<int64_t> strides;
};

struct MapLaunch {
    const NineToothedMapProgram *program;                      // of the plan, which outlives the recipe
    std::vector<Py_ssize_t> operands;                          // argument of each operand
    std::vector<std::pair<Py_ssize_t, Py_ssize_t>> scalars;    // (constant, argument)
};

struct Recipe {
    Kind kind;
    void *function;
    std::vector<Slot> slots;
    std::vector<int> ints;
    std::vector<double> doubles;  // linear: scale (unless it is an argument) and bound
    Py_ssize_t scale_position = -1;
    std::vector<MapLaunch> launches;
};

constexpr const char *kCapsule = "ninetoothed_amd.recipe";

// ---- signatures ------------------------------------------------------------------------------------

struct Key {
    char bytes[1024];
    size_t length = 0;
    bool fits = true;
    void put(const void *data, size_t size) {
        if (length + size > sizeof(bytes)) {
            fits = false;
            return;
        }
        std::memcpy(bytes + length, data, size);
        length += size;
    }
    template <typename T>
    void value(T v) {
        put(&v, sizeof(v));
    }
};

// an ordinary tensor: its own class, dense strides, sizes that are numbers, no transform around it
const at::TensorImpl *ordinary(PyObject *object) {
    if (!THPVariable_CheckExact(object)) return nullptr;
    const at::Tensor &tensor = THPVariable_Unpack(object);
    if (!tensor.defined()) return nullptr;
    const at::TensorImpl *impl = tensor.unsafeGetTensorImpl();
    if (impl->layout() != at::kStrided || impl->has_symbolic_sizes_strides() || impl->is_nested() || impl->is_python_dispatch() || !impl->has_storage()) return nullptr;
    constexpr c10::DispatchKeySet transforms({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched, c10::DispatchKey::Functionalize});
    if (impl->key_set().has_any(transforms)) return nullptr;
    return impl;
}

bool number(PyObject *object) { return PyFloat_CheckExact(object) || PyLong_CheckExact(object) || PyBool_Check(object); }

// flags: a character per argument, 't' a tensor, 's' a scalar, 'c' a scalar whose value belongs to the signature
bool read_signature(PyObject *args, PyObject *kwargs, const char *flags, Py_ssize_t count, Key &key) {
    if (!PyTuple_CheckExact(args) || PyTuple_GET_SIZE(args) != count) return false;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *arg = PyTuple_GET_ITEM(args, i);
        if (flags[i] == 't') {
            const at::TensorImpl *impl = ordinary(arg);
            if (impl == nullptr) return false;
            const auto sizes = impl->sizes();
            const auto strides = impl->strides();
            key.value((int8_t)c10::typeMetaToScalarType(impl->dtype()));
            key.value((int8_t)impl->device().type());
            key.value((int8_t)impl->device().index());
            key.value((int8_t)sizes.size());
            key.put(sizes.data(), sizes.size() * sizeof(int64_t));
            key.put(strides.data(), strides.size() * sizeof(int64_t));
            continue;
        }
        if (!number(arg)) return false;
        key.value((char)(PyFloat_CheckExact(arg) ? 'f' : PyBool_Check(arg) ? 'b' : 'i'));
        if (flags[i] == 'c') {
            if (PyFloat_CheckExact(arg)) {
                key.value(PyFloat_AS_DOUBLE(arg));
            } else {
                int overflow = 0;
                const long long value = PyLong_AsLongLongAndOverflow(arg, &overflow);
                if (overflow) return false;
                key.value(value);
            }
        }
    }
    if (kwargs != Py_None && kwargs != nullptr) {
        if (!PyDict_CheckExact(kwargs)) return false;
        PyObject *name, *setting;
        Py_ssize_t at = 0;
        while (PyDict_Next(kwargs, &at, &name, &setting)) {
            if (!PyLong_CheckExact(setting)) return false;
            Py_ssize_t size = 0;
            const char *text = PyUnicode_AsUTF8AndSize(name, &size);
            if (text == nullptr) {
                PyErr_Clear();
                return false;
            }
            int overflow = 0;
            const long long value = PyLong_AsLongLongAndOverflow(setting, &overflow);
            if (overflow) return false;
            key.value((int32_t)size);
            key.put(text, (size_t)size);
            key.value(value);
        }
    }
    return key.fits;
}

// ---- launches --------------------------------------------------------------------------------------

PyObject *g_current_device = nullptr, *g_current_stream = nullptr;  // torch's own functions
PyObject *g_check = nullptr;                                        // raises for a result that is not 0

// the current stream of the current device, as torch has it for this thread
bool current_stream(void *&stream) {
    PyObject *device = PyObject_CallNoArgs(g_current_device);
    if (device == nullptr) return false;
    PyObject *handle = PyObject_CallOneArg(g_current_stream, device);
    Py_DECREF(device);
    if (handle == nullptr) return false;
    stream = PyLong_AsVoidPtr(handle);
    Py_DECREF(handle);
    return !PyErr_Occurred();
}

// (throws for a tensor whose memory may not be seen)
char *address(PyObject *args, Py_ssize_t position) { return (char *)THPVariable_Unpack(PyTuple_GET_ITEM(args, position)).data_ptr(); }

// The interpreter's lock is let go while this lives.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// Whether the library answered: `result` is its result.  (Where it ended with an exception a Python exception is set: whether
// something has been launched is not known.)
template <typename Call>
bool in_library(Call call, int &result) {
    bool answered = false;
    {
        Unlocked unlocked;
        try {
            result = call();
            answered = true;
        } catch (...) {
        }
    }
    if (!answered) PyErr_SetString(PyExc_RuntimeError, "The launch ended with a C++ exception (out of host memory?).");
    return answered;
}

// Whether the library answered; everything that is read from Python objects is read before the lock of the interpreter is let go
// (a launch may wait for room in the stream's queue, and what makes room may be a Python callback).  Throws, with nothing
// launched, what the tensors throw.
bool launch(const Recipe &recipe, PyObject *args, void *stream, int &result) {
    if (recipe.kind == kMap) {
        std::vector<NineToothedMapProgram> programs;  // copies: other threads launch the same plan
        programs.reserve(recipe.launches.size());
        for (const MapLaunch &each : recipe.launches) {
            programs.push_back(*each.program);
            NineToothedMapProgram &program = programs.back();
            for (size_t slot = 0; slot < each.operands.size(); ++slot) program.operands[slot].data = address(args, each.operands[slot]);
            for (const auto &scalar : each.scalars) program.value_constants[scalar.first] = PyFloat_AsDouble(PyTuple_GET_ITEM(args, scalar.second));
        }
        if (PyErr_Occurred()) return false;
        const auto function = (decltype(&launch_nt_map))recipe.function;
        return in_library(
            [&] {
                int answer = 0;
                for (const NineToothedMapProgram &program : programs)
                    if (answer == 0) answer = function(stream, &program);
                return answer;
            },
            result);
    }
    constexpr size_t kMaxSlots = 6;
    NineToothedTensor t[kMaxSlots];
    double floats[kMaxSlots];
    int64_t truths[kMaxSlots];
    for (size_t i = 0; i < recipe.slots.size(); ++i) {
        const Slot &slot = recipe.slots[i];
        t[i] = NineToothedTensor{nullptr, const_cast<uint64_t *>(slot.shape.data()), const_cast<int64_t *>(slot.strides.data())};
        if (slot.what == Slot::kTensor) {
            t[i].data = address(args, slot.position) + slot.offset;
        } else if (slot.what == Slot::kFloat) {
            floats[i] = PyFloat_AsDouble(PyTuple_GET_ITEM(args, slot.position));
            t[i] = NineToothedTensor{&floats[i], nullptr, nullptr};
        } else if (slot.what == Slot::kTruth) {
            truths[i] = PyObject_IsTrue(PyTuple_GET_ITEM(args, slot.position));
            t[i] = NineToothedTensor{&truths[i], nullptr, nullptr};
        } else {
            t[i] = NineToothedTensor{nullptr, nullptr, nullptr};
        }
    }
    double scale = recipe.doubles.empty() ? 1.0 : recipe.doubles[0];
    if (recipe.scale_position >= 0) scale = PyFloat_AsDouble(PyTuple_GET_ITEM(args, recipe.scale_position));
    if (PyErr_Occurred()) return false;
    const int *n = recipe.ints.data();
    void *f = recipe.function;
    return in_library(
        [&]() -> int {
            switch (recipe.kind) {
                case kMatmul: return ((decltype(&launch_nt_matmul))f)(stream, t[0], t[1], t[2], n[0], n[1], n[2], n[3], n[4]);
                case kAddmm: return ((decltype(&launch_nt_addmm))f)(stream, t[0], t[1], t[2], t[3], t[4], t[5], n[0], n[1], n[2], n[3]);
                case kLinear: return ((decltype(&launch_nt_linear))f)(stream, t[0], t[1], t[2], n[0], scale, recipe.doubles[1], t[3], n[1], n[2], n[3], n[4]);
                case kSoftmax: return ((decltype(&launch_nt_softmax))f)(stream, t[0], t[1], n[0], n[1]);
                case kAttention: return ((decltype(&launch_nt_attention))f)(stream, t[0], t[1], t[2], t[3], t[4], t[5], n[0], n[1], n[2]);
                case kConv2d: return ((decltype(&launch_nt_conv2d))f)(stream, t[0], t[1], t[2], n[0], n[1], n[2], n[3], n[4], n[5]);
                case kConv2dStrided:
                    return ((decltype(&launch_nt_conv2d_strided))f)(stream, t[0], t[1], t[2], n[0], n[1], n[2], n[3], n[4], n[5], n[6], n[7], n[8], n[9]);
                case kMap: break;  // (above)
            }
            return NINETOOTHED_NO_KERNEL;
        },
        result);
}

// ---- module ----------------------------------------------------------------------------------------

// signature(args, kwargs, flags) -> bytes, or None
PyObject *signature(PyObject *, PyObject *arguments) {
    PyObject *args, *kwargs;
    const char *flags;
    Py_ssize_t count;
    if (!PyArg_ParseTuple(arguments, "OOy#", &args, &kwargs, &flags, &count)) return nullptr;
    Key key;
    if (!read_signature(args, kwargs, flags, count, key)) Py_RETURN_NONE;
    return PyBytes_FromStringAndSize(key.bytes, (Py_ssize_t)key.length);
}

// run(prepared, args, kwargs, flags) -> the plan that `prepared` ({signature: (recipe, plan)}) holds for these arguments, launched; None
// when there is none, or nothing was launched because the linear entry point does not take the operands
PyObject *run(PyObject *, PyObject *const *arguments, Py_ssize_t given) {
    if (given != 4 || !PyDict_CheckExact(arguments[0]) || !PyBytes_CheckExact(arguments[3])) {
        PyErr_SetString(PyExc_TypeError, "run(prepared, args, kwargs, flags)");
        return nullptr;
    }
    PyObject *args = arguments[1];
    if (PyDict_GET_SIZE(arguments[0]) == 0) Py_RETURN_NONE;
    Key key;
    if (!read_signature(args, arguments[2], PyBytes_AS_STRING(arguments[3]), PyBytes_GET_SIZE(arguments[3]), key)) Py_RETURN_NONE;
    PyObject *text = PyBytes_FromStringAndSize(key.bytes, (Py_ssize_t)key.length);
    if (text == nullptr) return nullptr;
    PyObject *entry = PyDict_GetItemWithError(arguments[0], text);
    Py_DECREF(text);
    if (entry == nullptr) {
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_NONE;
    }
    Py_INCREF(entry);  // (another thread may change the dictionary while the launch is under way)
    PyObject *outcome = nullptr;
    void *stream = nullptr;
    if (const Recipe *recipe = (const Recipe *)PyCapsule_GetPointer(PyTuple_GET_ITEM(entry, 0), kCapsule); recipe != nullptr && current_stream(stream)) {
        int result = 0;
        bool answered = false, thrown = false;
        try {
            answered = launch(*recipe, args, stream, result);
        } catch (...) {  // (nothing has been launched: the way through Python reports it)
            thrown = true;
            PyErr_Clear();
        }
        if (thrown || (answered && recipe->kind == kLinear && result == NINETOOTHED_NO_KERNEL)) {
            outcome = Py_None;
            Py_INCREF(outcome);
        } else if (answered && result == 0) {
            outcome = PyTuple_GET_ITEM(entry, 1);
            Py_INCREF(outcome);
        } else if (answered) {
            PyObject *raised = PyObject_CallFunction(g_check, "i", result);
            if (raised != nullptr) PyErr_SetString(PyExc_SystemError, "a failed launch was not reported");
            Py_XDECREF(raised);
        }
    }
    Py_DECREF(entry);
    return outcome;
}

// recipe(kind, address, slots, ints, doubles, scale_position, launches): slots of ("t", position, offset, shape, strides),
// ("f", position), ("b", position) or None; launches of (program address, operand positions, [(constant, position)])
PyObject *make_recipe(PyObject *, PyObject *arguments) {
    const char *kind;
    unsigned long long function;
    PyObject *slots, *ints, *doubles, *launches;
    Py_ssize_t scale_position;
    if (!PyArg_ParseTuple(arguments, "sKO!O!O!nO!", &kind, &function, &PyTuple_Type, &slots, &PyTuple_Type, &ints, &PyTuple_Type, &doubles, &scale_position, &PyTuple_Type, &launches))
        return nullptr;
    auto recipe = std::make_unique<Recipe>();
    size_t index = 0;
    while (index < sizeof(kKinds) / sizeof(kKinds[0]) && std::strcmp(kKinds[index], kind) != 0) ++index;
    constexpr Py_ssize_t kSlots[] = {3, 6, 4, 2, 6, 3, 3, 0}, kInts[] = {5, 4, 5, 2, 3, 6, 10, 0};
    if (index == sizeof(kKinds) / sizeof(kKinds[0]) || PyTuple_GET_SIZE(slots) != kSlots[index] || PyTuple_GET_SIZE(ints) != kInts[index] ||
        (index == kLinear && PyTuple_GET_SIZE(doubles) != 2)) {
        PyErr_SetString(PyExc_ValueError, "no such recipe");
        return nullptr;
    }
    recipe->kind = (Kind)index;
    recipe->function = (void *)(uintptr_t)function;
    recipe->scale_position = scale_position;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(slots); ++i) {
        Slot slot;
        PyObject *item = PyTuple_GET_ITEM(slots, i);
        if (item != Py_None) {
            const char *what;
            PyObject *shape = nullptr, *strides = nullptr;
            long long offset = 0;
            if (!PyArg_ParseTuple(item, "sn|LO!O!", &what, &slot.position, &offset, &PyTuple_Type, &shape, &PyTuple_Type, &strides)) return nullptr;
            slot.what = what[0] == 't' ? Slot::kTensor : what[0] == 'f' ? Slot::kFloat : Slot::kTruth;
            slot.offset = offset;
            for (Py_ssize_t d = 0; shape != nullptr && d < PyTuple_GET_SIZE(shape); ++d) slot.shape.push_back(PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(shape, d)));
            for (Py_ssize_t d = 0; strides != nullptr && d < PyTuple_GET_SIZE(strides); ++d) slot.strides.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(strides, d)));
        }
        recipe->slots.push_back(std::move(slot));
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(ints); ++i) recipe->ints.push_back((int)PyLong_AsLong(PyTuple_GET_ITEM(ints, i)));
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(doubles); ++i) recipe->doubles.push_back(PyFloat_AsDouble(PyTuple_GET_ITEM(doubles, i)));
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(launches); ++i) {
        unsigned long long program;
        PyObject *operands, *scalars;
        if (!PyArg_ParseTuple(PyTuple_GET_ITEM(launches, i), "KO!O!", &program, &PyTuple_Type, &operands, &PyTuple_Type, &scalars)) return nullptr;
        MapLaunch each{(const NineToothedMapProgram *)(uintptr_t)program, {}, {}};
        for (Py_ssize_t slot = 0; slot < PyTuple_GET_SIZE(operands); ++slot) each.operands.push_back(PyLong_AsSsize_t(PyTuple_GET_ITEM(operands, slot)));
        for (Py_ssize_t slot = 0; slot < PyTuple_GET_SIZE(scalars); ++slot) {
            Py_ssize_t constant, position;
            if (!PyArg_ParseTuple(PyTuple_GET_ITEM(scalars, slot), "nn", &constant, &position)) return nullptr;
            each.scalars.emplace_back(constant, position);
        }
        recipe->launches.push_back(std::move(each));
    }
    if (PyErr_Occurred()) return nullptr;
    PyObject *capsule = PyCapsule_New(recipe.get(), kCapsule, [](PyObject *self) { delete (Recipe *)PyCapsule_GetPointer(self, kCapsule); });
    if (capsule != nullptr) (void)recipe.release();
    return capsule;
}

// use(current_device, current_stream, check): the functions that say where a launch goes, and the one that raises for a result
PyObject *use(PyObject *, PyObject *arguments) {
    PyObject *device, *stream, *check;
    if (!PyArg_ParseTuple(arguments, "OOO", &device, &stream, &check)) return nullptr;
    Py_INCREF(device);
    Py_INCREF(stream);
    Py_INCREF(check);
    Py_XSETREF(g_current_device, device);
    Py_XSETREF(g_current_stream, stream);
    Py_XSETREF(g_check, check);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"signature", signature, METH_VARARGS, nullptr},
    {"run", (PyCFunction)(void *)run, METH_FASTCALL, nullptr},
    {"recipe", make_recipe, METH_VARARGS, nullptr},
    {"use", use, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "nt_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_nt_call() {
    PyObject *self = PyModule_Create(&module);
    // (tensors are read through torch's own headers: their layout belongs to this version)
    if (self != nullptr && PyModule_AddStringConstant(self, "torch_version", NT_TORCH_VERSION) != 0) Py_CLEAR(self);
    return self;
}
