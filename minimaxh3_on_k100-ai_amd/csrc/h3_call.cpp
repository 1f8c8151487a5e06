// The Python face's fast call into libh3mi355x.so: one C function that checks a
// launcher's arguments, fills its NineToothedTensor structs from the torch
// tensors and launches on the current stream.
//
// What bounds a small launch is the host: through ctypes, building the structs
// and the checks in Python took 12 us (SwiGLU, three tensors) to 30 us (the
// q/k/v pack, twelve) per call, most of it longer than the kernels of a
// 256-token block. Here a call takes the launch itself and under 2 us.
//
// call(plan, *args) calls the launcher once and returns True, or its status
// where that is not 0. It returns False without having called it for anything
// but the plain case (every tensor an exact torch.Tensor on the current GPU
// with the planned rank and dtype): the caller takes its Python path, which
// converts what can be converted and launches. After a status the caller must
// not launch again: a launcher ends with the thread's last HIP error, which an
// earlier call may have left, so its kernels may be queued all the same.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstring>
#include <utility>
#include <vector>

#include "../../include/h3mi355x.h"

namespace {

constexpr int kMaxArgs = 20;    // structs of a launch (the widest entry takes 17)
constexpr int kMaxInputs = 16;  // arguments of a call

// One argument: what it must be. kind:
//   b bf16   f fp32   c fp32, contiguous   d fp64   l int64   e float8_e4m3fn
//   u float8_e4m3fn or uint8   s a Python float or int
//   t the RoPE cache, bf16 [N, 96] (two structs: its cos and sin halves)
//   i an int64 per-token index, [B, S] or (B = 1) [S] of the first argument
//   w a uint8 workspace, or None for an empty one
struct Arg {
    char kind;
    int dim;
};

struct Plan {
    void *fn = nullptr;
    std::vector<Arg> args;
    std::vector<int> order;  // the launcher's structs, by argument (a cache expands in place)
    int fix_arg = -1, fix_dim = 0;  // argument fix_arg's size at fix_dim must be fix_size
    int64_t fix_size = 0;
};

void destroy_plan(PyObject *capsule) {
    delete static_cast<Plan *>(PyCapsule_GetPointer(capsule, "h3_plan"));
}

PyObject *get_device = nullptr;      // torch._C._cuda_getDevice
PyObject *get_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

// Calls fn(stream, a[0], ..., a[n - 1]).
template <size_t... I>
int invoke_n(void *fn, void *stream, const NineToothedTensor *a, std::index_sequence<I...>) {
    using Fn = NineToothedResult (*)(NineToothedStream, decltype((void)I, NineToothedTensor{})...);
    return static_cast<int>(reinterpret_cast<Fn>(fn)(stream, a[I]...));
}

template <size_t... N>
int invoke(void *fn, void *stream, const NineToothedTensor *a, size_t n, std::index_sequence<N...>) {
    using Call = int (*)(void *, void *, const NineToothedTensor *);
    static constexpr Call table[] = {
        [](void *f, void *s, const NineToothedTensor *x) { return invoke_n(f, s, x, std::make_index_sequence<N>{}); }...};
    return table[n](fn, stream, a);
}

// plan(address, kinds, order, fix): kinds "b3b1s0...": kind and rank of each
// argument; order: the launcher's arguments by index; fix: None or
// (argument, dim, size).
PyObject *make_plan(PyObject *, PyObject *pyargs) {
    unsigned long long address;
    const char *kinds;
    PyObject *order, *fix;
    if (!PyArg_ParseTuple(pyargs, "KsOO", &address, &kinds, &order, &fix)) return nullptr;
    auto *plan = new Plan;
    plan->fn = reinterpret_cast<void *>(static_cast<uintptr_t>(address));
    for (const char *p = kinds; p[0] != 0 && p[1] != 0; p += 2) plan->args.push_back({p[0], p[1] - '0'});
    size_t structs = 0;
    bool ok = PyTuple_Check(order) && plan->args.size() <= kMaxInputs && !plan->args.empty();
    for (Py_ssize_t i = 0; ok && i < PyTuple_GET_SIZE(order); ++i) {
        const long k = PyLong_AsLong(PyTuple_GET_ITEM(order, i));
        ok = k >= 0 && k < static_cast<long>(plan->args.size());
        if (!ok) break;
        plan->order.push_back(static_cast<int>(k));
        structs += plan->args[k].kind == 't' ? 2 : 1;
    }
    if (ok && fix != Py_None) {
        int a, d;
        long long n;
        ok = PyArg_ParseTuple(fix, "iiL", &a, &d, &n) && a >= 0 && a < static_cast<int>(plan->args.size()) && d >= 0 &&
             d < plan->args[a].dim;
        plan->fix_arg = a;
        plan->fix_dim = d;
        plan->fix_size = n;
    }
    if (!ok || structs > kMaxArgs) {
        delete plan;
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bad launch plan");
        return nullptr;
    }
    return PyCapsule_New(plan, "h3_plan", destroy_plan);
}

bool dtype_ok(char kind, at::ScalarType t) {
    switch (kind) {
        case 'b': return t == at::kBFloat16;
        case 't': return t == at::kBFloat16;
        case 'f':
        case 'c': return t == at::kFloat;
        case 'd': return t == at::kDouble;
        case 'l':
        case 'i': return t == at::kLong;
        case 'e': return t == at::kFloat8_e4m3fn;
        case 'u': return t == at::kFloat8_e4m3fn || t == at::kByte;
        case 'w': return t == at::kByte;
        default: return false;
    }
}

// Sizes and strides that stand in for a tensor's own (an index's leading 1, a
// cache's halves, an empty workspace).
struct Extra {
    int64_t size[2], stride[2];
};

PyObject *call(PyObject *, PyObject *const *argv, Py_ssize_t nargs) {
    if (nargs < 1) {
        PyErr_SetString(PyExc_TypeError, "call(plan, *args)");
        return nullptr;
    }
    auto *plan = static_cast<Plan *>(PyCapsule_GetPointer(argv[0], "h3_plan"));
    if (plan == nullptr) return nullptr;
    const size_t n = plan->args.size();
    if (static_cast<size_t>(nargs - 1) != n) Py_RETURN_FALSE;
    NineToothedTensor in[kMaxInputs];
    NineToothedTensor second[kMaxInputs];  // a cache's sin half
    Extra extra[kMaxInputs];
    double scalars[kMaxInputs];
    int device = -1;
    const at::Tensor *first = nullptr;
    try {
        for (size_t i = 0; i < n; ++i) {
            PyObject *o = argv[1 + i];
            const Arg &want = plan->args[i];
            if (want.kind == 's') {
                if (PyFloat_CheckExact(o)) {
                    scalars[i] = PyFloat_AS_DOUBLE(o);
                } else if (PyLong_CheckExact(o)) {
                    scalars[i] = PyLong_AsDouble(o);
                    if (scalars[i] == -1.0 && PyErr_Occurred()) {
                        PyErr_Clear();
                        Py_RETURN_FALSE;
                    }
                } else {
                    Py_RETURN_FALSE;
                }
                in[i] = {&scalars[i], nullptr, nullptr};
                continue;
            }
            if (want.kind == 'w' && o == Py_None) {
                extra[i] = {{0, 0}, {1, 1}};
                in[i] = {nullptr, reinterpret_cast<uint64_t *>(extra[i].size), extra[i].stride};
                continue;
            }
            if (!THPVariable_CheckExact(o)) Py_RETURN_FALSE;
            const at::Tensor &t = THPVariable_Unpack(o);
            if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !dtype_ok(want.kind, t.scalar_type()))
                Py_RETURN_FALSE;
            const bool short_index = want.kind == 'i' && t.dim() == 1;
            if (t.dim() != want.dim && !short_index) Py_RETURN_FALSE;
            const int d = static_cast<int>(t.get_device());
            if (device < 0) device = d;
            if (d != device) Py_RETURN_FALSE;
            if (want.kind == 'c' && !t.is_contiguous()) Py_RETURN_FALSE;
            if (static_cast<int>(i) == plan->fix_arg && t.size(plan->fix_dim) != plan->fix_size) Py_RETURN_FALSE;
            // sizes and strides are read by the launcher before this call returns.
            auto *sizes = reinterpret_cast<uint64_t *>(const_cast<int64_t *>(t.sizes().data()));
            auto *strides = const_cast<int64_t *>(t.strides().data());
            void *data = t.data_ptr();
            if (first == nullptr) first = &t;
            if (short_index) {
                if (first->dim() < 2 || first->size(0) != 1) Py_RETURN_FALSE;
                extra[i] = {{1, t.size(0)}, {0, t.stride(0)}};
                in[i] = {data, reinterpret_cast<uint64_t *>(extra[i].size), extra[i].stride};
            } else if (want.kind == 't') {
                if (t.size(1) != 96) Py_RETURN_FALSE;
                extra[i] = {{t.size(0), 48}, {t.stride(0), t.stride(1)}};
                in[i] = {data, reinterpret_cast<uint64_t *>(extra[i].size), extra[i].stride};
                second[i] = in[i];
                if (data != nullptr) second[i].data = static_cast<char *>(data) + 2 * 48 * t.stride(1);
            } else {
                in[i] = {data, sizes, strides};
            }
        }
    } catch (...) {  // a tensor without storage or with symbolic sizes
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
    if (device < 0) Py_RETURN_FALSE;
    // The launch goes to the current stream; another device than the current
    // one is switched to in Python.
    PyObject *current = PyObject_CallNoArgs(get_device);
    if (current == nullptr) return nullptr;
    const long cur = PyLong_AsLong(current);
    if (cur != device) {
        Py_DECREF(current);
        if (PyErr_Occurred()) return nullptr;
        Py_RETURN_FALSE;
    }
    PyObject *raw = PyObject_CallOneArg(get_raw_stream, current);
    Py_DECREF(current);
    if (raw == nullptr) return nullptr;
    void *stream = PyLong_AsVoidPtr(raw);
    Py_DECREF(raw);
    if (stream == nullptr && PyErr_Occurred()) return nullptr;
    NineToothedTensor a[kMaxArgs];
    size_t m = 0;
    for (int k : plan->order) {
        a[m++] = in[k];
        if (plan->args[k].kind == 't') a[m++] = second[k];
    }
    int status;
    Py_BEGIN_ALLOW_THREADS  // as ctypes does: a launch may wait for room in its queue
    status = invoke(plan->fn, stream, a, m, std::make_index_sequence<kMaxArgs + 1>{});
    Py_END_ALLOW_THREADS
    if (status == 0) Py_RETURN_TRUE;
    return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"plan", make_plan, METH_VARARGS, "plan(address, kinds, order, fix) -> launch plan"},
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL,
     "call(plan, *args) -> True, or the launcher's non-zero status; False if it was not called"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_h3call", "fast calls into libh3mi355x.so", -1, methods,
                      nullptr,               nullptr,   nullptr,                          nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__h3call() {
    PyObject *c = PyImport_ImportModule("torch._C");
    if (c == nullptr) return nullptr;
    get_device = PyObject_GetAttrString(c, "_cuda_getDevice");
    get_raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
    Py_DECREF(c);
    if (get_device == nullptr || get_raw_stream == nullptr) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", H3_TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
