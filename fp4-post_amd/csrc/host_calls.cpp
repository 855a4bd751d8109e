// Calls of the C ABI from Python in one step: outputs and scratch are allocated by torch's allocator, tensors become addresses and the entry point
// is called, without an interpreter's round trip for each of these.  Host code only; the arithmetic is libmetis_hip.so's.
//
//   call(name, device_index, specs, args) -> tuple of tensors, or the entry point's return code if it is not METIS_OK
//
// specs: one (type, size, ...) per tensor to allocate on the device, type 0 uint8, 1 bfloat16, 2 float32.  args: the entry point's arguments in order,
// each taken as the declaration in metis_hip.h says: for an integer whatever Python takes for an index (its low bits, as ctypes passes it), for a float
// whatever has a float value, for an address None, a tensor, an integer or the new tensor at a text of one character's distance from "0", for an array of
// structures (metis_linear_member, metis_lowrank_factor) a list of tuples of their 64-bit words, as many as the argument behind it says.  Anything else
// is a TypeError or a ValueError, before anything is allocated.  The interpreter's lock is released for the allocations and the call, as torch.empty and
// ctypes release it.
//
// Per call and new tensor the same through ctypes and torch.empty cost 5.1 and 1.7 us, here 3.9 and 1.0 (launch included): an eager decode step
// of five sequences (hidden 1536, 19 launches, 46 new tensors) 415 -> 367 us, a prompt of 411 tokens 462 -> 410, a small round trip 8.2 -> 6.8.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstddef>
#include <cstring>
#include <ATen/ops/empty.h>
#include <c10/util/SmallVector.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/metis_hip.h"

namespace {

enum Kind : uint8_t { kInteger, kReal, kAddress, kMembers, kFactors };
template <class T>
constexpr Kind kind_of()
{
    using P = std::remove_cv_t<std::remove_pointer_t<T>>;
    if (std::is_floating_point<T>::value) return kReal;
    if (!std::is_pointer<T>::value) return kInteger;
    if (std::is_same<P, metis_linear_member>::value) return kMembers;
    return std::is_same<P, metis_lowrank_factor>::value ? kFactors : kAddress;
}
template <class... A> struct Kinds { static constexpr Kind of[] = {kind_of<A>()...}; };
template <class... A> constexpr const Kind* kinds(int (*)(A...)) { return Kinds<A...>::of; }
// an array of structures is followed by their number
constexpr bool counted(const Kind* k, size_t n)
{
    for (size_t i = 0; i < n; ++i)
        if ((k[i] == kMembers || k[i] == kFactors) && (i + 1 == n || k[i + 1] != kInteger)) return false;
    return true;
}

// the words of the structures
constexpr Kind kMember[] = {kAddress, kAddress, kAddress, kAddress, kAddress, kInteger, kAddress, kAddress, kInteger, kInteger, kInteger, kAddress};
constexpr Kind kFactor[] = {kAddress, kAddress, kInteger};
static_assert(sizeof(metis_linear_member) == sizeof(kMember) * 8 && offsetof(metis_linear_member, r) == 5 * 8 && offsetof(metis_linear_member, N) == 8 * 8 &&
              offsetof(metis_linear_member, bias_is_f32) == 9 * 8 && offsetof(metis_linear_member, ldt) == 10 * 8, "kMember follows the declaration");
static_assert(sizeof(metis_lowrank_factor) == sizeof(kFactor) * 8 && offsetof(metis_lowrank_factor, r) == 2 * 8, "kFactor follows the declaration");

union Value {                                                  // (a float's bits lie in the word)
    int64_t i;
    double f;
};

template <class T>
T as(const Value& v)
{
    if constexpr (std::is_pointer<T>::value) return reinterpret_cast<T>(static_cast<uintptr_t>(v.i));
    else if constexpr (std::is_floating_point<T>::value) return static_cast<T>(v.f);
    else return static_cast<T>(v.i);
}

template <class... A, size_t... I>
int spread(int (*fn)(A...), const Value* v, std::index_sequence<I...>)
{
    return fn(as<A>(v[I])...);
}
template <class... A>
constexpr size_t arity(int (*)(A...)) { return sizeof...(A); }
template <class... A>
int spread_all(int (*fn)(A...), const Value* v) { return spread(fn, v, std::index_sequence_for<A...>()); }

struct Entry {
    const char* name;
    size_t args;
    const Kind* kinds;
    int (*run)(const Value*);
};
#define METIS_ENTRY(fn) {#fn, arity(fn), kinds(fn), [](const Value* v) { return spread_all(fn, v); }}
constexpr Entry kEntries[] = {
    METIS_ENTRY(metis_nvfp4_quant_row),
    METIS_ENTRY(metis_nvfp4_quant_col),
    METIS_ENTRY(metis_nvfp4_quant_col_padded),
    METIS_ENTRY(metis_nvfp4_quant_sr_row),
    METIS_ENTRY(metis_nvfp4_quant_sr_col),
    METIS_ENTRY(metis_nvfp4_quant_sr_both_padded),
    METIS_ENTRY(metis_nvfp4_quant_sr_both_centered),
    METIS_ENTRY(metis_nvfp4_quant_sr_both_copy),
    METIS_ENTRY(metis_nvfp4_quant_centered),
    METIS_ENTRY(metis_nvfp4_quant_row_decode),
    METIS_ENTRY(metis_nvfp4_quant_row_deferred),
    METIS_ENTRY(metis_nvfp4_quant_row_resident),
    METIS_ENTRY(metis_nvfp4_quant_lowrank_residual),
    METIS_ENTRY(metis_nvfp4_quant_project_deferred),
    METIS_ENTRY(metis_nvfp4_roundtrip),
    METIS_ENTRY(metis_token_mean_quant_deferred),
    METIS_ENTRY(metis_rmsnorm),
    METIS_ENTRY(metis_rmsnorm_colmean),
    METIS_ENTRY(metis_rmsnorm_backward),
    METIS_ENTRY(metis_rmsnorm_nvfp4_quant),
    METIS_ENTRY(metis_rmsnorm_nvfp4_quant_decode),
    METIS_ENTRY(metis_rmsnorm_nvfp4_quant_deferred),
    METIS_ENTRY(metis_decode_quant_project_deferred),
    METIS_ENTRY(metis_decode_prepare_deferred),
    METIS_ENTRY(metis_linear_fwd_grouped),
    METIS_ENTRY(metis_linear_fwd_grouped_bf16),
    METIS_ENTRY(metis_linear_fwd_grouped_centered),
    METIS_ENTRY(metis_linear_fwd_grouped_operand),
    METIS_ENTRY(metis_linear_fwd_tiled),
    METIS_ENTRY(metis_linear_fwd_tiled_grouped),
    METIS_ENTRY(metis_linear_dgrad),
    METIS_ENTRY(metis_linear_dgrad_ws),
    METIS_ENTRY(metis_linear_wgrad),
    METIS_ENTRY(metis_linear_wgrad_ws),
    METIS_ENTRY(metis_nvfp4_expand_tiled),
    METIS_ENTRY(metis_nvfp4_expand_tiled_centered),
    METIS_ENTRY(metis_nvfp4_expand_tiled_deferred),
    METIS_ENTRY(metis_nvfp4_expand_tiled_rht),
    METIS_ENTRY(metis_lowrank_project),
    METIS_ENTRY(metis_lowrank_project_rows_ws),
    METIS_ENTRY(metis_lowrank_project_rows_grouped),
    METIS_ENTRY(metis_lowrank_backward),
};
constexpr size_t kMaxArgs = 32, kMaxOuts = 32;
constexpr bool all_counted()
{
    for (const Entry& e : kEntries)
        if (e.args > kMaxArgs || !counted(e.kinds, e.args)) return false;
    return true;
}
static_assert(all_counted(), "at most kMaxArgs arguments, and a number behind every array of structures");
PyObject* g_index = nullptr;                                   // name -> position in kEntries

// the new tensors, and where their addresses go once they exist
struct Outputs {
    size_t count = 0;
    c10::SmallVector<std::pair<int64_t*, size_t>, 16> at;
};
// The interpreter's lock given up: an allocation may wait for the device, or for memory that it has to get back first.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// one argument or word of the given kind; false with a Python error set
bool value_of(PyObject* o, Kind kind, Outputs& outs, int64_t* v)
{
    if (kind == kReal) {
        const double f = PyFloat_AsDouble(o);
        memcpy(v, &f, sizeof f);
        return !(f == -1.0 && PyErr_Occurred());
    }
    if ((kind == kInteger || kind == kAddress) && PyLong_Check(o)) {   // (also bool; 64-bit seeds may use the sign bit)
        *v = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(o));
        return !(*v == -1 && PyErr_Occurred());
    }
    if (kind == kInteger) {
        PyObject* n = PyNumber_Index(o);
        if (!n) return false;
        *v = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(n));
        Py_DECREF(n);
        return !(*v == -1 && PyErr_Occurred());
    }
    if (kind == kAddress) {
        if (o == Py_None) { *v = 0; return true; }
        if (THPVariable_Check(o)) {
            *v = static_cast<int64_t>(reinterpret_cast<uintptr_t>(THPVariable_Unpack(o).data_ptr()));
            return true;
        }
        if (PyUnicode_Check(o) && PyUnicode_GET_LENGTH(o) == 1) {
            const int k = static_cast<int>(PyUnicode_READ_CHAR(o, 0)) - '0';
            if (k >= 0 && static_cast<size_t>(k) < outs.count) { outs.at.push_back({v, static_cast<size_t>(k)}); return true; }
        }
    }
    PyErr_Format(PyExc_TypeError, kind == kAddress ? "call: %s for an address" : "call: %s for a list of structures", Py_TYPE(o)->tp_name);
    return false;
}

PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != 4 || !PyTuple_Check(a[2]) || !PyTuple_Check(a[3])) {
        PyErr_SetString(PyExc_TypeError, "call(name, device_index, specs, args)");
        return nullptr;
    }
    PyObject* pos = PyDict_GetItemWithError(g_index, a[0]);
    if (!pos) {
        if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%S", a[0]);
        return nullptr;
    }
    const Entry& e = kEntries[PyLong_AsLong(pos)];
    const long device = PyLong_AsLong(a[1]);
    if (device == -1 && PyErr_Occurred()) return nullptr;

    static const at::ScalarType types[] = {at::kByte, at::kBFloat16, at::kFloat};
    struct { at::ScalarType type; size_t begin, dims; } spec[kMaxOuts];
    c10::SmallVector<int64_t, 64> sizes;
    Outputs outs;
    const Py_ssize_t count = PyTuple_GET_SIZE(a[2]);
    if (count > static_cast<Py_ssize_t>(kMaxOuts)) { PyErr_SetString(PyExc_ValueError, "call: too many tensors"); return nullptr; }
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* s = PyTuple_GET_ITEM(a[2], i);
        const Py_ssize_t dims = PyTuple_Check(s) ? PyTuple_GET_SIZE(s) - 1 : -1;
        const long type = dims >= 0 ? PyLong_AsLong(PyTuple_GET_ITEM(s, 0)) : -1;
        if (dims < 0 || type < 0 || type > 2) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "call: a spec is (0 | 1 | 2, size, ...)");
            return nullptr;
        }
        spec[i] = {types[type], sizes.size(), static_cast<size_t>(dims)};
        for (Py_ssize_t d = 0; d < dims; ++d) {
            sizes.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(s, d + 1)));
            if (sizes.back() == -1 && PyErr_Occurred()) return nullptr;
        }
        ++outs.count;
    }

    Value v[kMaxArgs];
    std::vector<int64_t> words[2];                             // arrays of structures; never moved once their words are asked for
    size_t arrays = 0;
    Py_ssize_t listed = 0;                                     // structures of the last array
    const size_t given = static_cast<size_t>(PyTuple_GET_SIZE(a[3]));
    if (given != e.args) {
        PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (%zu given)", e.name, e.args, given);
        return nullptr;
    }
    for (size_t i = 0; i < given; ++i) {
        PyObject* o = PyTuple_GET_ITEM(a[3], static_cast<Py_ssize_t>(i));
        const bool members = e.kinds[i] == kMembers;
        if (!PyList_Check(o) || (!members && e.kinds[i] != kFactors)) {
            if (!value_of(o, e.kinds[i], outs, &v[i].i)) return nullptr;
            if (i > 0 && (e.kinds[i - 1] == kMembers || e.kinds[i - 1] == kFactors) && v[i].i != listed) {
                PyErr_Format(PyExc_ValueError, "%s: %zd structures for %lld", e.name, listed, static_cast<long long>(v[i].i));
                return nullptr;
            }
            continue;
        }
        if (arrays == 2) { PyErr_SetString(PyExc_ValueError, "call: too many arrays"); return nullptr; }
        std::vector<int64_t>& w = words[arrays++];
        const Kind* layout = members ? kMember : kFactor;
        const Py_ssize_t size = members ? sizeof(kMember) : sizeof(kFactor);
        listed = PyList_GET_SIZE(o);
        w.resize(static_cast<size_t>(listed * size));
        for (Py_ssize_t k = 0; k < listed; ++k) {
            PyObject* m = k < PyList_GET_SIZE(o) ? PyList_GET_ITEM(o, k) : nullptr;
            if (!m || !PyTuple_Check(m) || PyTuple_GET_SIZE(m) != size) {
                PyErr_Format(PyExc_TypeError, "%s: a structure is a tuple of its %zd words", e.name, size);
                return nullptr;
            }
            for (Py_ssize_t j = 0; j < size; ++j)
                if (!value_of(PyTuple_GET_ITEM(m, j), layout[j], outs, &w[static_cast<size_t>(k * size + j)])) return nullptr;
        }
        v[i].i = static_cast<int64_t>(reinterpret_cast<uintptr_t>(w.data()));
    }
    int rc;
    c10::SmallVector<at::Tensor, 8> fresh;
    {
        Unlocked unlocked;
        const at::Device on(at::kCUDA, static_cast<at::DeviceIndex>(device));
        for (Py_ssize_t i = 0; i < count; ++i)
            fresh.push_back(at::empty(at::IntArrayRef(sizes.data() + spec[i].begin, spec[i].dims), at::TensorOptions().dtype(spec[i].type).device(on)));
        for (const auto& at : outs.at) *at.first = static_cast<int64_t>(reinterpret_cast<uintptr_t>(fresh[at.second].data_ptr()));
        rc = e.run(v);
    }
    if (rc != METIS_OK) return PyLong_FromLong(rc);
    PyObject* result = PyTuple_New(count);
    if (!result) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* t = THPVariable_Wrap(std::move(fresh[static_cast<size_t>(i)]));
        if (!t) { Py_DECREF(result); return nullptr; }
        PyTuple_SET_ITEM(result, i, t);                        // the reference moves into the tuple
    }
    return result;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&call)), METH_FASTCALL,
                          "call(name, device_index, specs, args): allocate, call an entry point, return the new tensors or its return code"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_metis_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__metis_host()
{
    PyObject* m = PyModule_Create(&module_def);
    g_index = PyDict_New();
    if (!m || !g_index) return nullptr;
    for (size_t i = 0; i < sizeof(kEntries) / sizeof(kEntries[0]); ++i) {
        PyObject* key = PyUnicode_InternFromString(kEntries[i].name);
        PyObject* val = PyLong_FromSize_t(i);
        if (!key || !val || PyDict_SetItem(g_index, key, val)) return nullptr;
        Py_DECREF(key);
        Py_DECREF(val);
    }
    return m;
}
