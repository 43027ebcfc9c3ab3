// The small operators of guffin_amd.hip as Python calls without an interpreter's work in them: their tensors are allocated and the
// library's entry points called from here.  These operators run for 3 to 10 us; a call through ctypes with its allocations took 6 to 12
// (a receipt and a product 13.7 us, of which the device worked 10.8), so the host was what bounded them.
//
// Every function takes its operator's usual form alone -- plain device tensors, outputs to be allocated -- and returns None for
// anything else, which the Python function it stands in front of then handles (or refuses) as it always did.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>

namespace {

// Entry points of libguffin_hip.so, bound by address (the library is the interpreter's to load).
struct Library {
    uint64_t (*receipt_bytes)(uint32_t, uint32_t);
    int (*group_sums)(void*, const float*, float*, uint32_t, uint32_t);
    uint32_t (*gemv_packed_slices)(int, uint32_t, uint32_t);
    int (*gemv_packed)(void*, int, const void*, const float*, const float*, float*, float*, uint32_t, uint32_t, uint32_t);
    int (*repack)(void*, int, const void*, void*, uint32_t, uint32_t);
    uint64_t (*select_workspace_bytes)(uint32_t, uint32_t, uint32_t);
    int (*select_candidates_fresh)(void*, const float*, uint32_t, uint32_t, uint32_t, const void*, const void*, void*, void*, void*);
    uint64_t (*draft_law_workspace_bytes)(uint32_t);
    int (*draft_law_fresh)(void*, const float*, uint32_t, const void*, uint64_t, uint64_t, const void*, void*, void*, uint32_t*, uint32_t*);
    int (*spec_accept)(void*, const void*, const void*, const uint32_t*, const void*, uint64_t, uint64_t, const void*, void*, uint32_t*);
};
constexpr const char* kNames[] = {"receipt_bytes", "group_sums", "gemv_packed_slices", "gemv_packed", "repack", "select_workspace_bytes",
                                  "select_candidates_fresh", "draft_law_workspace_bytes", "draft_law_fresh", "spec_accept"};
constexpr Py_ssize_t kCount = sizeof(kNames) / sizeof(kNames[0]);
static_assert(sizeof(Library) == kCount * sizeof(void*));
Library g_lib;
uint32_t g_candidates_bytes, g_law_bytes, g_result_bytes;
PyObject* g_check;     // raises the library's error for a code
PyObject* g_options;   // the class of a sampler's options

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
at::TensorOptions on(const at::Device& device, at::ScalarType type) { return at::TensorOptions().dtype(type).device(device); }

// a plain tensor in device memory, or null
const at::Tensor* tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}
bool word(PyObject* o, uint32_t& to) {
    if (!PyLong_CheckExact(o)) return false;
    to = static_cast<uint32_t>(PyLong_AsUnsignedLongLongMask(o));
    return true;
}
// what ctypes takes for a c_uint64: any integer, its low 64 bits
bool wide(PyObject* o, uint64_t& to) {
    if (!PyLong_CheckExact(o)) return false;
    to = PyLong_AsUnsignedLongLongMask(o);
    return true;
}
// the bytes of a sampler's options (a ctypes structure; other objects with 20 bytes are not) while they live
struct Options {
    Py_buffer view {};
    bool held = false;
    explicit Options(PyObject* o) {
        if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_options) return;
        held = PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0;
        if (!held) PyErr_Clear();
    }
    ~Options() { if (held) PyBuffer_Release(&view); }
};

// the call without the interpreter's lock; false with an exception set where the library refuses it
template <typename Call>
bool done(Call call) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = call();
    Py_END_ALLOW_THREADS
    if (rc == 0) return true;
    PyObject* raised = PyObject_CallFunction(g_check, "i", rc);
    if (raised) {   // it always raises
        Py_DECREF(raised);
        PyErr_SetString(PyExc_RuntimeError, "guffin_amd: an entry point failed");
    }
    return false;
}

// C++ exceptions (an allocation that fails) leave as the Python exceptions torch makes of them
#define GUFFIN_ENTER HANDLE_TH_ERRORS
#define GUFFIN_LEAVE END_HANDLE_TH_ERRORS

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != kCount + 5) { PyErr_SetString(PyExc_TypeError, "bind: the entry points' addresses, three record sizes, the error function, the options' class"); return nullptr; }
    void* at[kCount];
    for (Py_ssize_t i = 0; i < kCount; ++i) {
        at[i] = PyLong_AsVoidPtr(args[i]);
        if (!at[i]) { if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "bind: no address for %s", kNames[i]); return nullptr; }
    }
    if (!word(args[kCount], g_candidates_bytes) || !word(args[kCount + 1], g_law_bytes) || !word(args[kCount + 2], g_result_bytes)) {
        PyErr_SetString(PyExc_TypeError, "bind: record sizes are integers");
        return nullptr;
    }
    std::memcpy(&g_lib, at, sizeof(g_lib));
    Py_INCREF(args[kCount + 3]);
    Py_XSETREF(g_check, args[kCount + 3]);
    Py_INCREF(args[kCount + 4]);
    Py_XSETREF(g_options, args[kCount + 4]);
    Py_RETURN_NONE;
}

PyObject* group_sums(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    const at::Tensor* x = n == 1 ? tensor(args[0]) : nullptr;
    if (!x || x->dim() != 2) Py_RETURN_NONE;
    const uint32_t rows = static_cast<uint32_t>(x->size(0)), K = static_cast<uint32_t>(x->size(1));
    const uint64_t bytes = g_lib.receipt_bytes(rows, K);
    if (bytes == 0) Py_RETURN_NONE;
    const int64_t words = K / 16 + K / 32;
    const at::Tensor out = at::empty({static_cast<int64_t>(bytes / 4)}, on(x->device(), at::kFloat)).as_strided({rows, words}, {words, 1});
    void *const s = stream(), *const to = out.data_ptr();
    const void* const from = x->data_ptr();
    if (!done([&] { return g_lib.group_sums(s, static_cast<const float*>(from), static_cast<float*>(to), rows, K); })) return nullptr;
    return THPVariable_Wrap(out);
    GUFFIN_LEAVE
}

PyObject* gemv_packed(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    uint32_t dtype, N;
    if (n != 5 || !word(args[0], dtype) || !word(args[4], N)) Py_RETURN_NONE;
    const at::Tensor *tiles = tensor(args[1]), *x = tensor(args[2]), *sums = tensor(args[3]);
    if (!tiles || !x || !sums || x->dim() != 2) Py_RETURN_NONE;
    const uint32_t rows = static_cast<uint32_t>(x->size(0)), K = static_cast<uint32_t>(x->size(1));
    const uint32_t planes = g_lib.gemv_packed_slices(static_cast<int>(dtype), K, N);
    if (planes == 0) Py_RETURN_NONE;
    // a single plane is the result itself; several and their sum are one allocation
    const int64_t before = planes == 1 ? 0 : int64_t(planes) * rows;
    const at::Tensor all = at::empty({before + rows, int64_t(N)}, on(x->device(), at::kFloat));
    const at::Tensor out = before ? all.narrow(0, before, rows) : all;
    void *const s = stream(), *const first = all.data_ptr(), *const last = out.data_ptr();
    const void *const w = tiles->data_ptr(), *const xp = x->data_ptr(), *const xs = sums->data_ptr();
    if (!done([&] { return g_lib.gemv_packed(s, static_cast<int>(dtype), w, static_cast<const float*>(xp), static_cast<const float*>(xs),
                                             static_cast<float*>(first), static_cast<float*>(last), rows, K, N); })) return nullptr;
    return THPVariable_Wrap(out);
    GUFFIN_LEAVE
}

PyObject* repack(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    uint32_t dtype, K, N;
    const at::Tensor* canonical = n == 4 ? tensor(args[1]) : nullptr;
    if (!canonical || !word(args[0], dtype) || !word(args[2], K) || !word(args[3], N)) Py_RETURN_NONE;
    const at::Tensor tiles = at::empty_like(*canonical);
    void *const s = stream(), *const to = tiles.data_ptr();
    const void* const from = canonical->data_ptr();
    if (!done([&] { return g_lib.repack(s, static_cast<int>(dtype), from, to, K, N); })) return nullptr;
    return THPVariable_Wrap(tiles);
    GUFFIN_LEAVE
}

PyObject* pair(const at::Tensor& a, const at::Tensor& b) { return Py_BuildValue("(NN)", THPVariable_Wrap(a), THPVariable_Wrap(b)); }

PyObject* select_candidates(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    uint32_t retain;
    const at::Tensor* logits = n == 2 ? tensor(args[0]) : nullptr;
    if (!logits || logits->dim() != 2 || !word(args[1], retain)) Py_RETURN_NONE;
    const uint32_t rows = static_cast<uint32_t>(logits->size(0)), vocab = static_cast<uint32_t>(logits->size(1));
    const uint64_t bytes = g_lib.select_workspace_bytes(rows, vocab, retain);
    const at::Device here(at::kCUDA);
    const at::Tensor ws = at::empty({static_cast<int64_t>(bytes)}, on(here, at::kByte));
    const at::Tensor result = at::empty({int64_t(rows) * g_candidates_bytes}, on(here, at::kByte));
    const at::Tensor status = at::empty({int64_t(rows)}, on(here, at::kInt));
    void *const s = stream(), *const w = ws.data_ptr(), *const r = result.data_ptr(), *const st = status.data_ptr();
    const void* const from = logits->data_ptr();
    if (!done([&] { return g_lib.select_candidates_fresh(s, static_cast<const float*>(from), rows, vocab, retain, nullptr, nullptr, w, r, st); })) return nullptr;
    return pair(result, status);
    GUFFIN_LEAVE
}

PyObject* draft_law(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    uint64_t seed, step;
    const at::Tensor* logits = n == 4 ? tensor(args[0]) : nullptr;
    if (!logits || !wide(args[2], seed) || !wide(args[3], step)) Py_RETURN_NONE;
    const Options options(args[1]);
    if (!options.held) Py_RETURN_NONE;
    const uint32_t vocab = static_cast<uint32_t>(logits->numel());
    const at::Device here(at::kCUDA);
    const at::Tensor ws = at::empty({static_cast<int64_t>(g_lib.draft_law_workspace_bytes(vocab))}, on(here, at::kByte));
    const at::Tensor law = at::empty({int64_t(g_law_bytes)}, on(here, at::kByte));
    const at::Tensor proposal = at::empty({1}, on(here, at::kInt)), status = at::empty({1}, on(here, at::kInt));
    void *const s = stream(), *const w = ws.data_ptr(), *const l = law.data_ptr();
    auto *const p = static_cast<uint32_t*>(proposal.data_ptr()), *const st = static_cast<uint32_t*>(status.data_ptr());
    const void* const from = logits->data_ptr();
    if (!done([&] { return g_lib.draft_law_fresh(s, static_cast<const float*>(from), vocab, options.view.buf, seed, step, nullptr, w, l, p, st); })) return nullptr;
    return Py_BuildValue("(NNN)", THPVariable_Wrap(law), THPVariable_Wrap(proposal), THPVariable_Wrap(status));
    GUFFIN_LEAVE
}

PyObject* spec_accept(PyObject*, PyObject* const* args, Py_ssize_t n) {
    GUFFIN_ENTER
    uint64_t seed, step;
    if (n != 7 || !wide(args[4], seed) || !wide(args[5], step)) Py_RETURN_NONE;
    const at::Tensor *cands = tensor(args[0]), *law = tensor(args[1]), *proposal = tensor(args[2]), *status = args[6] == Py_None ? nullptr : tensor(args[6]);
    if (!cands || !law || !proposal || (args[6] != Py_None && !status)) Py_RETURN_NONE;
    const Options options(args[3]);
    if (!options.held) Py_RETURN_NONE;
    const at::Tensor result = at::empty({int64_t(g_result_bytes)}, on(at::Device(at::kCUDA), at::kByte));
    void *const s = stream(), *const r = result.data_ptr();
    auto* const st = status ? static_cast<uint32_t*>(status->data_ptr()) : nullptr;
    const void *const c = cands->data_ptr(), *const l = law->data_ptr(), *const p = proposal->data_ptr();
    if (!done([&] { return g_lib.spec_accept(s, c, l, static_cast<const uint32_t*>(p), options.view.buf, seed, step, nullptr, r, st); })) return nullptr;
    return THPVariable_Wrap(result);
    GUFFIN_LEAVE
}

#define GUFFIN_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {GUFFIN_METHOD(bind), GUFFIN_METHOD(group_sums), GUFFIN_METHOD(gemv_packed), GUFFIN_METHOD(repack),
                           GUFFIN_METHOD(select_candidates), GUFFIN_METHOD(draft_law), GUFFIN_METHOD(spec_accept), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_operators", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__operators() { return PyModule_Create(&g_module); }
