// CPython entry points of the three calls a program makes per BitLinear -- BitLinearKernel.forward,
// bitnet_int8xint2_linear and quant_input (gpu/model.py:21-75 of the reference) -- and of the weight
// layout converters (gpu/pack_weight.py), between torch tensors and the C ABI of libbitlinear_hip.so; and the wait
// for a decode step's tokens (await_words).
//
// What bounds a small call is the host: the kernels of a one-token 2560 x 2560 forward take 3.5 us,
// and issuing them from Python (three torch.empty, torch.cuda.current_stream, the argument checks
// and the conversion of twelve ctypes arguments) took 15.4 us per call, back to back; from here it
// takes 5.5 (8 tokens of 6912 -> 2560: 18.1 -> 8.8 as two kernels, 6.9 as one).  The checks read the tensors' C++
// objects, the workspaces are one caching-allocator block, the output is allocated without the
// operator dispatcher, and the stream is read from torch's own thread-local state.  The functions
// of the library are taken by address (bind), so this file links to torch only and serves
// whichever libbitlinear_hip.so was opened.
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <chrono>
#include <cstdint>
#include <mutex>
#include <vector>

namespace {

typedef void (*product_fn)(int8_t*, int8_t*, uint16_t*, uint16_t*, uint16_t*, int, int, int, void*);
typedef int (*status_fn)();
typedef const char* (*status_string_fn)(int);
typedef int (*ws_num_fn)(int, int);
typedef int (*quant_fn)(const void*, void*, void*, int, int, int, void*);
typedef int (*forward_fn)(const void*, const void*, void*, const void*, void*, void*, int, int, int, int, void*);
typedef int (*forward_seg_fn)(const void*, const void*, void*, const void*, const int*, int, void*, void*, int, int, int, int,
                              void*);
typedef int (*pack_fn)(const void*, void*, void*, int, int, void*);
typedef int (*unpack_fn)(const void*, void*, int, int, void*);

struct Bound {
    product_fn product = nullptr;
    status_fn last_status = nullptr;
    status_string_fn status_string = nullptr;
    ws_num_fn ws_num = nullptr;
    quant_fn quant = nullptr;
    forward_fn forward = nullptr;
    forward_seg_fn forward_seg = nullptr;
    pack_fn pack = nullptr;
    unpack_fn unpack = nullptr;
    PyObject* error = nullptr;  // BitLinearLibraryError
} g_bound;

const at::Tensor* tensor_of(PyObject* o) {
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "bitlinear: expected a tensor, got %s", Py_TYPE(o)->tp_name);
        return nullptr;
    }
    return &THPVariable_Unpack(o);
}

bool check_device(std::initializer_list<const at::Tensor*> tensors) {
    for (const at::Tensor* t : tensors) {
        if (!t->is_cuda()) {
            PyErr_SetString(PyExc_ValueError, "bitlinear: all tensors must live on the GPU (no CPU path exists)");
            return false;
        }
        if (!t->is_contiguous()) {
            PyErr_SetString(PyExc_ValueError, "bitlinear: tensors must be contiguous");
            return false;
        }
    }
    return true;
}

// rows of a [..., width] tensor; -1 with an exception set for a tensor without dimensions
int64_t flat_rows(const at::Tensor& t) {
    if (t.dim() < 1) {
        PyErr_SetString(PyExc_IndexError, "bitlinear: activations need at least one dimension");
        return -1;
    }
    int64_t m = 1;
    for (int64_t d = 0; d + 1 < t.dim(); ++d) m *= t.size(d);
    return m;
}

at::Tensor empty_like_rows(const at::Tensor& rows, int64_t width, at::ScalarType type) {
    c10::SmallVector<int64_t, 5> sizes(rows.sizes().begin(), rows.sizes().end());
    sizes.back() = width;
    return at::Tensor(at::detail::empty_cuda(sizes, type, rows.device(), std::nullopt));
}

// Addresses are taken in front of the part that runs without the interpreter lock: data_ptr() throws for a tensor without
// storage (vmap, tracing), and the checks before it pass for one.
template <class T = void>
T* address(const at::Tensor& t) {
    return static_cast<T*>(t.data_ptr());
}

// The interpreter lock is free while one of these lives, and held again behind it, an exception included
class Unlocked {
public:
    Unlocked() : state_(PyEval_SaveThread()) {}
    ~Unlocked() { PyEval_RestoreThread(state_); }
    Unlocked(const Unlocked&) = delete;

private:
    PyThreadState* state_;
};

// An int array that supports the buffer protocol, or None
class IntArray {
public:
    ~IntArray() {
        if (view_.buf) PyBuffer_Release(&view_);
    }
    bool open(PyObject* o) { return o == Py_None || PyObject_GetBuffer(o, &view_, PyBUF_SIMPLE) == 0; }
    const int* data() const { return static_cast<const int*>(view_.buf); }
    int size() const { return static_cast<int>(view_.len / static_cast<Py_ssize_t>(sizeof(int))); }

private:
    Py_buffer view_ = {};
};

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

PyObject* library_error(const char* entry, long long m, long long n, long long k, int status) {
    PyErr_Format(g_bound.error, "%s(M=%lld, N=%lld, K=%lld): status %d (%s)", entry, m, n, k, status,
                 g_bound.status_string(status));
    return nullptr;
}

bool arg_count(Py_ssize_t got, Py_ssize_t want, const char* name) {
    if (got == want) return true;
    PyErr_Format(PyExc_TypeError, "%s: expected %zd arguments, got %zd", name, want, got);
    return false;
}

// forward(input, weight, weight_scale, in_features, out_features, quant_mode, seg_ends)
// seg_ends: None, or an int array that supports the buffer protocol
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 7, "forward")) return nullptr;
    const at::Tensor *x = tensor_of(args[0]), *w = x ? tensor_of(args[1]) : nullptr, *ws = w ? tensor_of(args[2]) : nullptr;
    if (!ws || !check_device({x, w, ws})) return nullptr;
    const long long K = PyLong_AsLongLong(args[3]), N = PyLong_AsLongLong(args[4]), mode = PyLong_AsLongLong(args[5]);
    if (PyErr_Occurred()) return nullptr;
    if (x->scalar_type() != at::kBFloat16) {
        PyErr_SetString(PyExc_TypeError, "BitLinearKernel.forward expects bfloat16 activations");
        return nullptr;
    }
    const int64_t M = flat_rows(*x);
    if (M < 0) return nullptr;
    if (x->size(-1) != K) {
        PyErr_Format(PyExc_ValueError, "activation width %lld does not match in_features=%lld", (long long)x->size(-1), K);
        return nullptr;
    }
    if (w->dim() != 2 || w->size(0) != N || w->size(1) != K / 4 || w->scalar_type() != at::kChar) {
        PyErr_SetString(PyExc_ValueError, "weight must be int8 [out_features, in_features // 4] (the packed layout)");
        return nullptr;
    }
    const void *px = M ? address(*x) : nullptr, *pw = M ? address(*w) : nullptr, *pws = M ? address(*ws) : nullptr;
    const c10::DeviceGuard guard(x->device());
    at::Tensor out = empty_like_rows(*x, N, at::kBFloat16);
    if (M == 0) return THPVariable_Wrap(std::move(out));
    void* po = address(out);
    IntArray seg;
    if (!seg.open(args[6])) return nullptr;
    // the quantized rows and, behind them, their scales: one block that goes back to the allocator on return, as
    // tensors do (reused by later work on the same stream)
    const size_t q_bytes = ((size_t)M * (size_t)K + 255) & ~(size_t)255;
    int st = 0;
    {
        const c10::DataPtr block = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get()->allocate(q_bytes + 2 * (size_t)M);
        char* q = (char*)block.get();
        void* stream = current_stream();
        const Unlocked unlocked;
        st = seg.data() ? g_bound.forward_seg(px, pw, po, pws, seg.data(), seg.size(), q, q + q_bytes, (int)M, (int)N, (int)K,
                                              (int)mode, stream)
                        : g_bound.forward(px, pw, po, pws, q, q + q_bytes, (int)M, (int)N, (int)K, (int)mode, stream);
    }
    if (st) return library_error(seg.data() ? "bitlinear_forward_bf16_seg" : "bitlinear_forward_bf16", M, N, K, st);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// linear(input0, input1, s, ws, out)  -- out: a tensor or None
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 5, "linear")) return nullptr;
    const at::Tensor *a = tensor_of(args[0]), *w = a ? tensor_of(args[1]) : nullptr, *s = w ? tensor_of(args[2]) : nullptr,
                     *ws = s ? tensor_of(args[3]) : nullptr;
    if (!ws || !check_device({a, w, s, ws})) return nullptr;
    if (a->scalar_type() != at::kChar || w->scalar_type() != at::kChar) {
        PyErr_SetString(PyExc_TypeError, "input0 and input1 must be int8");
        return nullptr;
    }
    if (s->scalar_type() != at::kBFloat16 || ws->scalar_type() != at::kBFloat16) {
        PyErr_SetString(PyExc_TypeError, "s and ws must be bfloat16");
        return nullptr;
    }
    const int64_t M = flat_rows(*a);
    if (M < 0) return nullptr;
    if (w->dim() < 2) {
        PyErr_SetString(PyExc_IndexError, "bitlinear: the packed weight must be [N, K/4]");
        return nullptr;
    }
    const int64_t N = w->size(0), K = w->size(1) * 4;
    if (a->size(-1) != K) {
        PyErr_Format(PyExc_ValueError, "activation width %lld does not match packed weight K=%lld", (long long)a->size(-1),
                     (long long)K);
        return nullptr;
    }
    if (s->numel() < M) {
        PyErr_Format(PyExc_ValueError, "need one activation scale per row: %lld < %lld", (long long)s->numel(), (long long)M);
        return nullptr;
    }
    if (ws->numel() < g_bound.ws_num((int)N, (int)K)) {
        PyErr_SetString(PyExc_ValueError, "weight_scale has fewer slots than this shape uses");
        return nullptr;
    }
    int8_t *pa = nullptr, *pw = nullptr;
    uint16_t *ps = nullptr, *pws = nullptr;
    if (M > 0) pa = address<int8_t>(*a), pw = address<int8_t>(*w), ps = address<uint16_t>(*s), pws = address<uint16_t>(*ws);
    const c10::DeviceGuard guard(a->device());
    at::Tensor out;
    if (args[4] == Py_None) {
        out = empty_like_rows(*a, N, at::kBFloat16);
    } else {
        const at::Tensor* o = tensor_of(args[4]);
        if (!o) return nullptr;
        if (o->scalar_type() != at::kBFloat16 || o->numel() != M * N || !o->is_contiguous() || !o->is_cuda()) {
            PyErr_SetString(PyExc_ValueError, "out must be a contiguous bfloat16 GPU tensor of M x N elements");
            return nullptr;
        }
        out = *o;
    }
    if (M > 0) {  // no token rows: nothing to launch
        void* stream = current_stream();
        uint16_t* po = address<uint16_t>(out);
        int st = 0;
        {
            const Unlocked unlocked;
            g_bound.product(pa, pw, po, ps, pws, (int)M, (int)N, (int)K, stream);
            st = g_bound.last_status();
        }
        if (st) return library_error("bitlinear_int8xint2", M, N, K, st);
    }
    if (args[4] != Py_None) {
        Py_INCREF(args[4]);
        return args[4];
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// quant(input, mode) -> (q, s)
PyObject* quant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 2, "quant")) return nullptr;
    const at::Tensor* x = tensor_of(args[0]);
    if (!x || !check_device({x})) return nullptr;
    const long long mode = PyLong_AsLongLong(args[1]);
    if (PyErr_Occurred()) return nullptr;
    if (x->scalar_type() != at::kBFloat16) {
        PyErr_SetString(PyExc_TypeError, "quant_input expects bfloat16");
        return nullptr;
    }
    const int64_t M = flat_rows(*x);
    if (M < 0) return nullptr;
    const int64_t K = x->size(-1);
    const void* px = M ? address(*x) : nullptr;
    const c10::DeviceGuard guard(x->device());
    at::Tensor q = empty_like_rows(*x, K, at::kChar), s = empty_like_rows(*x, 1, at::kBFloat16);
    if (M > 0) {
        void *stream = current_stream(), *pq = address(q), *ps = address(s);
        int st = 0;
        {
            const Unlocked unlocked;
            st = g_bound.quant(px, pq, ps, (int)M, (int)K, (int)mode, stream);
        }
        if (st) {
            PyErr_Format(g_bound.error, "bitlinear_quant_absmax(M=%lld, K=%lld): status %d (%s)", (long long)M, (long long)K,
                         st, g_bound.status_string(st));
            return nullptr;
        }
    }
    PyObject* pq = THPVariable_Wrap(std::move(q));
    PyObject* ps = pq ? THPVariable_Wrap(std::move(s)) : nullptr;
    PyObject* pair = ps ? PyTuple_Pack(2, pq, ps) : nullptr;
    Py_XDECREF(pq);
    Py_XDECREF(ps);
    return pair;
    END_HANDLE_TH_ERRORS
}

// Pinned words that a kernel can raise a flag in: reading one after the stream has got there costs no copy.  A caller
// takes a word for the length of its call; the list grows to the largest number of calls that were under way at once.
class PinnedFlag {
public:
    PinnedFlag() {
        std::lock_guard<std::mutex> hold(mutex());
        if (words().empty())
            word_ = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        else {
            word_ = std::move(words().back());
            words().pop_back();
        }
        *value() = 0;
    }
    ~PinnedFlag() {
        std::lock_guard<std::mutex> hold(mutex());
        words().push_back(std::move(word_));
    }
    volatile int32_t* value() const { return (volatile int32_t*)word_.data_ptr(); }

private:
    static std::mutex& mutex() {
        static std::mutex m;
        return m;
    }
    static std::vector<at::Tensor>& words() {  // lives until the process ends: torch's allocator may be gone before it
        static auto* w = new std::vector<at::Tensor>;
        return *w;
    }
    at::Tensor word_;
};

// pack(weight): ternary int8 [N, K] on the GPU, contiguous, N % 16 == 0 and K % 32 == 0 -> packed int8 [N, K / 4].
// Waits for the stream, since a weight outside {-1, 0, 1} is the caller's error and is reported here.
PyObject* pack(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 1, "pack")) return nullptr;
    const at::Tensor* w = tensor_of(args[0]);
    if (!w || !check_device({w})) return nullptr;
    if (w->dim() != 2 || w->scalar_type() != at::kChar) {
        PyErr_SetString(PyExc_TypeError, "pack: expected int8 [N, K]");
        return nullptr;
    }
    const int64_t N = w->size(0), K = w->size(1);
    const void* pw = address(*w);
    const c10::DeviceGuard guard(w->device());
    at::Tensor out = empty_like_rows(*w, K / 4, at::kChar);
    int st = 0;
    bool bad = false;
    {
        const PinnedFlag flag;
        const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream();
        void* po = address(out);
        const Unlocked unlocked;
        st = g_bound.pack(pw, po, (void*)flag.value(), (int)N, (int)K, (void*)stream.stream());
        if (!st) {
            stream.synchronize();
            bad = *flag.value() != 0;
        }
    }
    if (st) return library_error("bitlinear_pack_int2", 1, N, K, st);
    if (bad) {
        PyErr_SetString(PyExc_ValueError, "weights must be ternary (-1, 0, +1)");
        return nullptr;
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// unpack(packed, N, K): the inverse; packed holds N * K / 4 bytes
PyObject* unpack(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 3, "unpack")) return nullptr;
    const at::Tensor* p = tensor_of(args[0]);
    if (!p || !check_device({p})) return nullptr;
    const long long N = PyLong_AsLongLong(args[1]), K = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (p->element_size() != 1 || N < 0 || K < 0 || p->numel() * 4 != N * K) {
        PyErr_SetString(PyExc_ValueError, "unpack: expected N * K / 4 bytes");
        return nullptr;
    }
    const void* pp = address(*p);
    const c10::DeviceGuard guard(p->device());
    at::Tensor out(at::detail::empty_cuda({N, K}, at::kChar, p->device(), std::nullopt));
    void *stream = current_stream(), *po = address(out);
    int st = 0;
    {
        const Unlocked unlocked;
        st = g_bound.unpack(pp, po, (int)N, (int)K, stream);
    }
    if (st) return library_error("bitlinear_unpack_int2", 1, N, K, st);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// await_words(tensor, unset, microseconds): a contiguous int64 tensor in host memory that a kernel writes; whether all of its words
// have become another value than `unset` within that time.  Looks at the words themselves: waiting for the stream takes some 15 us more
// (a marker behind the kernel, and its signal).
PyObject* await_words(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (!arg_count(nargs, 3, "await_words")) return nullptr;
    const at::Tensor* t = tensor_of(args[0]);
    if (!t) return nullptr;
    const long long unset = PyLong_AsLongLong(args[1]), limit = PyLong_AsLongLong(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (!t->device().is_cpu() || t->scalar_type() != at::kLong || !t->is_contiguous()) {
        PyErr_SetString(PyExc_TypeError, "await_words: expected contiguous int64 words in host memory");
        return nullptr;
    }
    const volatile int64_t* word = (const volatile int64_t*)t->data_ptr();
    const int64_t count = t->numel();
    bool all = true;
    {
        const Unlocked unlocked;
        const auto end = std::chrono::steady_clock::now() + std::chrono::microseconds(limit);
        for (int64_t i = 0; all && i < count; ++i)
            for (int n = 1; word[i] == unset; ++n)
                if (n % 256 == 0 && std::chrono::steady_clock::now() > end) {
                    all = false;
                    break;
                }
        std::atomic_thread_fence(std::memory_order_acquire);
    }
    return PyBool_FromLong(all);
    END_HANDLE_TH_ERRORS
}

// bind(error_class, product, last_status, status_string, ws_num, quant, forward, forward_seg, pack, unpack): the
// library's functions by address
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (!arg_count(nargs, 10, "bind")) return nullptr;
    void* fn[9];
    for (int i = 0; i < 9; ++i) {
        fn[i] = PyLong_AsVoidPtr(args[i + 1]);
        if (!fn[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null function address");
            return nullptr;
        }
    }
    g_bound.product = (product_fn)fn[0];
    g_bound.last_status = (status_fn)fn[1];
    g_bound.status_string = (status_string_fn)fn[2];
    g_bound.ws_num = (ws_num_fn)fn[3];
    g_bound.quant = (quant_fn)fn[4];
    g_bound.forward = (forward_fn)fn[5];
    g_bound.forward_seg = (forward_seg_fn)fn[6];
    g_bound.pack = (pack_fn)fn[7];
    g_bound.unpack = (unpack_fn)fn[8];
    Py_INCREF(args[0]);
    Py_XSETREF(g_bound.error, args[0]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
    {"forward", (PyCFunction)(void*)forward, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void*)linear, METH_FASTCALL, nullptr},
    {"quant", (PyCFunction)(void*)quant, METH_FASTCALL, nullptr},
    {"pack", (PyCFunction)(void*)pack, METH_FASTCALL, nullptr},
    {"unpack", (PyCFunction)(void*)unpack, METH_FASTCALL, nullptr},
    {"await_words", (PyCFunction)(void*)await_words, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() { return PyModule_Create(&module); }
