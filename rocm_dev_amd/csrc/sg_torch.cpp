// Host side of the Python entry points (rocm_dev_amd/api.py), in C++: from tensors to one call of the C ABI.
//
// A decode projection takes 2-20 us on the device and its launch about 2 us on the host; the same call through Python -
// the layout checks, a device context, the current stream, ctypes - took 10-14 us, so every eager caller was bound by
// it.  Each function here does what the Python of the same name does when the operands are plain: real HIP tensors on the
// current device with the expected types, shapes and strides.  Anything else - another device, a wrong layout, a tensor
// subclass - returns None before anything is enqueued, and the Python function takes over, with its checks and its error
// messages; so the rules live there, and these functions only have to recognise the case in which none of them applies.
//
// The launch runs without the interpreter lock, as a ctypes call does.  Nothing is kept between calls.
#include <Python.h>

#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <climits>

#include "../../include/sgemm.h"

namespace {

// entry points of the libsgemm.so that the package has loaded (bind)
#define SG_ENTRIES(X)                                                                                               \
    X(sg_skinny_gemm_auto) X(sg_skinny_gemm_rowcol) X(sg_skinny_gemm_bf16act) X(sg_sparse24_gemm)                   \
    X(sg_sparse24_compress) X(sg_fp8_encode_rows) X(sg_fp8_decode_rows) X(sg_fp8_reduce_rows) X(sg_tiled_sum_reduce)
#define SG_POINTER(name) decltype(&::name) p_##name = nullptr;
SG_ENTRIES(SG_POINTER)
#undef SG_POINTER

bool fp8(at::ScalarType t) { return t == at::kByte || t == at::kFloat8_e4m3fn; }
const uint8_t* bytes(const at::Tensor& t) { return static_cast<const uint8_t*>(t.const_data_ptr()); }
constexpr bool kOptional = true;

// The operands of one call.  `plain` turns false as soon as one of them is not what the entry point takes as it is.
struct Operands {
    bool plain = true;
    int device = -1;

    // Tensor `o` of `dims` dimensions; nullptr (with plain still true) for None where that is allowed.
    const at::Tensor* tensor(PyObject* o, int dims, bool optional = false) {
        if (!plain) return nullptr;
        if (optional && o == Py_None) return nullptr;
        if (!THPVariable_Check(o)) return fail();
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.unsafeGetTensorImpl()->is_python_dispatch()) return fail();
        if (dims >= 0 && t.dim() != dims) return fail();
        if (device < 0) device = t.device().index();
        if (t.device().index() != device) return fail();
        return &t;
    }
    const at::Tensor* fail() {
        plain = false;
        return nullptr;
    }
    void need(bool ok) { plain = plain && ok; }

    const at::Tensor* row_major(PyObject* o, int dims) {
        const at::Tensor* t = tensor(o, dims);
        if (t && !t->is_contiguous()) return fail();
        return t;
    }
    // a contiguous float vector of `length` elements, or None
    const float* factors(PyObject* o, int64_t length) {
        const at::Tensor* t = tensor(o, 1, kOptional);
        if (!t) return nullptr;
        need(t->scalar_type() == at::kFloat && t->size(0) == length && t->is_contiguous());
        return plain ? static_cast<const float*>(t->const_data_ptr()) : nullptr;
    }
    // the one-word scale: any shape with an element
    const float* scale(PyObject* o, bool optional = false) {
        const at::Tensor* t = tensor(o, -1, optional);
        if (!t) return nullptr;
        need(t->scalar_type() == at::kFloat && t->numel() >= 1 && t->is_contiguous());
        return plain ? static_cast<const float*>(t->const_data_ptr()) : nullptr;
    }
    // every size the C ABI takes is an int
    int size(int64_t v) {
        need(v >= 0 && v <= INT_MAX);
        return plain ? (int)v : 0;
    }
    // row stride of a [n, columns] matrix with contiguous columns (one row: any stride will do)
    int row_stride(const at::Tensor& t) {
        const int64_t rows = t.size(0), cols = t.size(1);
        need((cols <= 1 || t.stride(1) == 1) && (rows <= 1 || t.stride(0) >= cols));
        return size(rows > 1 ? t.stride(0) : std::max(t.stride(0), cols));
    }
    // device pointers are taken on the tensor's own device, which has to be the current one
    bool ready() {
        return plain && device >= 0 && c10::hip::current_device() == device;
    }
    void* stream() const { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
};

// D [m, n] = A [m, k] x B [n, weight columns]^T
struct Gemm {
    const at::Tensor *A = nullptr, *B = nullptr, *D = nullptr;
    int m = 0, n = 0, k = 0, b_stride = 0;
    // k_per_column: k over B's columns (2 for compressed 2:4 values)
    Gemm(Operands& o, PyObject* a, PyObject* b, PyObject* d, at::ScalarType a_type, int k_per_column = 1) {
        A = o.row_major(a, 2);
        B = o.tensor(b, 2);
        D = o.row_major(d, 2);
        if (!o.plain) return;
        o.need((a_type == at::kByte ? fp8(A->scalar_type()) : A->scalar_type() == a_type) && fp8(B->scalar_type()) &&
               D->scalar_type() == at::kBFloat16);
        o.need(A->size(1) == B->size(1) * k_per_column && D->size(0) == A->size(0) && D->size(1) == B->size(0));
        m = o.size(A->size(0));
        n = o.size(B->size(0));
        k = o.size(A->size(1));
        b_stride = o.row_stride(*B);
    }
    const uint8_t* a() const { return bytes(*A); }
    const uint8_t* b() const { return bytes(*B); }
    void* d() const { return D->mutable_data_ptr(); }
};

template <class Launch>
PyObject* enqueue(Launch&& launch) {
    int rc;
    {
        struct Unlocked {      // (not the macros: an exception out of the launch must find the lock held again)
            PyThreadState* state = PyEval_SaveThread();
            ~Unlocked() { PyEval_RestoreThread(state); }
        } unlocked;
        rc = launch();
    }
    return PyLong_FromLong(rc);
}

// One entry point: `call` returns its result, or nullptr where the Python function has to take over - also by throwing (a
// tensor without storage, say).  The Python callers pass their arguments by position.
template <class Call>
PyObject* entry(Py_ssize_t got, Py_ssize_t want, Call&& call) {
    if (got != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, got);
        return nullptr;
    }
    try {
        if (PyObject* result = call()) return result;
    } catch (const std::exception&) {
    }
    Py_RETURN_NONE;
}

using Args = PyObject* const*;

// A, B, D, scale
PyObject* skinny_gemm_fastpath(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 4, [&]() -> PyObject* {
        Operands o;
        const Gemm g(o, v[0], v[1], v[2], at::kByte);
        const float* s = o.scale(v[3]);
        if (!o.ready()) return nullptr;
        const uint8_t *a = g.a(), *b = g.b();
        void *d = g.d(), *st = o.stream();
        return enqueue([&] { return p_sg_skinny_gemm_auto(a, b, d, s, g.m, g.n, g.k, g.b_stride, st); });
    });
}

// A, B, D, scale or None, row_scales or None, col_scales or None
PyObject* skinny_gemm_rowcol(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 6, [&]() -> PyObject* {
        Operands o;
        const Gemm g(o, v[0], v[1], v[2], at::kByte);
        const float* s = o.scale(v[3], kOptional);
        const float* rs = o.factors(v[4], g.m);
        const float* cs = o.factors(v[5], g.n);
        if (!o.ready()) return nullptr;
        const uint8_t *a = g.a(), *b = g.b();
        void *d = g.d(), *st = o.stream();
        return enqueue([&] { return p_sg_skinny_gemm_rowcol(a, b, d, s, rs, cs, g.m, g.n, g.k, g.b_stride, st); });
    });
}

// X, B, D, scale or None, col_scales or None, row_scales_out or None
PyObject* skinny_gemm_bf16act(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 6, [&]() -> PyObject* {
        Operands o;
        const Gemm g(o, v[0], v[1], v[2], at::kBFloat16);
        const float* s = o.scale(v[3], kOptional);
        const float* cs = o.factors(v[4], g.n);
        float* rs = const_cast<float*>(o.factors(v[5], g.m));
        if (!o.ready()) return nullptr;
        const uint8_t *a = g.a(), *b = g.b();
        void *d = g.d(), *st = o.stream();
        return enqueue([&] { return p_sg_skinny_gemm_bf16act(a, b, d, s, cs, rs, g.m, g.n, g.k, g.b_stride, st); });
    });
}

// A, vals, meta, D, scale
PyObject* sparse24_gemm(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 5, [&]() -> PyObject* {
        Operands o;
        const Gemm g(o, v[0], v[1], v[3], at::kByte, 2);
        const at::Tensor* meta = o.row_major(v[2], 2);
        const float* s = o.scale(v[4]);
        if (!o.plain) return nullptr;
        o.need(g.B->is_contiguous() && g.k % 8 == 0);
        o.need(meta->scalar_type() == at::kByte && meta->size(0) == g.n && meta->size(1) == g.k / 8);
        if (!o.ready()) return nullptr;
        const uint8_t *a = g.a(), *b = g.b(), *mt = bytes(*meta);
        void *d = g.d(), *st = o.stream();
        return enqueue([&] { return p_sg_sparse24_gemm(a, b, mt, d, s, g.m, g.n, g.k, st); });
    });
}

// B, vals, meta
PyObject* sparse24_compress(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 3, [&]() -> PyObject* {
        Operands o;
        const at::Tensor* B = o.tensor(v[0], 2);
        const at::Tensor* vals = o.row_major(v[1], 2);
        const at::Tensor* meta = o.row_major(v[2], 2);
        if (!o.plain) return nullptr;
        const int64_t rows = B->size(0), cols = B->size(1);
        o.need(fp8(B->scalar_type()) && fp8(vals->scalar_type()) && meta->scalar_type() == at::kByte && cols % 8 == 0);
        o.need(vals->size(0) == rows && vals->size(1) == cols / 2 && meta->size(0) == rows && meta->size(1) == cols / 8);
        const int b_stride = o.row_stride(*B), n = o.size(rows), k = o.size(cols);
        if (!o.ready()) return nullptr;
        const uint8_t* b = bytes(*B);
        uint8_t *va = static_cast<uint8_t*>(vals->mutable_data_ptr()), *mt = static_cast<uint8_t*>(meta->mutable_data_ptr());
        void* st = o.stream();
        return enqueue([&] { return p_sg_sparse24_compress(b, va, mt, n, k, b_stride, st); });
    });
}

// The bf16 matrix [rows, cols], its codes and its row scales ([nbuf, rows, cols] and [nbuf, rows] with buffers)
struct Codec {
    const at::Tensor *X = nullptr, *Q = nullptr, *S = nullptr;
    int rows = 0, cols = 0, nbuf = 1;
    Codec(Operands& o, PyObject* x, PyObject* q, PyObject* s, bool buffers) {
        X = o.row_major(x, 2);
        Q = o.row_major(q, buffers ? 3 : 2);
        S = o.row_major(s, buffers ? 2 : 1);
        if (!o.plain) return;
        const int b = buffers ? 1 : 0;
        o.need(X->scalar_type() == at::kBFloat16 && fp8(Q->scalar_type()) && S->scalar_type() == at::kFloat);
        o.need(Q->size(b) == X->size(0) && Q->size(b + 1) == X->size(1) && S->size(b) == X->size(0));
        if (buffers) {
            o.need(S->size(0) == Q->size(0));
            nbuf = o.size(Q->size(0));
        }
        rows = o.size(X->size(0));
        cols = o.size(X->size(1));
    }
};

// X, Q, scales
PyObject* fp8_encode_rows(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 3, [&]() -> PyObject* {
        Operands o;
        const Codec c(o, v[0], v[1], v[2], false);
        if (!o.ready()) return nullptr;
        const void* x = c.X->const_data_ptr();
        uint8_t* q = static_cast<uint8_t*>(c.Q->mutable_data_ptr());
        float* s = static_cast<float*>(c.S->mutable_data_ptr());
        void* st = o.stream();
        return enqueue([&] { return p_sg_fp8_encode_rows(x, q, s, c.rows, c.cols, st); });
    });
}

// Q, scales, Y
PyObject* fp8_decode_rows(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 3, [&]() -> PyObject* {
        Operands o;
        const Codec c(o, v[2], v[0], v[1], false);
        if (!o.ready()) return nullptr;
        const uint8_t* q = bytes(*c.Q);
        const float* s = static_cast<const float*>(c.S->const_data_ptr());
        void *y = c.X->mutable_data_ptr(), *st = o.stream();
        return enqueue([&] { return p_sg_fp8_decode_rows(q, s, y, c.rows, c.cols, st); });
    });
}

// Q, scales, Y
PyObject* fp8_reduce_rows(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 3, [&]() -> PyObject* {
        Operands o;
        const Codec c(o, v[2], v[0], v[1], true);
        if (!o.ready()) return nullptr;
        const uint8_t* q = bytes(*c.Q);
        const float* s = static_cast<const float*>(c.S->const_data_ptr());
        void *y = c.X->mutable_data_ptr(), *st = o.stream();
        const size_t stride = (size_t)c.Q->stride(0);
        return enqueue([&] { return p_sg_fp8_reduce_rows(q, s, y, c.nbuf, stride, c.rows, c.cols, st); });
    });
}

// A, B, D
PyObject* tiled_sum_reduce(PyObject*, Args v, Py_ssize_t nargs) {
    return entry(nargs, 3, [&]() -> PyObject* {
        Operands o;
        const at::Tensor* A = o.row_major(v[0], 3);
        const at::Tensor* B = o.row_major(v[1], 3);
        const at::Tensor* D = o.row_major(v[2], 2);
        if (!o.plain) return nullptr;
        o.need(A->scalar_type() == at::kFloat && B->scalar_type() == at::kFloat && D->scalar_type() == at::kFloat);
        o.need(B->sizes() == A->sizes() && D->size(0) == A->size(1) && D->size(1) == A->size(2));
        const int b = o.size(A->size(0)), m = o.size(A->size(1)), n = o.size(A->size(2));
        if (!o.ready()) return nullptr;
        const float *pa = static_cast<const float*>(A->const_data_ptr()), *pb = static_cast<const float*>(B->const_data_ptr());
        float* pd = static_cast<float*>(D->mutable_data_ptr());
        void* st = o.stream();
        return enqueue([&] { return p_sg_tiled_sum_reduce(pa, pb, pd, b, m, n, st); });
    });
}

// bind(handle of libsgemm.so)
PyObject* bind(PyObject*, PyObject* arg) {
    void* handle = PyLong_AsVoidPtr(arg);
    if (PyErr_Occurred()) return nullptr;
#define SG_RESOLVE(name)                                                                    \
    p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(handle, #name));                  \
    if (!p_##name) {                                                                        \
        PyErr_SetString(PyExc_ImportError, "libsgemm.so has no " #name ": build it again"); \
        return nullptr;                                                                     \
    }
    SG_ENTRIES(SG_RESOLVE)
#undef SG_RESOLVE
    Py_RETURN_NONE;
}

#define SG_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         SG_METHOD(skinny_gemm_fastpath),
                         SG_METHOD(skinny_gemm_rowcol),
                         SG_METHOD(skinny_gemm_bf16act),
                         SG_METHOD(sparse24_gemm),
                         SG_METHOD(sparse24_compress),
                         SG_METHOD(fp8_encode_rows),
                         SG_METHOD(fp8_decode_rows),
                         SG_METHOD(fp8_reduce_rows),
                         SG_METHOD(tiled_sum_reduce),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__torch_host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", SG_TORCH_VERSION) != 0) {   // what it was built against (_lib.py)
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
