// Host side of the hot ops in C++: argument checks, output allocation and
// launch of one op per call, without the interpreter's share (a Python op of
// _CUDA.py spends 12-15 us on argument checks, tensor allocations, views, the
// stream lookup and ctypes, the launch itself about 3 us of it; here 5.5 us in
// all.  A QLinear module of M = 16, K = N = 4096, whose two kernels take 12 us:
// 38 -> 16 us a call).
//
// Every function returns the op's outputs, or None for any argument that it
// does not take as it stands (another dtype, device or shape, a view that is
// not contiguous, a tensor subclass with its own dispatch, an argument that
// the library refuses): the Python op then goes through its own checks, which
// name what is wrong, so the set of accepted calls and the errors are the
// Python ops' own.  None means that nothing was launched: a failed launch is
// raised here, as the Python op raises it (the kernel may have run, and an
// in-place residual must not be added twice).  Outputs come from torch's
// caching allocator, launches go to the current stream of the tensors' device,
// nothing synchronises.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <initializer_list>

#include "../../include/signrot_hip.h"

namespace {

struct Bad {};     // an argument this file does not take
struct Raised {};  // a Python exception is set

// the interpreter lock is not held while allocating and launching
struct NoGil {
    PyThreadState *s;
    NoGil() : s(PyEval_SaveThread()) {}
    ~NoGil() { PyEval_RestoreThread(s); }
};

// a torch.Tensor or Parameter itself: a subclass may see every attribute and
// call that the Python op makes of it
const at::Tensor &plain(PyObject *o, at::ScalarType dt) {
    if (!THPVariable_CheckExact(o)) throw Bad();
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != dt ||
        !t.has_storage() || !t.is_contiguous() || t.is_neg() || t.is_conj() ||
        t.key_set().has(c10::DispatchKey::Python) ||
        t.key_set().has(c10::DispatchKey::FuncTorchBatched) ||
        t.key_set().has(c10::DispatchKey::Functionalize))
        throw Bad();
    return t;
}

// an argument that may be None: its data pointer or null
void *opt_ptr(PyObject *o, at::ScalarType dt, int64_t numel, at::Device dev) {
    if (o == Py_None) return nullptr;
    const at::Tensor &t = plain(o, dt);
    if (t.numel() != numel || t.device() != dev) throw Bad();
    return t.data_ptr();
}

void *ptr(PyObject *o, at::ScalarType dt, int64_t numel, at::Device dev) {
    if (o == Py_None) throw Bad();
    return opt_ptr(o, dt, numel, dev);
}

int64_t as_int(PyObject *o) {
    if (!PyLong_CheckExact(o)) throw Bad();
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        throw Bad();
    }
    return v;
}

float as_float(PyObject *o) {
    if (PyFloat_CheckExact(o)) return (float)PyFloat_AS_DOUBLE(o);
    return (float)as_int(o);
}

bool as_bool(PyObject *o) {
    if (!PyBool_Check(o)) throw Bad();
    return o == Py_True;
}

void *stream_of(at::Device dev) {
    return (void *)c10::hip::getCurrentHIPStream(dev.index()).stream();
}

at::Tensor alloc(at::IntArrayRef sizes, at::ScalarType dt, at::Device dev) {
    return at::empty(sizes, at::TensorOptions().dtype(dt).device(dev));
}

c10::SmallVector<int64_t, 6> with_last(const at::Tensor &x, int64_t last) {
    c10::SmallVector<int64_t, 6> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return s;
}

// The library's answer: nothing for success, Bad for arguments that it refuses
// (its entry points check them before any launch), else the exception that
// _native.call raises.
void check(int rc, const char *entry) {
    if (rc == SRQ_OK) return;
    if (rc == SRQ_EINVAL || rc == SRQ_EUNSUPPORTED) throw Bad();
    PyObject *mod = PyImport_ImportModule("signrot_amd._native");
    PyObject *type = mod ? PyObject_GetAttrString(mod, "NativeError") : nullptr;
    if (type) PyErr_Format(type, "%s failed (%d): %s", entry, rc, srq_last_error());
    Py_XDECREF(type);
    Py_XDECREF(mod);
    throw Raised();
}

// The outputs of an op that has run: an error in here is raised.
PyObject *wrap(std::initializer_list<at::Tensor> ts) {
    PyObject *r = nullptr;
    try {
        if (ts.size() == 1) return THPVariable_Wrap(*ts.begin());
        r = PyTuple_New((Py_ssize_t)ts.size());
        if (!r) throw Raised();
        Py_ssize_t i = 0;
        for (const at::Tensor &t : ts) {
            PyObject *o = THPVariable_Wrap(t);
            if (!o) throw Raised();
            PyTuple_SET_ITEM(r, i++, o);
        }
        return r;
    } catch (...) {
        Py_XDECREF(r);
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "srq_host: output not wrapped");
        throw Raised();
    }
}

// Runs one op's body; anything it does not take becomes None.
template <typename F>
PyObject *guarded(Py_ssize_t have, Py_ssize_t want, F body) {
    try {
        if (have != want) throw Bad();
        return body();
    } catch (const Raised &) {
        return nullptr;
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

constexpr auto kU8 = at::kByte, kI8 = at::kChar, kI32 = at::kInt, kF16 = at::kHalf,
               kF32 = at::kFloat;

// x [..., n] as rows of n >= 2 (n even)
const at::Tensor &rows_of(PyObject *o, int64_t &rows, int64_t &n) {
    const at::Tensor &x = plain(o, kF16);
    if (x.dim() < 1) throw Bad();
    n = x.size(-1);
    if (n < 2 || n % 2 || x.numel() == 0) throw Bad();
    rows = x.numel() / n;
    return x;
}

void *had_table(PyObject *hadK, int64_t K, bool f32, at::Device dev) {
    if (K <= 1) return opt_ptr(hadK, f32 ? kF32 : kF16, K * K, dev);
    const at::Tensor &h = plain(hadK, f32 ? kF32 : kF16);
    if (h.dim() < 2 || h.size(-1) != K || h.size(-2) != K || h.numel() != K * K ||
        h.device() != dev)
        throw Bad();
    return h.data_ptr();
}

// had_sign_quant(x, hadK, K, sign, clip_ratio, fp32_had) -> (q, scale)
PyObject *had_sign_quant(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 6, [&]() -> PyObject * {
        int64_t rows, n;
        const at::Tensor &x = rows_of(a[0], rows, n);
        const at::Device dev = x.device();
        const int64_t K = as_int(a[2]);
        const bool f32 = as_bool(a[5]);
        void *h = had_table(a[1], K, f32, dev), *s = opt_ptr(a[3], kI8, n, dev);
        const float clip = as_float(a[4]);
        at::Tensor q, sc;
        int rc;
        {
            NoGil nogil;
            q = alloc(with_last(x, n / 2), kU8, dev);
            sc = alloc(with_last(x, 1), kF16, dev);
            rc = srq_had_sign_quant(x.data_ptr(), rows, n, K, h, (const int8_t *)s, f32 ? 1 : 0,
                                    clip, q.data_ptr(), sc.data_ptr(), stream_of(dev));
        }
        check(rc, "srq_had_sign_quant");
        return wrap({q, sc});
    });
}

// had_sign_asym_quant(x, hadK, K, sign, clip_ratio, int8_zero) -> (q, scale, zero)
PyObject *had_sign_asym_quant(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 6, [&]() -> PyObject * {
        int64_t rows, n;
        const at::Tensor &x = rows_of(a[0], rows, n);
        const at::Device dev = x.device();
        const int64_t K = as_int(a[2]);
        void *h = had_table(a[1], K, false, dev), *s = opt_ptr(a[3], kI8, n, dev);
        const float clip = as_float(a[4]);
        const bool i8 = as_bool(a[5]);
        at::Tensor q, sc, z;
        int rc;
        {
            NoGil nogil;
            q = alloc(with_last(x, n / 2), kU8, dev);
            sc = alloc(with_last(x, 1), kF16, dev);
            z = alloc(with_last(x, 1), i8 ? kI8 : kF16, dev);
            rc = i8 ? srq_had_sign_asym_quant_i8(x.data_ptr(), rows, n, K, h, (const int8_t *)s,
                                                 clip, q.data_ptr(), sc.data_ptr(),
                                                 (int8_t *)z.data_ptr(), stream_of(dev))
                    : srq_had_sign_asym_quant(x.data_ptr(), rows, n, K, h, (const int8_t *)s,
                                              clip, q.data_ptr(), sc.data_ptr(), z.data_ptr(),
                                              stream_of(dev));
        }
        check(rc, i8 ? "srq_had_sign_asym_quant_i8" : "srq_had_sign_asym_quant");
        return wrap({q, sc, z});
    });
}

// sym_quant_dynamic(x, clip_ratio, ndim) -> (q [..., n / 2], scale [..., 1]);
// ndim: the dimensions x must have, 0 for any
PyObject *sym_quant_dynamic(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 3, [&]() -> PyObject * {
        int64_t rows, n;
        const at::Tensor &x = rows_of(a[0], rows, n);
        const int64_t ndim = as_int(a[2]);
        if (ndim && x.dim() != ndim) throw Bad();
        const at::Device dev = x.device();
        const float clip = as_float(a[1]);
        at::Tensor q, sc;
        int rc;
        {
            NoGil nogil;
            q = alloc(with_last(x, n / 2), kU8, dev);
            sc = alloc(with_last(x, 1), kF16, dev);
            rc = srq_sym_quant_dynamic(x.data_ptr(), rows, n, clip, q.data_ptr(), sc.data_ptr(),
                                       stream_of(dev));
        }
        check(rc, "srq_sym_quant_dynamic");
        return wrap({q, sc});
    });
}

// rmsnorm_quant(x, eps, mean_dim, clip_ratio) -> (q, scale)
PyObject *rmsnorm_quant(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 4, [&]() -> PyObject * {
        int64_t rows, n;
        const at::Tensor &x = rows_of(a[0], rows, n);
        const at::Device dev = x.device();
        const float eps = as_float(a[1]), clip = as_float(a[3]);
        const int64_t mean_dim = as_int(a[2]);
        at::Tensor q, sc;
        int rc;
        {
            NoGil nogil;
            q = alloc(with_last(x, n / 2), kU8, dev);
            sc = alloc(with_last(x, 1), kF16, dev);
            rc = srq_rmsnorm_quant(x.data_ptr(), rows, n, eps, mean_dim, clip, nullptr,
                                   q.data_ptr(), sc.data_ptr(), stream_of(dev));
        }
        check(rc, "srq_rmsnorm_quant");
        return wrap({q, sc});
    });
}

// head_had_quant(x [B, H, D], scale, clip_ratio) -> (q [B, H D / 2], scale [B, 1])
PyObject *head_had_quant(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 3, [&]() -> PyObject * {
        const at::Tensor &x = plain(a[0], kF16);
        if (x.dim() != 3 || x.numel() == 0) throw Bad();
        const at::Device dev = x.device();
        const int64_t B = x.size(0), H = x.size(1), D = x.size(2);
        const float scale = as_float(a[1]), clip = as_float(a[2]);
        at::Tensor q, sc;
        int rc;
        {
            NoGil nogil;
            q = alloc({B, H * D / 2}, kU8, dev);
            sc = alloc({B, 1}, kF16, dev);
            rc = srq_head_had_quant(x.data_ptr(), B, H, D, scale, clip, q.data_ptr(),
                                    sc.data_ptr(), nullptr, stream_of(dev));
        }
        check(rc, "srq_head_had_quant");
        return wrap({q, sc});
    });
}

// the packed operands of a linear: A [..., K / 2], B [N, K / 2]
struct Operands {
    const at::Tensor &A, &B;
    int64_t M, N, K;
    at::Device dev;
    Operands(PyObject *a, PyObject *b) : A(plain(a, kU8)), B(plain(b, kU8)), dev(A.device()) {
        if (A.dim() < 1 || B.dim() != 2 || A.numel() == 0 || B.numel() == 0 ||
            A.size(-1) != B.size(1) || B.device() != dev)
            throw Bad();
        K = B.size(1) * 2;
        N = B.size(0);
        M = A.numel() / B.size(1);
    }
};

// w4a4_linear(A, a_scale, B, b_scale, bias, ndim) -> out [..., N]; scales and
// bias of any shape with M and N elements; ndim: A's dimensions, 0 for any
PyObject *w4a4_linear(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 6, [&]() -> PyObject * {
        const Operands o(a[0], a[2]);
        const int64_t ndim = as_int(a[5]);
        if (ndim && o.A.dim() != ndim) throw Bad();
        void *sa = ptr(a[1], kF16, o.M, o.dev), *sb = ptr(a[3], kF16, o.N, o.dev);
        void *bias = opt_ptr(a[4], kF16, o.N, o.dev);
        at::Tensor out, ws;
        int rc;
        {
            NoGil nogil;
            out = alloc(with_last(o.A, o.N), kF16, o.dev);
            const int64_t wb = srq_w4a4_linear_ws_bytes(o.M, o.N, o.K);
            if (wb > 0) {
                ws = alloc({wb}, kU8, o.dev);
                rc = srq_w4a4_linear_ws(o.A.data_ptr(), sa, o.B.data_ptr(), sb, bias, o.M, o.N,
                                        o.K, out.data_ptr(), ws.data_ptr(), wb,
                                        stream_of(o.dev));
            } else {
                rc = srq_w4a4_linear(o.A.data_ptr(), sa, o.B.data_ptr(), sb, bias, o.M, o.N, o.K,
                                     out.data_ptr(), stream_of(o.dev));
            }
            ws.reset();
        }
        check(rc, "srq_w4a4_linear");
        return wrap({out});
    });
}

// w4a4_linear_residual(A, a_scale, B, b_scale, residual, bias, out or None)
PyObject *w4a4_linear_residual(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 7, [&]() -> PyObject * {
        const Operands o(a[0], a[2]);
        if (o.A.dim() != 2) throw Bad();
        void *sa = ptr(a[1], kF16, o.M, o.dev), *sb = ptr(a[3], kF16, o.N, o.dev);
        void *res = ptr(a[4], kF16, o.M * o.N, o.dev);
        void *bias = opt_ptr(a[5], kF16, o.N, o.dev);
        void *given = opt_ptr(a[6], kF16, o.M * o.N, o.dev);
        at::Tensor out, ws;
        int rc;
        {
            NoGil nogil;
            if (!given) out = alloc({o.M, o.N}, kF16, o.dev);
            void *dst = given ? given : out.data_ptr();
            const int64_t wb = srq_w4a4_linear_ws_bytes(o.M, o.N, o.K);
            if (wb > 0) {
                ws = alloc({wb}, kU8, o.dev);
                rc = srq_w4a4_linear_residual_ws(o.A.data_ptr(), sa, o.B.data_ptr(), sb, bias,
                                                 res, o.M, o.N, o.K, dst, ws.data_ptr(), wb,
                                                 stream_of(o.dev));
            } else {
                rc = srq_w4a4_linear_residual(o.A.data_ptr(), sa, o.B.data_ptr(), sb, bias, res,
                                              o.M, o.N, o.K, dst, stream_of(o.dev));
            }
            ws.reset();
        }
        check(rc, "srq_w4a4_linear_residual");
        if (given) {
            Py_INCREF(a[6]);
            return a[6];
        }
        return wrap({out});
    });
}

// w4a4_linear_asym(A, a_scale, a_zero, B, b_scale, b_sum, bias, ndim) -> out [..., N]
PyObject *w4a4_linear_asym(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 8, [&]() -> PyObject * {
        const Operands o(a[0], a[3]);
        const int64_t ndim = as_int(a[7]);
        if (ndim && o.A.dim() != ndim) throw Bad();
        void *sa = ptr(a[1], kF16, o.M, o.dev), *za = ptr(a[2], kI8, o.M, o.dev);
        void *sb = ptr(a[4], kF16, o.N, o.dev), *wsum = ptr(a[5], kI32, o.N, o.dev);
        void *bias = opt_ptr(a[6], kF16, o.N, o.dev);
        at::Tensor out, ws;
        int rc;
        {
            NoGil nogil;
            out = alloc(with_last(o.A, o.N), kF16, o.dev);
            int64_t wb = 0;
            srq_w4a4_linear_asym_ws_bytes(o.M, o.N, o.K, &wb);
            if (wb > 0) ws = alloc({wb}, kU8, o.dev);
            rc = srq_w4a4_linear_asym_ws(o.A.data_ptr(), sa, (const int8_t *)za, o.B.data_ptr(),
                                         sb, (const int32_t *)wsum, bias, o.M, o.N, o.K,
                                         out.data_ptr(), wb > 0 ? ws.data_ptr() : nullptr,
                                         wb > 0 ? wb : 0, stream_of(o.dev));
            ws.reset();
        }
        check(rc, "srq_w4a4_linear_asym");
        return wrap({out});
    });
}

// w4a4_linear_swiglu(A, a_scale, B_il, b_scale_il) -> out [M, N / 2]
PyObject *w4a4_linear_swiglu(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 4, [&]() -> PyObject * {
        const Operands o(a[0], a[2]);
        if (o.A.dim() != 2) throw Bad();
        void *sa = ptr(a[1], kF16, o.M, o.dev), *sb = ptr(a[3], kF16, o.N, o.dev);
        at::Tensor out;
        int rc;
        {
            NoGil nogil;
            out = alloc({o.M, o.N / 2}, kF16, o.dev);
            rc = srq_w4a4_linear_swiglu(o.A.data_ptr(), sa, o.B.data_ptr(), sb, o.M, o.N, o.K,
                                        out.data_ptr(), stream_of(o.dev));
        }
        check(rc, "srq_w4a4_linear_swiglu");
        return wrap({out});
    });
}

// stream(t): the current stream of the tensor's device, as an address
PyObject *stream(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    return guarded(n_args, 1, [&]() -> PyObject * {
        if (!THPVariable_Check(a[0])) throw Bad();
        const at::Tensor &t = THPVariable_Unpack(a[0]);
        if (!t.is_cuda()) throw Bad();
        return PyLong_FromVoidPtr(stream_of(t.device()));
    });
}

#define OP(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {OP(had_sign_quant),       OP(had_sign_asym_quant),
                          OP(sym_quant_dynamic),    OP(rmsnorm_quant),
                          OP(head_had_quant),       OP(w4a4_linear),
                          OP(w4a4_linear_residual), OP(w4a4_linear_asym),
                          OP(w4a4_linear_swiglu),   OP(stream),
                          {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "srq_host",
                       "Checks, allocation and launch of the hot ops (None: the Python op's own "
                       "path takes the call).",
                       -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_srq_host() { return PyModule_Create(&kModule); }
