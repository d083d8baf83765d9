// Python extension module _fo_native: the per-call host path of ops.py and layers.py.
//
// The small calls of this framework are bound by the host: a kernel launch costs 2.7 us or more, and the checks, pointer
// objects and stream lookup of a call written in Python another 5 to 9.  Host time per call, before and with this module:
// the two layers of a decode step (128x4096x1024, whose kernels run 8.5 us) 17.3 -> 11.1 us, the all-reduce call
// 9.6 -> 4.0, the same with the normalisation 13.9 -> 6.8, the normalisation alone 9.3 -> 3.6.  Each function here does what its Python counterpart does
// for the arguments of an ordinary call: the same checks, then one call of the C ABI.  Whatever it does not
// recognise or its checks would refuse it leaves alone: it returns None without having called the C ABI, and the
// caller takes its Python path, which raises the proper error or handles the unusual argument.
//
// Functions that enqueue return the C ABI's error code; the layer functions return the output tensor, and raise what
// the C ABI refuses: a second call by another path could enqueue twice.
#include <ATen/ATen.h>
#include <ATen/ops/empty_native.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>

#include <algorithm>

#include "flashoverlap.h"

namespace {

// One argument list, read from left to right; `ok` stays true while every argument is of the expected kind.
struct Args {
    PyObject *const *a;
    Py_ssize_t n, i = 0;
    bool ok = true;

    PyObject *next() {
        if (i >= n) {
            ok = false;
            return Py_None;
        }
        return a[i++];
    }
    const at::Tensor *tensor() {
        PyObject *o = next();
        if (!THPVariable_Check(o)) {
            ok = false;
            return nullptr;
        }
        const at::Tensor &t = THPVariable_Unpack(o);
        // tensors that Python code dispatches on (fake tensors, wrapper subclasses) have no memory to point at
        if (!t.defined() || t.key_set().has(c10::DispatchKey::Python) || !t.has_storage()) ok = false;
        return &t;
    }
    // A tensor of no class but torch's own: what the other path makes of a subclass (its results' class, its hooks) stays with it.
    const at::Tensor *plain_tensor() {
        if (i < n && !THPVariable_CheckExact(a[i])) ok = false;
        return tensor();
    }
    const at::Tensor *tensor_or_none() {
        if (i < n && a[i] == Py_None) {
            i++;
            return nullptr;
        }
        return tensor();
    }
    int64_t integer() {
        PyObject *o = next();
        if (!PyLong_Check(o)) {
            ok = false;
            return 0;
        }
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow) ok = false;
        return v;
    }
    int int32() {
        const int64_t v = integer();
        if (v != (int32_t)v) ok = false;
        return (int)v;
    }
    void *pointer() {
        PyObject *o = next();
        if (!PyLong_Check(o)) {
            ok = false;
            return nullptr;
        }
        void *p = PyLong_AsVoidPtr(o);
        if (!p) {
            PyErr_Clear();
            ok = false;
        }
        return p;
    }
    double real() {
        PyObject *o = next();
        if (!PyFloat_Check(o)) ok = false;
        return ok ? PyFloat_AS_DOUBLE(o) : 0.0;
    }
    bool done() const { return ok && i == n; }
};

bool value_type(const at::Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
int dtype_of(const at::Tensor &t) { return t.scalar_type() == at::kHalf ? FO_F16 : FO_BF16; }
bool on_gpu(const at::Tensor &t) { return t.is_cuda() && t.is_contiguous(); }
bool values(const at::Tensor &t, const at::Tensor &like) { return t.scalar_type() == like.scalar_type() && on_gpu(t); }
bool gpu_ints(const at::Tensor &t) { return t.scalar_type() == at::kInt && on_gpu(t); }
bool host_ints(const at::Tensor &t) { return t.scalar_type() == at::kInt && t.is_cpu() && t.is_contiguous(); }
int32_t *ints(const at::Tensor &t) { return static_cast<int32_t *>(t.data_ptr()); }
fo_stream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The C ABI call, other Python threads running meanwhile (a launch waits while the hardware queue is full).
template <typename F>
int enqueue(F f) {
    PyThreadState *state = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(state);
    return rc;
}

struct Product {
    int M = 0, N = 0, K = 0;
    bool fits(const at::Tensor &A, const at::Tensor &B) {
        if (A.dim() != 2 || B.dim() != 2 || A.size(1) != B.size(1) || !value_type(A) || !on_gpu(A) || !values(B, A)) return false;
        const int64_t m = A.size(0), n = B.size(0), k = A.size(1);
        M = (int)m, N = (int)n, K = (int)k;
        return m == M && n == N && k == K && M > 0 && N > 0 && K > 0;
    }
    int64_t elems() const { return (int64_t)M * N; }
};

// The buffers an overlapped call indexes by tile, group and row (ops._check_signal_buffers).
struct Schedule {
    const at::Tensor *MM, *RA, *cseg_cpu, *cseg_gpu;
    int rLDN = 1, algo = 0;
    bool monitor = false;
    int tile_n = 0;

    bool fits(const Product &p, const at::Tensor *RE, const at::Tensor *D, int64_t W) {
        int32_t info[12];
        if (fo_algo_info(algo, info) || p.M % info[0] || p.N % info[1]) return false;
        tile_n = info[1];
        const int64_t TM = p.M / info[0], TN = p.N / info[1], G = cseg_gpu->numel();
        if (!gpu_ints(*MM) || !gpu_ints(*RA) || !host_ints(*cseg_cpu) || !gpu_ints(*cseg_gpu)) return false;
        if (RA->dim() != 2 || RA->size(0) != TM || RA->size(1) != TN || cseg_cpu->numel() != G) return false;
        if (MM->numel() < (monitor ? (TM + 1) * TN : std::max(G, TN))) return false;
        if (rLDN <= 0 || (TM * TN) % rLDN) return false;
        if (RE && (!gpu_ints(*RE) || RE->numel() < p.elems() / ((int64_t)rLDN * tile_n))) return false;
        return !D || (W > 0 && D->numel() >= p.elems() / W);
    }
    int TM() const { return (int)RA->size(0); }
    int TN() const { return (int)RA->size(1); }
    int G() const { return (int)cseg_gpu->numel(); }
};

bool acc_fits(const at::Tensor *acc, const Product &p, const at::Tensor &A) {
    return !acc || (acc->scalar_type() == A.scalar_type() && acc->numel() >= p.elems());
}

// allreduce(handle, A, B, C, MM, RA, rLDN, cSEG_CPU, cSEG_GPU, algo, monitor, acc | None)
PyObject *allreduce(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    fo_overlap_t *h = static_cast<fo_overlap_t *>(in.pointer());
    const at::Tensor *A = in.tensor(), *B = in.tensor(), *C = in.tensor();
    Schedule s;
    s.MM = in.tensor(), s.RA = in.tensor(), s.rLDN = in.int32();
    s.cseg_cpu = in.tensor(), s.cseg_gpu = in.tensor(), s.algo = in.int32(), s.monitor = in.integer() != 0;
    const at::Tensor *acc = in.tensor_or_none();
    Product p;
    if (!in.done() || !p.fits(*A, *B) || !values(*C, *A) || C->numel() != p.elems() || !s.fits(p, nullptr, nullptr, 1) ||
        !acc_fits(acc, p, *A))
        Py_RETURN_NONE;
    return PyLong_FromLong(enqueue([&] {
        return fo_overlap_gemm_allreduce(h, dtype_of(*A), p.M, p.N, p.K, A->data_ptr(), B->data_ptr(), C->data_ptr(), ints(*s.MM),
                                         ints(*s.RA), s.TM(), s.TN(), s.rLDN, ints(*s.cseg_cpu), ints(*s.cseg_gpu), s.G(), s.algo,
                                         s.monitor);
    }));
    END_HANDLE_TH_ERRORS
}

// allreduce_norm(handle, A, B, C, MM, RA, RA_cpu, rLDN, cSEG_CPU, cSEG_GPU, algo, monitor, acc | None, Y, weight, eps)
PyObject *allreduce_norm(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    fo_overlap_t *h = static_cast<fo_overlap_t *>(in.pointer());
    const at::Tensor *A = in.tensor(), *B = in.tensor(), *C = in.tensor();
    Schedule s;
    s.MM = in.tensor(), s.RA = in.tensor();
    const at::Tensor *RA_cpu = in.tensor();
    s.rLDN = in.int32();
    s.cseg_cpu = in.tensor(), s.cseg_gpu = in.tensor(), s.algo = in.int32(), s.monitor = in.integer() != 0;
    const at::Tensor *acc = in.tensor_or_none(), *Y = in.tensor(), *Wt = in.tensor();
    const double eps = in.real();
    Product p;
    if (!in.done() || !p.fits(*A, *B) || !values(*C, *A) || C->numel() != p.elems() || !s.fits(p, nullptr, nullptr, 1) ||
        !acc_fits(acc, p, *A) || !host_ints(*RA_cpu) || RA_cpu->numel() != s.RA->numel() || !values(*Y, *A) || !values(*Wt, *A) ||
        Y->numel() != p.elems() || Wt->numel() < p.N)
        Py_RETURN_NONE;
    return PyLong_FromLong(enqueue([&] {
        return fo_overlap_gemm_allreduce_norm(h, dtype_of(*A), p.M, p.N, p.K, A->data_ptr(), B->data_ptr(), C->data_ptr(),
                                              ints(*s.MM), ints(*s.RA), ints(*RA_cpu), s.TM(), s.TN(), s.rLDN, ints(*s.cseg_cpu),
                                              ints(*s.cseg_gpu), s.G(), s.algo, s.monitor, Y->data_ptr(), Wt->data_ptr(),
                                              (float)eps);
    }));
    END_HANDLE_TH_ERRORS
}

// reducescatter(handle, A, B, C, D, MM, RA, RE, rLDN, cSEG_CPU, cSEG_GPU, algo, monitor, acc | None, world)
PyObject *reducescatter(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    fo_overlap_t *h = static_cast<fo_overlap_t *>(in.pointer());
    const at::Tensor *A = in.tensor(), *B = in.tensor(), *C = in.tensor(), *D = in.tensor();
    Schedule s;
    s.MM = in.tensor(), s.RA = in.tensor();
    const at::Tensor *RE = in.tensor();
    s.rLDN = in.int32();
    s.cseg_cpu = in.tensor(), s.cseg_gpu = in.tensor(), s.algo = in.int32(), s.monitor = in.integer() != 0;
    const at::Tensor *acc = in.tensor_or_none();
    const int64_t W = in.integer();
    Product p;
    if (!in.done() || !p.fits(*A, *B) || !values(*C, *A) || C->numel() != p.elems() || !values(*D, *A) || !s.fits(p, RE, D, W) ||
        !acc_fits(acc, p, *A))
        Py_RETURN_NONE;
    return PyLong_FromLong(enqueue([&] {
        return fo_overlap_gemm_reducescatter(h, dtype_of(*A), p.M, p.N, p.K, A->data_ptr(), B->data_ptr(), C->data_ptr(),
                                             D->data_ptr(), ints(*s.MM), ints(*s.RA), ints(*RE), s.TM(), s.TN(), s.rLDN,
                                             ints(*s.cseg_cpu), ints(*s.cseg_gpu), s.G(), s.algo, s.monitor);
    }));
    END_HANDLE_TH_ERRORS
}

// Whether somebody follows the operators that run (a profiler or tracer, a function or dispatch mode, a transform): the
// layers then go through the registered ones.  Dispatch modes, tracers and transforms put keys of theirs among the ones
// that every dispatch includes.
bool followed() {
    return !(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() || at::hasCallbacks() ||
           at::impl::torch_function_mode_enabled();
}

bool norm_fits(const at::Tensor &X, const at::Tensor &Wt, int BM, int BN, const at::Tensor &RA) {
    if (X.dim() != 2 || !value_type(X) || !on_gpu(X) || !values(Wt, X) || Wt.numel() < X.size(1) || !gpu_ints(RA)) return false;
    const int64_t bs = X.size(0), dim = X.size(1);
    return bs == (int)bs && dim == (int)dim && BM > 0 && BN > 0 && bs % BM == 0 && dim % BN == 0 &&
           RA.numel() >= (bs / BM) * (dim / BN);
}

int norm_on_current(const at::Tensor &X, const at::Tensor &Y, const at::Tensor &Wt, int BM, int BN, int rldn, const at::Tensor &RA,
                    double eps) {
    return enqueue([&] {
        return fo_reorder_rmsnorm(dtype_of(X), X.data_ptr(), Y.data_ptr(), Wt.data_ptr(), (int)X.size(0), (int)X.size(1), BM, BN,
                                  rldn, ints(RA), (float)eps, current_stream());
    });
}

// reorder_rmsnorm(X, Y, weight, BM, BN, rldn, RA, eps), on the current stream
PyObject *reorder_rmsnorm(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    const at::Tensor *X = in.tensor(), *Y = in.tensor(), *Wt = in.tensor();
    const int BM = in.int32(), BN = in.int32(), rldn = in.int32();
    const at::Tensor *RA = in.tensor();
    const double eps = in.real();
    if (!in.done() || !norm_fits(*X, *Wt, BM, BN, *RA) || !values(*Y, *X) || Y->numel() != X->numel()) Py_RETURN_NONE;
    return PyLong_FromLong(norm_on_current(*X, *Y, *Wt, BM, BN, rldn, *RA, eps));
    END_HANDLE_TH_ERRORS
}

// An output of a layer's call: what at::empty comes to once nobody follows the operators (asked before), without its way
// through the dispatcher (host time of the two layers of a decode step, medians of runs taking turns, 11.3 -> 10.9 us).
at::Tensor output(at::IntArrayRef sizes, const at::Tensor &like) {
    return at::native::empty_cuda(sizes, like.scalar_type(), at::kStrided, like.device(), false, std::nullopt);
}

// The output of a layer's call, or the error that the registered classes and operators raise for that code.
PyObject *output_of(int rc, const char *what, const at::Tensor &t) {
    TORCH_CHECK(rc == 0, "flashoverlap: ", what, " failed: ", fo_error_string(rc), " (code ", rc, ")");
    return THPVariable_Wrap(t);
}

// allreduce_layer(handle, x, weight, counter, RA, cSEG_CPU, cSEG_GPU, algo) -> out
PyObject *allreduce_layer(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    fo_overlap_t *h = static_cast<fo_overlap_t *>(in.pointer());
    const at::Tensor *A = in.plain_tensor(), *B = in.plain_tensor();
    Schedule s;
    s.MM = in.tensor(), s.RA = in.tensor(), s.cseg_cpu = in.tensor(), s.cseg_gpu = in.tensor(), s.algo = in.int32();
    Product p;
    if (followed() || !in.done() || !p.fits(*A, *B) || !s.fits(p, nullptr, nullptr, 1)) Py_RETURN_NONE;
    const at::Tensor out = output({p.M, p.N}, *A);
    const int rc = enqueue([&] {
        return fo_overlap_gemm_allreduce(h, dtype_of(*A), p.M, p.N, p.K, A->data_ptr(), B->data_ptr(), out.data_ptr(), ints(*s.MM),
                                         ints(*s.RA), s.TM(), s.TN(), 1, ints(*s.cseg_cpu), ints(*s.cseg_gpu), s.G(), s.algo, 0);
    });
    return output_of(rc, "gemm_allreduce_overlap", out);
    END_HANDLE_TH_ERRORS
}

// reducescatter_layer(handle, x, weight, counter, RA, RE, cSEG_CPU, cSEG_GPU, algo, world) -> out
PyObject *reducescatter_layer(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    fo_overlap_t *h = static_cast<fo_overlap_t *>(in.pointer());
    const at::Tensor *A = in.plain_tensor(), *B = in.plain_tensor();
    Schedule s;
    s.MM = in.tensor(), s.RA = in.tensor();
    const at::Tensor *RE = in.tensor();
    s.cseg_cpu = in.tensor(), s.cseg_gpu = in.tensor(), s.algo = in.int32();
    const int64_t W = in.integer();
    Product p;
    if (followed() || !in.done() || !p.fits(*A, *B) || W <= 0 || p.M % W || !s.fits(p, RE, nullptr, W)) Py_RETURN_NONE;
    const at::Tensor all = output({p.M, p.N}, *A), out = output({p.M / W, p.N}, *A);
    const int rc = enqueue([&] {
        return fo_overlap_gemm_reducescatter(h, dtype_of(*A), p.M, p.N, p.K, A->data_ptr(), B->data_ptr(), all.data_ptr(),
                                             out.data_ptr(), ints(*s.MM), ints(*s.RA), ints(*RE), s.TM(), s.TN(), 1,
                                             ints(*s.cseg_cpu), ints(*s.cseg_gpu), s.G(), s.algo, 0);
    });
    return output_of(rc, "gemm_reducescatter_overlap", out);
    END_HANDLE_TH_ERRORS
}

// reorder_rmsnorm_layer(x, weight, BM, BN, RA, eps) -> out
PyObject *reorder_rmsnorm_layer(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
    HANDLE_TH_ERRORS
    Args in{argv, argc};
    const at::Tensor *X = in.plain_tensor(), *Wt = in.plain_tensor();
    const int BM = in.int32(), BN = in.int32();
    const at::Tensor *RA = in.tensor();
    const double eps = in.real();
    if (followed() || !in.done() || !norm_fits(*X, *Wt, BM, BN, *RA)) Py_RETURN_NONE;
    const at::Tensor out = output(X->sizes(), *X);
    return output_of(norm_on_current(*X, out, *Wt, BM, BN, 1, *RA, eps), "reorder_rmsnorm", out);
    END_HANDLE_TH_ERRORS
}

#define FO_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FO_METHOD(allreduce),           FO_METHOD(allreduce_norm),      FO_METHOD(reducescatter),
                         FO_METHOD(reorder_rmsnorm),     FO_METHOD(allreduce_layer),     FO_METHOD(reducescatter_layer),
                         FO_METHOD(reorder_rmsnorm_layer), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fo_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fo_native(void) { return PyModule_Create(&module); }
