// The Python binding's call path in C++ (module mx230_amd._binding): the
// argument checks, output allocation and marshalling of the entry points a
// program calls once per layer or token, which in Python cost more than the
// short launches they enqueue. Each function takes the common case only
// (plain torch tensors on the GPU, torch's current stream) and returns
// NotImplemented for anything else, valid or not; mx230_amd/__init__.py then
// takes its own path, which accepts the rest or raises. A non-zero status of
// the C ABI comes back as an int.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "../../include/mxfa.h"

namespace {

// The C ABI, from the libmxfa the package has loaded (bind()).
struct {
    decltype(&mxfa_run_flash_lse) flash_lse;
    decltype(&mxfa_run_bwd_ws) bwd_ws;
    decltype(&mxfa_bwd_workspace_bytes) bwd_workspace_bytes;
    decltype(&mxfa_run_prefill) prefill;
    decltype(&mxfa_run_prefill_ws) prefill_ws;
    decltype(&mxfa_run_prefill_paged) prefill_paged;
    decltype(&mxfa_run_prefill_paged_ws) prefill_paged_ws;
} abi;

PyObject *other() { Py_RETURN_NOTIMPLEMENTED; }

// The tensor of a plain torch.Tensor (or Parameter) with its own GPU storage;
// null for subclasses, functorch and Python-dispatch tensors, views with lazy
// conjugation or negation, and other devices or layouts.
const at::Tensor *plain(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    using K = c10::DispatchKey;
    static const c10::DispatchKeySet special({K::Python, K::PythonTLSSnapshot, K::FuncTorchGradWrapper,
                                              K::FuncTorchBatched, K::Functionalize, K::Conjugate, K::Negative,
                                              K::ZeroTensor, K::BatchedNestedTensor});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
        t.key_set().has_any(special) || t.unsafeGetTensorImpl()->is_python_dispatch() ||
        t.unsafeGetTensorImpl()->has_symbolic_sizes_strides())
        return nullptr;
    return &t;
}

// [N, d] or [B, H, N, d], contiguous.
bool dims(const at::Tensor &t, int64_t (&n)[4]) {
    if ((t.dim() != 2 && t.dim() != 4) || !t.is_contiguous()) return false;
    for (int i = 0; i < 4; ++i) n[i] = t.dim() == 4 ? t.size(i) : i < 2 ? 1 : t.size(i - 2);
    for (int64_t x : n) {
        if (x < 1 || x > INT32_MAX) return false;
    }
    return true;
}
bool same(const int64_t (&a)[4], const int64_t (&b)[4]) {
    return a[0] == b[0] && a[1] == b[1] && a[2] == b[2] && a[3] == b[3];
}

bool is_mxfa_type(const at::Tensor &t) {
    return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat;
}

void *current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

bool number(PyObject *o, double *v) {
    if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
    *v = PyFloat_AsDouble(o);
    return !PyErr_Occurred() || (PyErr_Clear(), false);
}
bool integer(PyObject *o, int *v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long x = PyLong_AsLongAndOverflow(o, &over);
    if (over != 0 || x < INT32_MIN || x > INT32_MAX) return false;
    *v = (int)x;
    return true;
}

// The shape of q, k, v (all of one type, K and V alike).
bool shape_of(const at::Tensor *q, const at::Tensor *k, const at::Tensor *v, PyObject *causal, PyObject *scale,
              mxfa_shape *s) {
    int64_t nq[4], nk[4], nv[4];
    double sc;
    if (!q || !k || !v || !is_mxfa_type(*q) || k->scalar_type() != q->scalar_type() ||
        v->scalar_type() != q->scalar_type() || !dims(*q, nq) || !dims(*k, nk) || !dims(*v, nv) || !same(nk, nv) ||
        nk[0] != nq[0] || nk[2] != nq[2] || nk[3] != nq[3] || !PyBool_Check(causal) || !number(scale, &sc))
        return false;
    *s = mxfa_shape{(int)nq[0], (int)nq[1], (int)nk[1], (int)nq[2], (int)nq[3], causal == Py_True,
                    q->scalar_type() == at::kBFloat16 ? MXFA_BF16 : MXFA_F32, (float)sc};
    return true;
}

PyObject *status(int rc) { return PyLong_FromLong(rc); }

// Runs f; a C++ exception becomes the Python one torch gives it (its
// OutOfMemoryError among them).
template <class F>
PyObject *guarded(F f) {
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

// attention_fwd(q, k, v, causal, scale) -> (o, lse)
PyObject *attention_fwd(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 5 || abi.flash_lse == nullptr) return other();
    return guarded([&]() -> PyObject * {
        const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
        mxfa_shape s;
        if (!shape_of(q, k, v, a[3], a[4], &s)) return other();
        at::Tensor o = at::empty_like(*q), lse = at::empty({s.B, s.Hq, s.N}, q->options().dtype(at::kFloat));
        void *stream = current_stream();
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = abi.flash_lse(&s, q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(),
                           static_cast<float *>(lse.data_ptr()), stream);
        Py_END_ALLOW_THREADS;
        if (rc != 0) return status(rc);
        return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(o)), THPVariable_Wrap(std::move(lse)));
    });
}

// attention_bwd(q, k, v, o, lse, do, causal, scale) -> (dq, dk, dv)
PyObject *attention_bwd(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 8 || abi.bwd_ws == nullptr) return other();
    return guarded([&]() -> PyObject * {
        const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]), *o = plain(a[3]), *lse = plain(a[4]),
                         *g = plain(a[5]);
        mxfa_shape s;
        if (!o || !lse || !g || !shape_of(q, k, v, a[6], a[7], &s)) return other();
        const int64_t nq[4] = {s.B, s.Hq, s.N, s.d};
        int64_t no[4], ng[4];
        if (o->scalar_type() != q->scalar_type() || g->scalar_type() != q->scalar_type() || !dims(*o, no) ||
            !dims(*g, ng) || !same(no, nq) || !same(ng, nq) || lse->scalar_type() != at::kFloat ||
            !lse->is_contiguous() || lse->numel() != (int64_t)s.B * s.Hq * s.N)
            return other();
        at::Tensor delta = at::empty({s.B, s.Hq, s.N}, q->options().dtype(at::kFloat));
        at::Tensor dq = at::empty_like(*q), dk = at::empty_like(*k), dv = at::empty_like(*v), ws;
        const size_t nws = abi.bwd_workspace_bytes(&s);
        if (nws > 0) ws = at::empty({(int64_t)nws}, q->options().dtype(at::kByte));
        void *stream = current_stream(), *wp = nws > 0 ? ws.data_ptr() : nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = abi.bwd_ws(&s, q->data_ptr(), k->data_ptr(), v->data_ptr(), o->data_ptr(), g->data_ptr(),
                        static_cast<const float *>(lse->data_ptr()), static_cast<float *>(delta.data_ptr()),
                        dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), wp, nws, stream);
        Py_END_ALLOW_THREADS;
        if (rc != 0) return status(rc);
        return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(dq)), THPVariable_Wrap(std::move(dk)),
                             THPVariable_Wrap(std::move(dv)));
    });
}

// A 2-D tensor of contiguous rows, at least `rows` x `cols`: its row stride.
bool rows_of(const at::Tensor *t, at::ScalarType type, int64_t rows, int64_t cols, int *stride) {
    if (!t || t->scalar_type() != type || t->dim() != 2 || (t->size(1) > 1 && t->stride(1) != 1) ||
        t->size(0) < rows || t->size(1) < cols)
        return false;
    const int64_t s = t->size(0) > 1 ? t->stride(0) : std::max(t->size(1), cols);
    if (s < 0 || s > INT32_MAX) return false;
    *stride = (int)s;
    return true;
}

// prefill(q, kcache, vcache, out, table or None, block_size, pos0, n_head,
// n_kv_head, head_dim, scale, split, workspace): the launch's status (the
// workspace given where split)
PyObject *prefill(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 13 || abi.prefill == nullptr) return other();
    return guarded([&]() -> PyObject * {
        const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]), *out = plain(a[3]);
        const bool paged = a[4] != Py_None, split = a[11] == Py_True;
        const at::Tensor *table = paged ? plain(a[4]) : nullptr, *ws = split ? plain(a[12]) : nullptr;
        int block = 0, pos0, heads, kv_heads, hd, qs, ks, vs, os;
        double sc;
        if (!q || !is_mxfa_type(*q) || q->dim() != 2 || (paged && !table) || (split && !ws) ||
            (paged && (!integer(a[5], &block) || block < 1)) || !integer(a[6], &pos0) || !integer(a[7], &heads) ||
            !integer(a[8], &kv_heads) || !integer(a[9], &hd) || !number(a[10], &sc) || !PyBool_Check(a[11]) ||
            pos0 < 0 || heads < 1 || kv_heads < 1 || hd < 1 || q->size(0) < 1 || q->size(0) > INT32_MAX)
            return other();
        const int64_t n_tok = q->size(0), seen = pos0 + n_tok, crows = paged ? 1 : seen;
        if (!rows_of(q, q->scalar_type(), 1, (int64_t)heads * hd, &qs) ||
            !rows_of(k, q->scalar_type(), crows, (int64_t)kv_heads * hd, &ks) ||
            !rows_of(v, q->scalar_type(), crows, (int64_t)kv_heads * hd, &vs) || ks != vs ||
            !rows_of(out, q->scalar_type(), n_tok, (int64_t)heads * hd, &os))
            return other();
        if (paged && (table->scalar_type() != at::kInt || table->dim() != 1 || table->stride(0) != 1 ||
                      table->numel() < (seen + block - 1) / block))
            return other();
        if (split && !ws->is_contiguous()) return other();
        const mxfa_prefill_shape s{(int)n_tok, heads, kv_heads, hd, pos0, qs, ks, os,
                                   q->scalar_type() == at::kBFloat16 ? MXFA_BF16 : MXFA_F32, (float)sc};
        const void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
        const int *tp = paged ? static_cast<const int *>(table->data_ptr()) : nullptr;
        void *op = out->data_ptr(), *wp = split ? ws->data_ptr() : nullptr, *stream = current_stream();
        const size_t nws = split ? (size_t)ws->numel() * ws->element_size() : 0;
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        if (paged) {
            rc = split ? abi.prefill_paged_ws(&s, qp, kp, vp, op, tp, block, wp, nws, stream)
                       : abi.prefill_paged(&s, qp, kp, vp, op, tp, block, stream);
        } else {
            rc = split ? abi.prefill_ws(&s, qp, kp, vp, op, wp, nws, stream) : abi.prefill(&s, qp, kp, vp, op, stream);
        }
        Py_END_ALLOW_THREADS;
        return status(rc);
    });
}

// bind(addresses of the ABI functions, in the order of `abi`)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 7) {
        PyErr_SetString(PyExc_TypeError, "bind: 7 addresses expected");
        return nullptr;
    }
    void *f[7];
    for (int i = 0; i < 7; ++i) {
        f[i] = PyLong_AsVoidPtr(a[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    abi.flash_lse = reinterpret_cast<decltype(abi.flash_lse)>(f[0]);
    abi.bwd_ws = reinterpret_cast<decltype(abi.bwd_ws)>(f[1]);
    abi.bwd_workspace_bytes = reinterpret_cast<decltype(abi.bwd_workspace_bytes)>(f[2]);
    abi.prefill = reinterpret_cast<decltype(abi.prefill)>(f[3]);
    abi.prefill_ws = reinterpret_cast<decltype(abi.prefill_ws)>(f[4]);
    abi.prefill_paged = reinterpret_cast<decltype(abi.prefill_paged)>(f[5]);
    abi.prefill_paged_ws = reinterpret_cast<decltype(abi.prefill_paged_ws)>(f[6]);
    Py_RETURN_NONE;
}

#define MXFA_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MXFA_METHOD(bind), MXFA_METHOD(attention_fwd), MXFA_METHOD(attention_bwd),
                         MXFA_METHOD(prefill), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) { return PyModule_Create(&module); }
