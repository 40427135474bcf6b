// The Python layer's calls in native code: femto_native.
//
// A decode call of a few sequences keeps the GPU busy for 4-10 us, and in
// Python its checks, its strides and a ctypes call of 27 arguments cost the
// host 18 us, so every small call ran at the host's pace.  The functions here
// make the same checks on the tensors' C++ objects, allocate the output, look
// up the stream's workspace in the dict that the Python layer keeps, and call
// the library through the pointers that the Python layer passes to bind() (so
// both use one loaded library).
//
// None means "not handled here": a check failed, the call is empty, there is
// no workspace yet, an argument is not a plain tensor or int, or the tensor
// library threw.  Nothing has been launched then, and the caller takes its
// Python path, which allocates, raises or returns as it always did.  An error
// of the library itself raises RuntimeError with the library's message.
#include <Python.h>

#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "femto_attn.h"

namespace {

decltype(&femto_attn_last_error) g_last_error;
decltype(&femto_paged_attention_gemv) g_gemv;
decltype(&femto_paged_attention_gemv_workspace_size) g_gemv_ws;
decltype(&femto_paged_attention_gemm) g_gemm;
decltype(&femto_paged_attention_gemm_workspace_size) g_gemm_ws;
decltype(&femto_qk_norm_rope_cache_write) g_prologue;
decltype(&femto_flash_attention) g_flash;

// Thrown (and caught in `guarded`) where the Python path has to take over.
struct NotHere {};
inline void need(bool ok) {
    if (!ok) throw NotHere{};
}

// Exactly torch.Tensor or torch.nn.Parameter: subclasses may override what is read here.
const at::Tensor& tensor(PyObject* o) {
    need(THPVariable_CheckExact(o));
    return THPVariable_Unpack(o);
}

int64_t integer(PyObject* o) {
    need(PyLong_CheckExact(o));
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
    need(!overflow);
    return v;
}

int int32(int64_t v) {
    need(v >= INT32_MIN && v <= INT32_MAX);
    return (int)v;
}

int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return FEMTO_F32;
        case at::kHalf: return FEMTO_F16;
        case at::kBFloat16: return FEMTO_BF16;
        default: throw NotHere{};
    }
}

void* stream_of(const at::Tensor& t) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

const int32_t* i32(const at::Tensor& t) { return static_cast<const int32_t*>(t.const_data_ptr()); }

// (pointer, bytes) of the (device, stream) entry of a workspace dict, 256-byte aligned as the Python
// layer aligns it; the entry has to hold nbytes + 256.
struct Workspace {
    void* ptr = nullptr;
    size_t bytes = 0;
    at::Tensor hold;  // another thread may replace the dict's entry during the call
};
Workspace workspace(PyObject* dict, const at::Tensor& on, void* stream, size_t nbytes) {
    Workspace w;
    if (nbytes == 0) return w;
    need(PyDict_CheckExact(dict));
    PyObject* key = Py_BuildValue("(iK)", (int)on.device().index(), (unsigned long long)(uintptr_t)stream);
    need(key != nullptr);
    PyObject* o = PyDict_GetItemWithError(dict, key);  // borrowed
    Py_DECREF(key);
    if (!o) PyErr_Clear();
    need(o != nullptr);
    const at::Tensor& t = tensor(o);
    need((size_t)t.numel() >= nbytes + 256);
    const uintptr_t p = (uintptr_t)t.data_ptr(), a = (p + 255) & ~(uintptr_t)255;
    w.ptr = (void*)a;
    w.bytes = (size_t)t.numel() - (a - p);
    w.hold = t;
    return w;
}

// The checks that the decode and the prefill call share (_check_paged in _C.py).
void check_paged(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& tables,
                 const at::Tensor& kv_lens, bool contiguous_q, int64_t unit_bytes, int64_t unit_elems) {
    need(q.is_cuda() && k.is_cuda() && v.is_cuda());
    need(!contiguous_q || q.is_contiguous());
    need(q.dim() == 3 && k.dim() == 4 && v.dim() == 4 && k.sizes() == v.sizes());
    need(k.is_contiguous() && v.is_contiguous());
    const int64_t d = q.size(2);
    need(d == k.size(3) && q.stride(2) == 1);
    need(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type());
    need(tables.scalar_type() == at::kInt && kv_lens.scalar_type() == at::kInt);
    need(tables.dim() == 2 && (tables.size(1) <= 1 || tables.stride(1) == 1));
    need(kv_lens.dim() == 1 && kv_lens.is_contiguous());
    need(tables.device() == q.device() && kv_lens.device() == q.device());
    need(k.size(2) == 16 && d > 0 && d <= 128);
    need((d * q.element_size()) % unit_bytes == 0 && d % unit_elems == 0);
    need(k.size(1) > 0 && q.size(0) % k.size(1) == 0);
}

// The library call and its result.  The result's Python object is made first and whatever the library
// throws is an error: nothing can decline the call once the library has been entered (the Python path
// would make it a second time, on a q that the first may have overwritten).
template <typename F>
PyObject* launch(const at::Tensor& out, F call) {
    PyObject* result = THPVariable_Wrap(out);
    need(result != nullptr);
    int rc;
    PyThreadState* gil = PyEval_SaveThread();
    try {
        rc = call();
    } catch (...) {
        rc = -1;
    }
    PyEval_RestoreThread(gil);
    if (rc == 0) return result;
    Py_DECREF(result);
    PyErr_SetString(PyExc_RuntimeError, rc < 0 ? "femto_native: the library threw" : g_last_error());
    return nullptr;
}

template <typename F>
PyObject* guarded(Py_ssize_t n, Py_ssize_t want, F f) {
    try {
        need(n == want && g_gemv);
        return f();
    } catch (const NotHere&) {
    } catch (const std::exception&) {  // raised again, as Python sees it, by the Python path
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

// gemv(q, k_pool, v_pool, tables, kv_lens, max_kv_len, contiguous_q, max_kv_len_limit, workspaces)
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 9, [&]() -> PyObject* {
        const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &tab = tensor(a[3]), &len = tensor(a[4]);
        const int max_kv = int32(integer(a[5]));
        check_paged(q, k, v, tab, len, a[6] == Py_True, 16, 1);
        const int64_t H = q.size(0), B = q.size(1);
        need(B > 0 && B == tab.size(0) && B == len.size(0));
        need(a[7] == Py_None || max_kv <= integer(a[7]));
        const int dt = dtype_code(q);
        void* st = stream_of(q);
        const Workspace w = workspace(a[8], q, st, g_gemv_ws(int32(B), int32(H), max_kv));
        at::Tensor out = at::empty({H, B, q.size(2)}, q.options());
        const void *qp = q.const_data_ptr(), *kp = k.const_data_ptr(), *vp = v.const_data_ptr();
        const int32_t *tp = i32(tab), *lp = i32(len);
        void* op = out.data_ptr();
        return launch(out, [&] {
            return g_gemv(dt, qp, q.stride(0), q.stride(1), op, out.stride(0), out.stride(1), kp, vp, k.size(0), (int)k.size(1),
                          (int)k.size(2), (int)k.size(3), k.stride(0), k.stride(1), k.stride(2), tp, (int)tab.size(1),
                          tab.stride(0), lp, (int)B, (int)H, max_kv, w.ptr, w.bytes, st);
        });
    });
}

// gemm(q, k_pool, v_pool, cu_seqlens, max_q_len, tables, kv_lens, positions, contiguous_q, workspaces)
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 10, [&]() -> PyObject* {
        const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &cu = tensor(a[3]);
        const at::Tensor &tab = tensor(a[5]), &len = tensor(a[6]), &pos = tensor(a[7]);
        const int max_q = int32(integer(a[4]));
        check_paged(q, k, v, tab, len, a[8] == Py_True, 1, 16);
        need(cu.scalar_type() == at::kInt && cu.is_contiguous() && cu.device() == q.device());
        need(pos.scalar_type() == at::kInt && pos.is_contiguous() && pos.device() == q.device());
        const int64_t H = q.size(0), T = q.size(1), B = cu.numel() - 1;
        need(B > 0 && T > 0 && B == tab.size(0) && B == len.size(0) && T == pos.numel());
        need(q.scalar_type() != at::kFloat);
        const int dt = dtype_code(q);
        void* st = stream_of(q);
        const Workspace w = workspace(a[9], q, st, g_gemm_ws(int32(B), int32(T), max_q, int32(H), (int)k.size(1),
                                                             int32(tab.size(1))));
        at::Tensor out = at::empty({H, T, q.size(2)}, q.options());
        const void *qp = q.const_data_ptr(), *kp = k.const_data_ptr(), *vp = v.const_data_ptr();
        const int32_t *cp = i32(cu), *tp = i32(tab), *lp = i32(len), *pp = i32(pos);
        void* op = out.data_ptr();
        return launch(out, [&] {
            return g_gemm(dt, qp, q.stride(0), q.stride(1), op, out.stride(0), out.stride(1), kp, vp, k.size(0), (int)k.size(1),
                          (int)k.size(2), (int)k.size(3), k.stride(0), k.stride(1), k.stride(2), cp, (int)B, (int)T, max_q, (int)H,
                          tp, (int)tab.size(1), tab.stride(0), lp, pp, w.ptr, w.bytes, st);
        });
    });
}

// prologue(q, k, v, q_weight, k_weight, eps, cos, sin, positions, k_pool, v_pool, tables, cu_seqlens | None,
//          max_q_len, out | None)
PyObject* prologue(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 15, [&]() -> PyObject* {
        const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &wq = tensor(a[3]), &wk = tensor(a[4]);
        const at::Tensor &cos = tensor(a[6]), &sin = tensor(a[7]), &pos = tensor(a[8]);
        const at::Tensor &kp = tensor(a[9]), &vp = tensor(a[10]), &tab = tensor(a[11]);
        need(PyFloat_CheckExact(a[5]));
        const float eps = (float)PyFloat_AS_DOUBLE(a[5]);
        const int max_q = int32(integer(a[13]));
        need(q.is_cuda());
        for (const at::Tensor* t : {&k, &v, &wq, &wk, &cos, &sin, &kp, &vp, &pos, &tab}) need(t->device() == q.device());
        need(q.dim() == 3 && k.dim() == 3 && v.dim() == 3 && k.sizes() == v.sizes());
        need(q.size(0) == k.size(0) && q.size(2) == k.size(2) && q.size(2) == 128);
        need(q.stride(2) == 1 && k.stride(2) == 1 && v.stride(2) == 1);
        need(wq.numel() == 128 && wk.numel() == 128 && wq.is_contiguous() && wk.is_contiguous());
        for (const at::Tensor* t : {&k, &v, &wq, &wk, &kp, &vp}) need(t->scalar_type() == q.scalar_type());
        need(cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat);
        need(cos.dim() == 2 && cos.sizes() == sin.sizes() && cos.strides() == sin.strides() && cos.stride(1) == 1 &&
             cos.size(1) >= 128);
        need(kp.dim() == 4 && kp.sizes() == vp.sizes() && kp.is_contiguous() && vp.is_contiguous());
        need(k.size(1) == kp.size(1) && kp.size(3) == 128 && kp.size(2) == 16);
        need(k.size(1) > 0 && q.size(1) % k.size(1) == 0);
        need(pos.scalar_type() == at::kInt && pos.is_contiguous());
        need(tab.scalar_type() == at::kInt && tab.dim() == 2 && (tab.size(1) <= 1 || tab.stride(1) == 1));
        const int64_t T = q.size(0), B = tab.size(0);
        need(T > 0 && B > 0 && pos.numel() == T);
        const int32_t* cp = nullptr;
        if (a[12] == Py_None) {
            need(T == B);
        } else {
            const at::Tensor& cu = tensor(a[12]);
            need(cu.scalar_type() == at::kInt && cu.is_contiguous() && cu.device() == q.device() && cu.numel() - 1 == B);
            cp = i32(cu);
        }
        const int dt = dtype_code(q);
        at::Tensor out = a[14] == Py_None ? at::empty_like(q) : tensor(a[14]);
        need(out.sizes() == q.sizes() && out.scalar_type() == q.scalar_type() && out.stride(2) == 1 &&
             out.device() == q.device());
        void* st = stream_of(q);
        const void *qd = q.const_data_ptr(), *kd = k.const_data_ptr(), *vd = v.const_data_ptr();
        const void *wqd = wq.const_data_ptr(), *wkd = wk.const_data_ptr();
        const float* cd = static_cast<const float*>(cos.const_data_ptr());
        const float* sd = static_cast<const float*>(sin.const_data_ptr());
        void *od = out.data_ptr(), *kpd = kp.data_ptr(), *vpd = vp.data_ptr();
        const int32_t *pd = i32(pos), *td = i32(tab);
        const int H = int32(q.size(1)), rows = int32(cos.size(0)), tokens = int32(T), seqs = int32(B);
        return launch(out, [&] {
            return g_prologue(dt, qd, q.stride(0), q.stride(1), kd, k.stride(0), k.stride(1), vd, v.stride(0), v.stride(1), od,
                              out.stride(0), out.stride(1), wqd, wkd, eps, cd, sd, cos.stride(0), rows, kpd, vpd, kp.size(0), H,
                              (int)kp.size(1), (int)kp.size(2), (int)kp.size(3), kp.stride(0), kp.stride(1), kp.stride(2), cp, seqs,
                              tokens, max_q, pd, td, (int)tab.size(1), tab.stride(0), st);
        });
    });
}

// flash(q, k, v)
PyObject* flash(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded(n, 3, [&]() -> PyObject* {
        const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
        for (const at::Tensor* t : {&q, &k, &v})
            need(t->is_cuda() && t->dim() == 4 && t->is_contiguous() && (uintptr_t)t->const_data_ptr() % 16 == 0);
        need(k.sizes() == v.sizes() && q.size(0) == k.size(0) && q.size(3) == k.size(3) && q.size(3) == 128);
        need(k.size(1) > 0 && q.size(1) % k.size(1) == 0);
        need(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type() && q.scalar_type() != at::kFloat);
        const int dt = dtype_code(q);
        at::Tensor out = at::empty_like(q);
        void* st = stream_of(q);
        const void *qp = q.const_data_ptr(), *kp = k.const_data_ptr(), *vp = v.const_data_ptr();
        void* op = out.data_ptr();
        const int B = int32(q.size(0)), H = int32(q.size(1)), KVH = int32(k.size(1)), Tq = int32(q.size(2)),
                  Tk = int32(k.size(2));
        return launch(out, [&] {
            return g_flash(dt, qp, q.stride(0), q.stride(1), q.stride(2), kp, k.stride(0), k.stride(1), k.stride(2), vp,
                           v.stride(0), v.stride(1), v.stride(2), op, out.stride(0), out.stride(1), out.stride(2), B, H, KVH, Tq,
                           Tk, 128, st);
        });
    });
}

// bind({function name: address}): the library's entry points.
PyObject* bind(PyObject*, PyObject* names) {
    auto get = [&](const char* name, auto& fn) {
        PyObject* o = PyDict_Check(names) ? PyDict_GetItemString(names, name) : nullptr;
        void* p = o ? PyLong_AsVoidPtr(o) : nullptr;
        if (!p && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "femto_native.bind: no address of %s", name);
        if (p) fn = reinterpret_cast<std::decay_t<decltype(fn)>>(p);
        return p != nullptr;
    };
    if (!get("femto_attn_last_error", g_last_error) || !get("femto_paged_attention_gemv_workspace_size", g_gemv_ws) ||
        !get("femto_paged_attention_gemm", g_gemm) || !get("femto_paged_attention_gemm_workspace_size", g_gemm_ws) ||
        !get("femto_qk_norm_rope_cache_write", g_prologue) || !get("femto_flash_attention", g_flash) ||
        !get("femto_paged_attention_gemv", g_gemv))
        return nullptr;
    Py_RETURN_NONE;
}

#define FEMTO_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"gemv", FEMTO_FAST(gemv)},
    {"gemm", FEMTO_FAST(gemm)},
    {"prologue", FEMTO_FAST(prologue)},
    {"flash", FEMTO_FAST(flash)},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "femto_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_femto_native() { return PyModule_Create(&module); }
