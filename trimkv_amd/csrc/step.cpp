// What a decode step asks of the host for every layer, in native code: the checks of a deferred append, the views of a layer that update()
// returns, and the launch that appends and attends.  A layer of a short step lasts less on the GPU (8.8 us, 32 segments of 540 rows) than its
// update and attention took in Python (16.4 us): the host bounds such a step, not the device.
//
// Everything here is the usual case only.  A call that is not that returns None (or 0), and the caller goes the general way.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <ATen/ATen.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "trimkv_hip.h"

namespace {

// attributes of cache_utils._Slab
PyObject *s_step, *s_pending, *s_lens, *s_max_len, *s_total, *s_k, *s_v, *s_lb, *s_pos, *s_cu;

struct Held {      // a reference of our own
    PyObject* p;
    explicit Held(PyObject* o) : p(o) {}
    ~Held() { Py_XDECREF(p); }
    Held(const Held&) = delete;
    Held& operator=(const Held&) = delete;
    operator PyObject*() const { return p; }
};

// The step arguments that the layer keeps (a bytearray, its first part filled in), or NULL.
trimkv_append_step* step_of(PyObject* slab) {
    Held b(PyObject_GetAttr(slab, s_step));      // the layer holds it as well
    if (!b.p) { PyErr_Clear(); return nullptr; }
    return PyByteArray_CheckExact(b.p) && PyByteArray_GET_SIZE(b.p) == (Py_ssize_t)sizeof(trimkv_append_step) ? (trimkv_append_step*)PyByteArray_AS_STRING(b.p) : nullptr;
}
long long number(PyObject* slab, PyObject* name) {
    Held o(PyObject_GetAttr(slab, name));
    return o.p ? PyLong_AsLongLong(o.p) : -1;
}
bool plain(PyObject* o) { return THPVariable_CheckExact(o); }

// defer(slab, k, v, lb, pos) -> True: the row is remembered (what _SlabBacked._defer does); None: not the usual case, nothing has changed
PyObject* defer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) { PyErr_SetString(PyExc_TypeError, "defer(slab, k, v, lb, pos)"); return nullptr; }
    PyObject* slab = a[0];
    trimkv_append_step* s = step_of(slab);
    if (!s || !plain(a[1]) || !plain(a[2]) || !plain(a[3]) || !plain(a[4])) Py_RETURN_NONE;
    Held pending(PyObject_GetAttr(slab, s_pending)), slab_k(PyObject_GetAttr(slab, s_k)), slab_lb(PyObject_GetAttr(slab, s_lb));
    if (!pending.p || !slab_k.p || !slab_lb.p) return nullptr;
    if (pending.p != Py_None || !plain(slab_k) || !plain(slab_lb)) Py_RETURN_NONE;
    const at::Tensor &k = THPVariable_Unpack(a[1]), &v = THPVariable_Unpack(a[2]), &lb = THPVariable_Unpack(a[3]), &pos = THPVariable_Unpack(a[4]);
    const at::Tensor &kept = THPVariable_Unpack(slab_k.p), &kept_lb = THPVariable_Unpack(slab_lb.p);
    const int64_t H = s->kv_heads, B = s->nseg / H, D = s->head_dim;
    if (!k.is_cuda() || !v.is_cuda() || !lb.is_cuda() || k.dim() != 4 || v.dim() != 4 || lb.dim() != 3 || k.scalar_type() != kept.scalar_type() || v.scalar_type() != kept.scalar_type() ||
        lb.scalar_type() != kept_lb.scalar_type() || pos.scalar_type() != at::kLong || pos.device() != k.device()) Py_RETURN_NONE;
    const int64_t *kz = k.sizes().data(), *vz = v.sizes().data(), *lz = lb.sizes().data();
    if (kz[0] != B || kz[1] != H || kz[2] != 1 || kz[3] != D || vz[0] != B || vz[1] != H || vz[2] != 1 || vz[3] != D || lz[0] != B || lz[1] != H || lz[2] != 1) Py_RETURN_NONE;
    const int64_t *ks = k.strides().data(), *vs = v.strides().data(), *ls = lb.strides().data();
    const uintptr_t kp = (uintptr_t)k.data_ptr(), vp = (uintptr_t)v.data_ptr();
    if (ks[3] != 1 || (ks[0] | ks[1]) % 8 || vs[0] != ks[0] || vs[1] != ks[1] || vs[3] != 1 || (kp | vp) % 16) Py_RETURN_NONE;
    int64_t p0 = 0, p1 = 0;
    if (pos.dim() == 3) {
        const int64_t* pz = pos.sizes().data();
        if (pz[0] != B || pz[1] != H || pz[2] != 1) Py_RETURN_NONE;
        p0 = pos.strides()[0]; p1 = pos.strides()[1];
    } else if (pos.dim() != 1 || pos.numel() < 1) Py_RETURN_NONE;
    const long long max_len = number(slab, s_max_len), total = number(slab, s_total);
    if (PyErr_Occurred()) return nullptr;
    if (max_len + 1 > s->cap) Py_RETURN_NONE;
    Held lens(PyObject_GetAttr(slab, s_lens));
    if (!lens.p) return nullptr;
    Held args(Py_BuildValue("(KKLLKLLKLL)", (unsigned long long)kp, (unsigned long long)vp, (long long)ks[0], (long long)ks[1], (unsigned long long)(uintptr_t)lb.data_ptr(),
                            (long long)ls[0], (long long)ls[1], (unsigned long long)(uintptr_t)pos.data_ptr(), (long long)p0, (long long)p1));
    if (!args.p) return nullptr;
    Held row(PyTuple_Pack(5, args.p, a[1], a[2], a[3], a[4])), longer(PyLong_FromLongLong(max_len + 1)), more(PyLong_FromLongLong(total + s->nseg));
    if (!row.p || !longer.p || !more.p) return nullptr;
    Py_buffer view;
    if (PyObject_GetBuffer(lens, &view, PyBUF_CONTIG)) { PyErr_Clear(); Py_RETURN_NONE; }
    const bool fits = view.itemsize == 8 && view.len == s->nseg * 8;
    if (fits) for (int64_t i = 0; i < s->nseg; ++i) ++((int64_t*)view.buf)[i];
    PyBuffer_Release(&view);
    if (!fits) Py_RETURN_NONE;
    if (PyObject_SetAttr(slab, s_pending, row) || PyObject_SetAttr(slab, s_max_len, longer) || PyObject_SetAttr(slab, s_total, more)) return nullptr;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

PyObject* wrapped(const at::Tensor (&t)[4]) {
    Held out(PyTuple_New(4));
    if (!out.p) return nullptr;
    for (int i = 0; i < 4; ++i) {
        PyObject* o = THPVariable_Wrap(t[i]);
        if (!o) return nullptr;
        PyTuple_SET_ITEM(out.p, i, o);
    }
    Py_INCREF(out.p);
    return out.p;
}

// Nobody follows operations and no gradient is recorded: no mode, no tracer or transform of functorch, no profiler, nothing below autograd.
bool unwatched() {
    using c10::DispatchKey;
    const auto tls = c10::impl::tls_local_dispatch_key_set();
    return !c10::GradMode::is_enabled() && !c10::InferenceMode::is_enabled() && !at::hasCallbacks() && !c10::impl::dispatch_mode_enabled() &&
           (tls.included_ - c10::DispatchKeySet({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView})).empty() && !tls.excluded_.has(DispatchKey::ADInplaceOrView);
}

// What base.as_strided(sizes, strides) is without gradients, the view's base and version counter among it, made without the dispatcher's ways there (0.9 us
// for the four; 128 layers' steps of 32 segments of 512 .. 544 rows, which the host bounds, 1512 .. 1534 -> 1439 .. 1467 us in four processes each).
at::Tensor view_of(const at::Tensor& base, c10::IntArrayRef sizes, c10::IntArrayRef strides) {
    auto impl = c10::make_intrusive<at::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(base.storage()), base.key_set(), base.dtype());
    impl->set_sizes_and_strides(sizes, strides, base.storage_offset());
    if (base.is_inference()) return at::Tensor(std::move(impl));
    return torch::autograd::make_variable_differentiable_view(at::Tensor(std::move(impl)), torch::autograd::ViewInfo(base, nullptr, nullptr), std::nullopt, true, torch::autograd::CreationMeta::NO_GRAD_MODE);
}

// views(slab, n) -> the first n rows of K, V, log beta and positions, [B, H, n, ...]; n < 0: all rows with the segments one behind the other, [nseg cap, ...]
PyObject* views(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2) { PyErr_SetString(PyExc_TypeError, "views(slab, n)"); return nullptr; }
    const trimkv_append_step* s = step_of(a[0]);
    const long long rows = PyLong_AsLongLong(a[1]);
    if (PyErr_Occurred()) return nullptr;
    if (!s) { PyErr_SetString(PyExc_RuntimeError, "views: the layer has no step arguments"); return nullptr; }
    PyObject* const names[4] = {s_k, s_v, s_lb, s_pos};
    const int64_t H = s->kv_heads, B = s->nseg / H, D = s->head_dim, cap = s->cap;
    const bool direct = unwatched();
    at::Tensor out[4];
    for (int i = 0; i < 4; ++i) {
        Held o(PyObject_GetAttr(a[0], names[i]));
        if (!o.p) return nullptr;
        if (!THPVariable_Check(o.p)) { PyErr_SetString(PyExc_TypeError, "views: not a tensor"); return nullptr; }
        const at::Tensor& t = THPVariable_Unpack(o.p);
        // the slab's own tensor, [nseg, cap, D] or [nseg, cap], whole: what lies outside of it is as_strided's to refuse
        const bool slab = direct && rows <= cap && plain(o) && !t.is_view() && !t.requires_grad() && t.layout() == c10::kStrided && t.is_contiguous() &&
                          t.numel() == s->nseg * cap * (i < 2 ? D : 1);
        if (slab && rows < 0) out[i] = view_of(t, {s->nseg * cap, i < 2 ? D : 1}, {i < 2 ? D : 1, 1});
        else if (slab && i < 2) out[i] = view_of(t, {B, H, rows, D}, {H * cap * D, cap * D, D, 1});
        else if (slab) out[i] = view_of(t, {B, H, rows}, {H * cap, cap, 1});
        else if (rows < 0) out[i] = t.view({s->nseg * cap, i < 2 ? D : 1});
        else if (i < 2) out[i] = t.as_strided({B, H, rows, D}, {H * cap * D, cap * D, D, 1});
        else out[i] = t.as_strided({B, H, rows}, {H * cap, cap, 1});
    }
    return wrapped(out);
    END_HANDLE_TH_ERRORS
}

// fits(query, key, slab) -> query heads per KV head if this is the usual decode step of a dense cache (one query row per sequence, `slab`'s append
// deferred to it, `key` the layer's rows), else 0
PyObject* fits(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) { PyErr_SetString(PyExc_TypeError, "fits(query, key, slab)"); return nullptr; }
    const trimkv_append_step* s = step_of(a[2]);
    if (!s || !plain(a[0]) || !plain(a[1])) return PyLong_FromLong(0);
    Held pending(PyObject_GetAttr(a[2], s_pending)), cu(PyObject_GetAttr(a[2], s_cu)), slab_k(PyObject_GetAttr(a[2], s_k));
    if (!pending.p || !cu.p || !slab_k.p) return nullptr;
    const at::Tensor &q = THPVariable_Unpack(a[0]), &key = THPVariable_Unpack(a[1]);
    if (pending.p == Py_None || cu.p != Py_None || !plain(slab_k) || !q.is_cuda() || q.dim() != 4 || key.dim() != 4) return PyLong_FromLong(0);
    const int64_t H = s->kv_heads, B = s->nseg / H, G = q.size(1) / H;
    if (q.size(0) != B || q.size(1) != G * H || q.size(2) != 1 || q.size(3) != s->head_dim || q.scalar_type() != THPVariable_Unpack(slab_k.p).scalar_type() ||
        key.const_data_ptr() != s->k_slab || key.size(2) != number(a[2], s_max_len)) return PyErr_Occurred() ? nullptr : PyLong_FromLong(0);
    return PyLong_FromLong((long)G);
    END_HANDLE_TH_ERRORS
}

// attend(slab, query, group, scale, rows, count, pieces, workspace, workspace_bytes, stream, entry) -> the output, or the entry point's status.
// query contiguous, [.., D] or [B, Hq, 1, D] (the output is [B, 1, Hq, D] then); `entry`: the address of trimkv_append_attend_step.
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 11) { PyErr_SetString(PyExc_TypeError, "attend takes 11 arguments"); return nullptr; }
    trimkv_append_step* s = step_of(a[0]);
    if (!s || !THPVariable_Check(a[1])) { PyErr_SetString(PyExc_TypeError, "attend: no step arguments, or no tensor"); return nullptr; }
    Held pending(PyObject_GetAttr(a[0], s_pending));
    if (!pending.p) return nullptr;
    PyObject* row = PyTuple_Check(pending.p) && PyTuple_GET_SIZE(pending.p) == 5 ? PyTuple_GET_ITEM(pending.p, 0) : nullptr;
    if (!row || !PyTuple_Check(row) || PyTuple_GET_SIZE(row) != 10) { PyErr_SetString(PyExc_RuntimeError, "attend: no row is waiting"); return nullptr; }
    long long in[10], more[8];
    for (int i = 0; i < 10; ++i) in[i] = (long long)PyLong_AsUnsignedLongLongMask(PyTuple_GET_ITEM(row, i));
    const double scale = PyFloat_AsDouble(a[3]);
    for (int i = 0; i < 8; ++i) more[i] = i == 0 ? PyLong_AsLongLong(a[2]) : (long long)PyLong_AsUnsignedLongLongMask(a[i + 3]);
    if (PyErr_Occurred()) return nullptr;
    const at::Tensor& q = THPVariable_Unpack(a[1]);
    const at::Tensor out = q.dim() == 4 ? at::empty({q.size(0), q.size(2), q.size(1), q.size(3)}, q.options()) : at::empty(q.sizes(), q.options());
    s->q = q.const_data_ptr(); s->out = out.data_ptr();
    s->k_new = (const void*)in[0]; s->v_new = (const void*)in[1]; s->kv_stride_b = in[2]; s->kv_stride_h = in[3];
    s->lb_new = (const void*)in[4]; s->lb_stride_b = in[5]; s->lb_stride_h = in[6];
    s->pos_new = (const int64_t*)in[7]; s->pos_stride_b = in[8]; s->pos_stride_h = in[9];
    s->group = more[0]; s->scale = scale; s->len = more[1]; s->count = more[2];
    s->pieces = (const int32_t*)more[3]; s->workspace = (void*)more[4]; s->workspace_bytes = more[5];
    const trimkv_append_step mine = *s;      // another thread may run during the launch
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ((int (*)(const trimkv_append_step*, void*))(uintptr_t)more[7])(&mine, (void*)more[6]);
    Py_END_ALLOW_THREADS
    if (rc) return PyLong_FromLong(rc);
    if (PyObject_SetAttr(a[0], s_pending, Py_None)) return nullptr;
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"defer", (PyCFunction)(void*)defer, METH_FASTCALL, nullptr}, {"views", (PyCFunction)(void*)views, METH_FASTCALL, nullptr},
                         {"fits", (PyCFunction)(void*)fits, METH_FASTCALL, nullptr}, {"attend", (PyCFunction)(void*)attend, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_step", "Host side of decode steps in native code.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__step(void) {
    const struct { PyObject** at; const char* name; } names[] = {{&s_step, "step"}, {&s_pending, "pending"}, {&s_lens, "lens"}, {&s_max_len, "max_len"}, {&s_total, "total"},
                                                                 {&s_k, "k"}, {&s_v, "v"}, {&s_lb, "lb"}, {&s_pos, "pos"}, {&s_cu, "cu"}};
    for (const auto& x : names)
        if (!(*x.at = PyUnicode_InternFromString(x.name))) return nullptr;
    return PyModule_Create(&module);
}
