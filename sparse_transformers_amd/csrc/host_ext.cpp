// The eager entry points' host side: argument checks, output tensors and the call of the C ABI without a Python statement or
// a ctypes conversion per argument (15 us less per layer step than the same in Python, which was level with the kernels).
//
// Every function takes the common form of its call only -- plain tensors (or parameters) of the right type, shape, layout
// and device -- and returns None for anything else: the Python code behind it then does what the form needs (copies, views)
// or raises what it always raised.  A failed C call returns its status as an int.  Nothing is kept between calls but the
// addresses of the library's functions.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "../../include/sparse_mlp_amd.h"

namespace {

decltype(&st_predictor_mask_ex) f_predictor;
decltype(&st_cache_update_forward) f_update_forward;
decltype(&st_mlp_forward) f_mlp_forward;
decltype(&st_cache_create) f_cache_create;
decltype(&st_cache_destroy) f_cache_destroy;
decltype(&st_cache_load_weights_begin) f_load_begin;
decltype(&st_cache_max_intermediate) f_max_intermediate;

// A plain tensor with memory of its own on a GPU (no subclass, no wrapper of a transform); nullptr: not one.
const at::Tensor *gpu_tensor(PyObject *o)
{
    if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg()) return nullptr;
    using c10::DispatchKey;
    constexpr c10::DispatchKeySet wrapped{DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize,
                                          DispatchKey::Python, DispatchKey::ZeroTensor};
    if (t.key_set().has_any(wrapped) || !t.has_storage()) return nullptr;
    return &t;
}

int code_of(const at::Tensor &t)   // -1: a type the fast path leaves to Python
{
    switch (t.scalar_type()) {
    case at::kFloat: return ST_F32;
    case at::kHalf: return ST_F16;
    case at::kBFloat16: return ST_BF16;
    default: return -1;
    }
}

bool rows_of(const at::Tensor &t, int64_t cols) { return t.dim() == 2 && t.size(1) == cols && t.is_contiguous(); }

bool same_kind(const at::Tensor &t, const at::Tensor &like) { return t.scalar_type() == like.scalar_type() && t.device() == like.device(); }

bool bytes_of(const at::Tensor &t, const at::Tensor &like, int64_t n)
{
    return (t.scalar_type() == at::kBool || t.scalar_type() == at::kByte) && t.device() == like.device() && t.numel() == n && t.is_contiguous();
}

bool workspace_of(const at::Tensor &t, const at::Tensor &like)
{
    return t.scalar_type() == at::kByte && t.device() == like.device() && t.is_contiguous();
}

PyObject *none() { Py_RETURN_NONE; }

// The library call without the interpreter's lock (the tensors are the caller's or local, so they outlive it).
template <typename F> int launched(F f)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

template <typename F> PyObject *guarded(F f)
{
    try {
        return f();
    } catch (...) {   // (nothing has been launched: allocation and metadata calls only come before the launch)
        return none();
    }
}

// predictor_mask(x, down, up, thr, ge, out, t_ws, scores, flags, stream) -> mask | status | None
PyObject *predictor_mask(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 10 || !f_predictor) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *x = gpu_tensor(a[0]), *down = gpu_tensor(a[1]), *up = gpu_tensor(a[2]);
        if (!x || !down || !up || x->dim() != 2 || !x->is_contiguous()) return none();
        const int64_t B = x->size(0), H = x->size(1);
        if (!rows_of(*down, H)) return none();
        const int64_t r = down->size(0);
        if (!rows_of(*up, r) || !same_kind(*down, *x) || !same_kind(*up, *x)) return none();
        const int64_t I = up->size(0);
        const int code = code_of(*x);
        if (code < 0) return none();
        at::Tensor mask, t_ws;
        if (a[5] != Py_None) {
            const at::Tensor *o = gpu_tensor(a[5]);
            if (!o || o->scalar_type() != at::kBool || !bytes_of(*o, *x, I)) return none();
        }
        const at::Tensor *ws = nullptr, *scores = nullptr;
        if (a[6] != Py_None) {
            ws = gpu_tensor(a[6]);
            if (!ws || ws->scalar_type() != at::kFloat || ws->numel() < B * r || ws->device() != x->device()) return none();
        }
        if (a[7] != Py_None) {
            scores = gpu_tensor(a[7]);
            if (!scores || scores->scalar_type() != at::kFloat || scores->numel() < B * I || scores->device() != x->device() ||
                !scores->is_contiguous())
                return none();
        }
        const double thr = PyFloat_AsDouble(a[3]);
        const int ge = PyObject_IsTrue(a[4]);
        const long flags = PyLong_AsLong(a[8]);
        void *stream = PyLong_AsVoidPtr(a[9]);
        if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
        if (!ws) { t_ws = at::empty({B, r}, x->options().dtype(at::kFloat)); ws = &t_ws; }
        if (a[5] == Py_None) mask = at::empty({I}, x->options().dtype(at::kBool));
        else mask = *gpu_tensor(a[5]);
        const void *px = x->data_ptr(), *pd = down->data_ptr(), *pu = up->data_ptr();
        float *pt = static_cast<float *>(ws->data_ptr()), *ps = scores ? static_cast<float *>(scores->data_ptr()) : nullptr;
        uint8_t *pm = static_cast<uint8_t *>(mask.data_ptr());
        const int rc = launched([&] { return f_predictor(px, B, H, pd, r, pu, I, code, (float)thr, ge, (int)flags, pt, ps, pm, stream); });
        if (rc != ST_OK) return PyLong_FromLong(rc);
        if (a[5] != Py_None) { Py_INCREF(a[5]); return a[5]; }
        return THPVariable_Wrap(mask);
    });
}

// update_forward(handle, like, mask, x, out, workspace, I, hint, act, stream) -> out | status | None
// `like`: a tensor of the cache's type and device, [., H].
PyObject *update_forward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 10 || !f_update_forward) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *like = gpu_tensor(a[1]), *mask = gpu_tensor(a[2]), *x = gpu_tensor(a[3]), *ws = gpu_tensor(a[5]);
        if (!like || !mask || !x || !ws || !rows_of(*x, like->size(1)) || !same_kind(*x, *like)) return none();
        void *handle = PyLong_AsVoidPtr(a[0]), *stream = PyLong_AsVoidPtr(a[9]);
        const int64_t I = PyLong_AsLongLong(a[6]), hint = PyLong_AsLongLong(a[7]);
        const long act = PyLong_AsLong(a[8]);
        if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
        if (!handle || !bytes_of(*mask, *x, I) || !workspace_of(*ws, *x)) return none();
        at::Tensor out;
        if (a[4] == Py_None) {
            out = at::empty_like(*x);
        } else {
            const at::Tensor *o = gpu_tensor(a[4]);
            if (!o || !rows_of(*o, x->size(1)) || o->size(0) != x->size(0) || !same_kind(*o, *x)) return none();
            out = *o;
        }
        const uint8_t *pm = static_cast<const uint8_t *>(mask->data_ptr());
        const void *px = x->data_ptr();
        void *po = out.data_ptr(), *pw = ws->data_ptr();
        const int64_t B = x->size(0), bytes = ws->numel();
        const int rc = launched([&] {
            return f_update_forward(static_cast<st_cache *>(handle), pm, px, B, hint, po, nullptr, 0, pw, bytes, (int)act, stream);
        });
        if (rc != ST_OK) return PyLong_FromLong(rc);
        if (a[4] != Py_None) { Py_INCREF(a[4]); return a[4]; }
        return THPVariable_Wrap(out);
    });
}

// mlp_forward(x, gate | None, up, down, n, n_dev | None, out | None, combined | None, hint, workspace, act, stream, operator) ->
// out | status | None.  `out` and `combined` are contiguous [B, H] and [B, (gate and up: 2) n].  The operator's form makes them
// so as the last thing before the launch, and its `down` is the matrix [H, n]: only as the transposed view of packed rows is it
// read in place (n = H does not make a row-major one packed rows).  The cache's form hands over packed rows [>= n, H].
PyObject *mlp_forward(PyObject *, PyObject *const *a, Py_ssize_t n_args)
{
    if (n_args != 13 || !f_mlp_forward) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *x = gpu_tensor(a[0]), *up = gpu_tensor(a[2]), *down = gpu_tensor(a[3]), *ws = gpu_tensor(a[9]);
        const at::Tensor *gate = a[1] == Py_None ? nullptr : gpu_tensor(a[1]);
        if (!x || !up || !down || !ws || (a[1] != Py_None && !gate) || x->dim() != 2 || !x->is_contiguous()) return none();
        const int64_t B = x->size(0), H = x->size(1), n = PyLong_AsLongLong(a[4]), hint = PyLong_AsLongLong(a[8]);
        const long act = PyLong_AsLong(a[10]);
        void *stream = PyLong_AsVoidPtr(a[11]);
        const int as_operator = PyObject_IsTrue(a[12]);
        if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
        const int code = code_of(*x);
        if (code < 0 || n < 0 || !workspace_of(*ws, *x)) return none();
        auto packed = [&](const at::Tensor &t) { return rows_of(t, H) && t.size(0) >= n && same_kind(t, *x); };
        // (strides (1, H): packed rows [n, H], transposed)
        const bool view = down->dim() == 2 && down->size(0) == H && down->size(1) == n && n > 0 && down->stride(0) == 1 &&
                          down->stride(1) == H && same_kind(*down, *x);
        if (!packed(*up) || (gate && !packed(*gate)) || !(as_operator ? view : packed(*down))) return none();
        const int32_t *n_dev = nullptr;
        if (a[5] != Py_None) {
            const at::Tensor *t = gpu_tensor(a[5]);
            if (!t || t->scalar_type() != at::kInt || t->numel() < 1 || t->device() != x->device()) return none();
            n_dev = static_cast<const int32_t *>(t->data_ptr());
        }
        const int64_t cols = (gate ? 2 : 1) * n;
        auto buffer = [&](const at::Tensor *t, int64_t width) {   // usable as it is, or once resized
            if (!t || !same_kind(*t, *x)) return false;
            const bool fits = t->dim() == 2 && t->size(0) == B && t->size(1) == width;
            return fits ? t->is_contiguous() : as_operator != 0;
        };
        const at::Tensor *comb = a[7] == Py_None ? nullptr : gpu_tensor(a[7]), *o = a[6] == Py_None ? nullptr : gpu_tensor(a[6]);
        if ((a[7] != Py_None && !buffer(comb, cols)) || (a[6] != Py_None && !buffer(o, H))) return none();
        if (o && comb && o->is_same(*comb) && cols != H) return none();   // (one tensor cannot become both)
        auto fit = [&](const at::Tensor *t, int64_t width) {
            if (t->dim() != 2 || t->size(0) != B || t->size(1) != width) t->resize_({B, width});
        };
        at::Tensor out;
        if (o) { fit(o, H); out = *o; } else { out = at::empty_like(*x); }
        if (comb) fit(comb, cols);
        const void *px = x->data_ptr(), *pg = gate ? gate->data_ptr() : nullptr, *pu = up->data_ptr(), *pd = down->data_ptr();
        void *po = out.data_ptr(), *pc = comb ? comb->data_ptr() : nullptr, *pw = ws->data_ptr();
        const int64_t bytes = ws->numel();
        const int rc = launched([&] {
            return f_mlp_forward(px, B, H, pg, pu, pd, n, n_dev, hint, po, pc, comb ? cols : 0, pw, bytes, (int)act, code, gate ? 1 : 0,
                                 stream);
        });
        if (rc != ST_OK) return PyLong_FromLong(rc);
        if (o) { Py_INCREF(a[6]); return a[6]; }
        return THPVariable_Wrap(out);
    });
}

// cache_build(gate | None, up, down, mask, H, state_words, stream) -> (handle, gate_pool | None, up_pool, downT_pool, gate_active |
// None, up_active, down_active, book) | status | None: a new cache's buffers and handle, its kernel launched.  The caller
// waits for it (st_cache_load_weights_end) and keeps the weights and the mask until then.  `book` (int32) holds the index list
// [2, I], the remembered mask (2 I bytes) and the state words, each at a multiple of 64 words.
PyObject *cache_build(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 7 || !f_load_begin) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *gate = a[0] == Py_None ? nullptr : gpu_tensor(a[0]), *up = gpu_tensor(a[1]), *down = gpu_tensor(a[2]),
                         *mask = gpu_tensor(a[3]);
        if (!up || !down || !mask || (a[0] != Py_None && !gate) || up->dim() != 2) return none();
        const int64_t I = up->size(0), H = up->size(1), hidden = PyLong_AsLongLong(a[4]), words = PyLong_AsLongLong(a[5]);
        void *stream = PyLong_AsVoidPtr(a[6]);
        if (PyErr_Occurred()) { PyErr_Clear(); return none(); }
        const int code = code_of(*up);
        if (code < 0 || I < 1 || I > f_max_intermediate() || H < 1 || H != hidden || words < 1) return none();
        if (!rows_of(*up, H) || !rows_of(*down, I) || down->size(0) != H || !same_kind(*down, *up)) return none();
        if (gate && (!rows_of(*gate, H) || gate->size(0) != I || !same_kind(*gate, *up))) return none();
        if (!bytes_of(*mask, *up, I)) return none();
        at::Tensor t[6];   // pools, packed rows
        for (int k = 0; k < 6; ++k)
            if (gate || k % 3 != 0) t[k] = at::empty({I, H}, up->options());
        auto whole = [](int64_t v) { return (v + 63) / 64 * 64; };
        const int64_t at_mask = whole(2 * I), at_state = at_mask + whole((2 * I + 3) / 4);
        at::Tensor book = at::empty({at_state + words}, up->options().dtype(at::kInt));
        int32_t *pb = static_cast<int32_t *>(book.data_ptr());
        auto ptr = [&](int k) { return t[k].defined() ? t[k].data_ptr() : nullptr; };
        const st_cache_buffers bufs = {ptr(0), ptr(1), ptr(2), ptr(3), ptr(4), ptr(5), pb, reinterpret_cast<uint8_t *>(pb + at_mask), pb + at_state};
        st_cache *c = f_cache_create(&bufs, I, H, code, gate ? 1 : 0);
        if (!c) return none();   // (the general path raises what it says)
        const void *pg = gate ? gate->data_ptr() : nullptr, *pu = up->data_ptr(), *pd = down->data_ptr();
        const uint8_t *pm = static_cast<const uint8_t *>(mask->data_ptr());
        const int rc = launched([&] { return f_load_begin(c, pg, pu, pd, pm, stream); });
        if (rc != ST_OK) {
            f_cache_destroy(c);
            return PyLong_FromLong(rc);
        }
        // from here on nothing throws: the kernel writes to these buffers
        auto wrap = [](const at::Tensor &v) -> PyObject * {
            if (!v.defined()) { Py_RETURN_NONE; }
            return THPVariable_Wrap(v);
        };
        PyObject *r = PyTuple_New(8);
        if (!r) return nullptr;
        PyTuple_SET_ITEM(r, 0, PyLong_FromVoidPtr(c));
        for (int k = 0; k < 6; ++k) PyTuple_SET_ITEM(r, 1 + k, wrap(t[k]));
        PyTuple_SET_ITEM(r, 7, wrap(book));
        return r;
    });
}

// bind(st_predictor_mask_ex, st_cache_update_forward, st_mlp_forward, st_cache_create, st_cache_destroy,
// st_cache_load_weights_begin, st_cache_max_intermediate): their addresses in the loaded library
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    constexpr int kFunctions = 7;
    if (n != kFunctions) {
        PyErr_SetString(PyExc_TypeError, "bind takes seven addresses");
        return nullptr;
    }
    void *p[kFunctions];
    for (int i = 0; i < kFunctions; ++i) {
        p[i] = PyLong_AsVoidPtr(a[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    f_predictor = reinterpret_cast<decltype(f_predictor)>(p[0]);
    f_update_forward = reinterpret_cast<decltype(f_update_forward)>(p[1]);
    f_mlp_forward = reinterpret_cast<decltype(f_mlp_forward)>(p[2]);
    f_cache_create = reinterpret_cast<decltype(f_cache_create)>(p[3]);
    f_cache_destroy = reinterpret_cast<decltype(f_cache_destroy)>(p[4]);
    f_load_begin = reinterpret_cast<decltype(f_load_begin)>(p[5]);
    f_max_intermediate = reinterpret_cast<decltype(f_max_intermediate)>(p[6]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {"predictor_mask", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(predictor_mask)), METH_FASTCALL, nullptr},
    {"update_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(update_forward)), METH_FASTCALL, nullptr},
    {"mlp_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(mlp_forward)), METH_FASTCALL, nullptr},
    {"cache_build", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(cache_build)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
