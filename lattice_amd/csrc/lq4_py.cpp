// CPython entry to the C ABI of liblattice_hip_q4.so for the calls an engine makes many times a token
// (built by lattice_amd/build.py next to the library; loaded by lattice_amd/backend.py).
//
// A launch costs the HIP runtime 2.2 us on this machine.  Through ctypes (argument objects, a structure filled
// field by field) and torch.cuda.current_stream() a one-row GEMV cost the host 6.8 us, i.e. two thirds of the call were
// spent before the library saw it; with these wrappers the same call takes 3.3 us (4096 x 1024, one row), an eight-row decode
// layer's host time falls from 39 to 24 us.
// The GIL is released around the call, as ctypes does: a call may allocate or wait on a full queue.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/lattice_hip_q4.h"

namespace {

PyObject* g_error = nullptr;  // Q4Error(code, message)
PyObject *g_handle, *g_data_ptr, *g_d_in, *g_d_out;

PyObject* finish(int rc) {
    if (rc == LQ4_OK) Py_RETURN_NONE;
    if (!g_error) return PyErr_Format(PyExc_RuntimeError, "[%d] %s", rc, lq4_last_error());
    PyObject* e = PyObject_CallFunction(g_error, "is", rc, lq4_last_error());
    if (e) {
        PyErr_SetObject(g_error, e);
        Py_DECREF(e);
    }
    return nullptr;
}

template <class T>
bool convert(PyObject* o, T* out) {
    if constexpr (std::is_pointer_v<T>) {
        *out = nullptr;
        if (o == Py_None) return true;
        void* p = PyLong_AsVoidPtr(o);
        if (!p && PyErr_Occurred()) return false;
        *out = static_cast<T>(p);
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) return false;
        *out = static_cast<T>(v);
        return true;
    } else if constexpr (std::is_signed_v<T>) {
        const long v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred()) return false;
        *out = static_cast<T>(v);
        return true;
    } else {
        const unsigned long long v = PyLong_AsUnsignedLongLong(o);
        if (v == ~0ull && PyErr_Occurred()) return false;
        if (sizeof(T) < 8 && v > 0xFFFFFFFFull) {
            PyErr_SetString(PyExc_OverflowError, "argument does not fit 32 bits");
            return false;
        }
        *out = static_cast<T>(v);
        return true;
    }
}

// One wrapper per C function: positional arguments in the C order, pointers and handles as integers (None = null).
template <auto Fn>
struct Wrap;

template <class... A, int (*Fn)(A...)>
struct Wrap<Fn> {
    template <size_t... I>
    static PyObject* go(PyObject* const* args, std::index_sequence<I...>) {
        std::tuple<A...> v;
        if (!(convert(args[I], &std::get<I>(v)) && ...)) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = Fn(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        return finish(rc);
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        if (n != static_cast<Py_ssize_t>(sizeof...(A)))
            return PyErr_Format(PyExc_TypeError, "expected %d arguments, got %d", static_cast<int>(sizeof...(A)), static_cast<int>(n));
        return go(args, std::index_sequence_for<A...>{});
    }
};

// lq4_gemv_fused_batch with the fields of lq4_gemv_fusion as arguments:
// (ctx, w, offset, n, k, x, batch, y, prologue, base, delta, gamma, eps, residual_out, epilogue, residual, copy_dst,
//  lora, scale, stream)
int fused(lq4_ctx* ctx, const lq4_weight* w, uint64_t off, uint32_t n, uint32_t k, const float* x, uint32_t batch, float* y,
          int prologue, const float* base, const float* delta, const float* gamma, float eps, float* residual_out,
          int epilogue, float* residual, float* copy_dst, const lq4_lora* lora, float scale, void* stream) {
    const lq4_gemv_fusion f{prologue, base, delta, gamma, eps, residual_out, epilogue, residual, copy_dst};
    return lq4_gemv_fused_batch(ctx, w, off, n, k, x, batch, y, &f, lora, scale, stream);
}

template <class T>
bool attribute(PyObject* o, PyObject* name, T* out) {
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) return false;
    const bool ok = convert(v, out);
    Py_DECREF(v);
    return ok;
}

// The adapter handle of (layer_idx, module) in `loaded` (a dict of projections with handle, d_in and d_out), null
// where there is none; false with an exception set.
bool adapter(PyObject* loaded, PyObject* layer, PyObject* module, uint32_t n, uint32_t k, const lq4_lora** out) {
    *out = nullptr;
    if (layer == Py_None || module == Py_None) return true;
    PyObject* key = PyTuple_Pack(2, layer, module);
    if (!key) return false;
    PyObject* p = PyDict_GetItemWithError(loaded, key);
    Py_DECREF(key);
    if (!p) return !PyErr_Occurred();
    uint32_t d_in, d_out;
    if (!attribute(p, g_d_in, &d_in) || !attribute(p, g_d_out, &d_out) || !attribute(p, g_handle, out)) return false;
    if (d_in != k || d_out != n) {
        PyErr_SetString(PyExc_AssertionError, "LoRA projection shape does not match the GEMV");
        return false;
    }
    return true;
}

// gemv_multi(ctx, projections, k, x, batch, loaded, layer_idx, scale, stream); a projection is
// (qw, n, y[, module[, qw_extra_offset]])
PyObject* multi(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (n_args != 9) return PyErr_Format(PyExc_TypeError, "expected 9 arguments");
    lq4_ctx* ctx;
    uint32_t k, batch;
    const float* x;
    float scale;
    void* stream;
    if (!convert(a[0], &ctx) || !convert(a[2], &k) || !convert(a[3], &x) || !convert(a[4], &batch) || !convert(a[7], &scale) ||
        !convert(a[8], &stream))
        return nullptr;
    if (!PyDict_Check(a[5])) return PyErr_Format(PyExc_TypeError, "loaded adapters must be a dict");
    PyObject* list = PySequence_Fast(a[1], "projections must be a sequence");
    if (!list) return nullptr;
    lq4_projection proj[LQ4_MAX_PROJECTIONS] = {};
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(list);
    bool ok = count <= LQ4_MAX_PROJECTIONS;
    if (!ok) PyErr_Format(PyExc_ValueError, "%zd projections, at most %d a call", count, LQ4_MAX_PROJECTIONS);
    for (Py_ssize_t i = 0; ok && i < count; ++i) {
        PyObject* p = PySequence_Fast(PySequence_Fast_GET_ITEM(list, i), "a projection is (qw, n, y[, module[, offset]])");
        if (!p) {
            ok = false;
            break;
        }
        const Py_ssize_t len = PySequence_Fast_GET_SIZE(p);
        PyObject** f = PySequence_Fast_ITEMS(p);
        PyObject* y = nullptr;
        ok = len >= 3;
        if (!ok) PyErr_SetString(PyExc_ValueError, "a projection is (qw, n, y[, module[, offset]])");
        ok = ok && attribute(f[0], g_handle, &proj[i].w) && convert(f[1], &proj[i].n) &&
             (y = PyObject_CallMethodNoArgs(f[2], g_data_ptr)) && convert(y, &proj[i].y_dev) &&
             adapter(a[5], a[6], len > 3 ? f[3] : Py_None, proj[i].n, k, &proj[i].lora) &&
             (len <= 4 || convert(f[4], &proj[i].w_extra_offset));
        proj[i].lora_scale = scale;
        Py_XDECREF(y);
        Py_DECREF(p);
    }
    Py_DECREF(list);
    if (!ok) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = lq4_gemv_multi(ctx, proj, static_cast<uint32_t>(count), k, x, batch, stream);
    Py_END_ALLOW_THREADS
    return finish(rc);
}

// gemv_chain(ctx, steps, stream); every step an object whose buffer is an lq4_chain_step
PyObject* chain(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (n_args != 3) return PyErr_Format(PyExc_TypeError, "expected 3 arguments");
    lq4_ctx* ctx;
    void* stream;
    if (!convert(a[0], &ctx) || !convert(a[2], &stream)) return nullptr;
    PyObject* list = PySequence_Fast(a[1], "steps must be a sequence");
    if (!list) return nullptr;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(list);
    std::vector<lq4_chain_step> steps(static_cast<size_t>(count));
    bool ok = true;
    for (Py_ssize_t i = 0; ok && i < count; ++i) {
        Py_buffer b;
        ok = PyObject_GetBuffer(PySequence_Fast_GET_ITEM(list, i), &b, PyBUF_SIMPLE) == 0;
        if (!ok) break;
        ok = b.len == static_cast<Py_ssize_t>(sizeof(lq4_chain_step));
        if (ok) memcpy(&steps[static_cast<size_t>(i)], b.buf, sizeof(lq4_chain_step));
        else PyErr_SetString(PyExc_TypeError, "a step is a ChainStep");
        PyBuffer_Release(&b);
    }
    Py_DECREF(list);
    if (!ok) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = lq4_gemv_chain(ctx, steps.data(), static_cast<uint32_t>(count), stream);
    Py_END_ALLOW_THREADS
    return finish(rc);
}

PyObject* set_error(PyObject*, PyObject* cls) {
    Py_INCREF(cls);
    Py_XSETREF(g_error, cls);
    Py_RETURN_NONE;
}

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
#define ABI(fn) FAST(#fn, Wrap<&fn>::call)
PyMethodDef methods[] = {
    ABI(lq4_gemv), ABI(lq4_gemm), ABI(lq4_gemv_q8), ABI(lq4_gemm_q8), ABI(lq4_gemv_q3), ABI(lq4_gemm_q3),
    ABI(lq4_residual_add_rmsnorm), ABI(lq4_silu_mul), ABI(lq4_add_and_copy), ABI(lq4_lora_apply),
    ABI(lq4_moe_route), ABI(lq4_moe_grouped_gemv), ABI(lq4_moe_shared_expert), ABI(lq4_moe_ffn),
    ABI(lq4_topk), ABI(lq4_lm_head_topk), ABI(lq4_lm_head_topk_static),
    FAST("gemv_fused_batch", Wrap<&fused>::call), FAST("gemv_multi", multi), FAST("gemv_chain", chain),
    {"set_error", set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lq4_py", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lq4_py(void) {
    g_handle = PyUnicode_InternFromString("handle");
    g_data_ptr = PyUnicode_InternFromString("data_ptr");
    g_d_in = PyUnicode_InternFromString("d_in");
    g_d_out = PyUnicode_InternFromString("d_out");
    if (!g_handle || !g_data_ptr || !g_d_in || !g_d_out) return nullptr;
    return PyModule_Create(&module);
}
